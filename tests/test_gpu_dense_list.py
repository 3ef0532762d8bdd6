"""Several tensors laid out for the host by one launch: more of them than one list holds, vectors among them, up to what goes
straight into the staging buffer and beyond it, and more than it holds.  Bytes (i8) are asked for one tensor at a time: the same
values by the launch of one."""
import numpy as np
import pytest

from tpu_compiler_amd import graphs, module

pytestmark = pytest.mark.gpu

RAGGED = [(1, 3, 5, 7), (2, 64, 16, 8), (1, 65, 1, 129), (3, 13, 1, 1), (1, 255, 13, 13), (2, 17, 9, 127), (1, 1, 1, 128), (1, 4, 3, 43)]


@pytest.mark.parametrize("shapes", [RAGGED[:2], RAGGED[:4], RAGGED[:5], RAGGED * 3 + RAGGED[:1],
                                    RAGGED * 3 + [(1, 70, 61, 67), (2, 129, 65, 131)]])
@pytest.mark.parametrize("i8", [False, True])
def test_every_tensor_of_a_graph(shapes, i8):
    g = graphs.Graph("list", 1)
    for i, s in enumerate(shapes):
        g.add(graphs.Op("tpu.input", "x%d" % i, [], s))
        g.add(graphs.Op("tpu.relu", "y%d" % i, ["x%d" % i], s))
    g.outputs = ["y%d" % i for i in range(len(shapes))]
    m = module()
    m.load(g)
    for k in range(2):
        xs = [np.random.default_rng(k + i).integers(-128, 128, s).astype(np.int8) for i, s in enumerate(shapes)]
        for i, x in enumerate(xs):
            m.set_tensor_i8("x%d" % i, x)
        m.invoke()
        if i8:
            every = {n: m.get_tensor_i8(n) for n in m.tensor_names()}
        else:
            every = m.get_all_tensor()
        for i, x in enumerate(xs):
            assert np.array_equal(every["x%d" % i], x) and np.array_equal(every["y%d" % i], np.maximum(x, 0)), i
    m.close()


# 56 MB that fit the staging buffer (32 MB) one by one: it is filled twice, a filling ends in the middle of the list, and the second
# read finds the buffers of the first
FILLINGS = [(1, 129, 300, 301), (1, 3, 5, 7), (2, 70, 251, 257), (3, 13, 1, 1), (1, 64, 331, 333)]


@pytest.mark.parametrize("order", [1, -1])
def test_more_than_the_staging_buffer_holds(order):
    shapes = FILLINGS[::order]
    g = graphs.Graph("fillings", 1)
    for i, s in enumerate(shapes):
        g.add(graphs.Op("tpu.input", "x%d" % i, [], s))
        g.add(graphs.Op("tpu.relu", "y%d" % i, ["x%d" % i], s))
    g.outputs = ["y%d" % i for i in range(len(shapes))]
    sizes = [int(np.prod(s)) for s in shapes for _ in range(2)]
    assert max(sizes) <= 32 << 20 < sum(sizes)
    m = module()
    m.load(g)
    for k in range(2):
        xs = [np.random.default_rng(k + i).integers(-128, 128, s).astype(np.int8) for i, s in enumerate(shapes)]
        for i, x in enumerate(xs):
            m.set_tensor_i8("x%d" % i, x)
        m.invoke()
        for every in (m.get_all_tensor(), m.get_all_tensor()):
            for i, x in enumerate(xs):
                assert np.array_equal(every["x%d" % i], x) and np.array_equal(every["y%d" % i], np.maximum(x, 0)), i
    m.close()


# one tensor of a list of one, as floats of more than one thread's turn (192 KB): straight into the staging buffer, by way of the device
@pytest.mark.parametrize("shape", [(1, 65, 31, 33), (2, 130, 61, 67)])
def test_one_tensor_alone(shape):
    g = graphs.Graph("alone", 1)
    g.add(graphs.Op("tpu.input", "x", [], shape))
    g.add(graphs.Op("tpu.relu", "y", ["x"], shape))
    g.outputs = ["y"]
    m = module()
    m.load(g)
    for k in range(2):
        x = np.random.default_rng(k).integers(-128, 128, shape).astype(np.int8)
        m.set_tensor_i8("x", x)
        m.invoke()
        assert np.array_equal(m.get_tensor("y"), np.maximum(x, 0)) and np.array_equal(m.get_tensor("x"), x)
    m.close()
