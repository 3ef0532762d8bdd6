"""What a loading module sends up and packs in shared launches: filters around a thread's 16 bytes and a copy's last dwords, one of
more than a pass of the copying and packing launches (1 MB, 32768 groups), 1x1 filters whose channels are packed 16 at a time and
those whose are not, all in one module."""
import numpy as np
import pytest

import oracle_graph
from tpu_compiler_amd import module
from tpu_compiler_amd.graphs import BASE_SEED, Builder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [
    [(20, 1), (7, 1)],                       # 140 bytes: 35 dwords
    [(16, 1), (1, 1), (5, 3)],               # one group of 16 channels, a layer of one channel
    [(17, 3), (48, 1), (33, 1), (12, 5)],
    [(1024, 1), (1040, 1), (1024, 1)],       # 1 064 960 bytes: a second pass of 16 bytes
    [(192, 3), (312, 3)],                    # 34 000 groups: a second pass of the packing
])
def test_filters_of_a_load_are_those_of_the_graph(layers):
    b = Builder("load", BASE_SEED + sum(oc for oc, _ in layers), 1, (6, 16))
    x, outs = b.input("input", 20, 6, 5), []
    for i, (oc, k) in enumerate(layers):
        x = b.conv("conv%d" % i, x, oc, k, stride=1, pad=k // 2, relu=i % 2 == 0)
        outs.append(x)
    g = b.finish(outs)
    want = oracle_graph.run(g)
    m = module()
    m.load(g)
    m.set_tensor("input", g.input_op().data.astype(np.float32))
    m.invoke()
    for i in range(len(layers)):
        name = "conv%d" % i
        assert np.array_equal(m.get_tensor_i8(name), want[name].reshape(g.by_name[name].shape)), name
    m.close()
