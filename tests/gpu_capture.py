"""HIP graphs of what a context issues, through the runtime that the library itself is linked with."""
import contextlib
import ctypes as C

from tpu_compiler_amd import capi

THREAD_LOCAL = 1     # hipStreamCaptureModeThreadLocal
NOT_READY = 600      # hipErrorNotReady


class Graph:
    """the calls made inside `with graph.recording():`, to be replayed"""

    def __init__(self, context_handle):
        self.lib = capi.bind()     # symbols of the HIP runtime resolve through the library's own dependencies
        self.stream = C.c_void_p(self.lib.tpuhip_ctx_stream(context_handle))
        self.graph, self.exec = C.c_void_p(), C.c_void_p()

    def _hip(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, "%s: %d" % (name, rc)

    @contextlib.contextmanager
    def recording(self):
        self._hip("hipStreamBeginCapture", self.stream, THREAD_LOCAL)
        try:
            yield self
        finally:
            self._hip("hipStreamEndCapture", self.stream, C.byref(self.graph))

    def nodes(self):
        n = C.c_size_t()
        self._hip("hipGraphGetNodes", self.graph, None, C.byref(n))
        return n.value

    def replay(self):
        if not self.exec:
            self._hip("hipGraphInstantiate", C.byref(self.exec), self.graph, None, None, C.c_size_t(0))
        self._hip("hipGraphLaunch", self.exec, self.stream)

    def idle(self):
        """whether everything issued to the stream has ended"""
        rc = self.lib.hipStreamQuery(self.stream)
        assert rc in (0, NOT_READY)
        return rc == 0

    def close(self):
        self._hip("hipStreamSynchronize", self.stream)
        if self.exec:
            self._hip("hipGraphExecDestroy", self.exec)
        if self.graph:
            self._hip("hipGraphDestroy", self.graph)
        self.graph, self.exec = C.c_void_p(), C.c_void_p()
