"""Stream capture of the library's stream for tests."""
import ctypes

from deers_amd import rocm


class _KernelNodeParams(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("params", ctypes.c_void_p), ("lds", ctypes.c_uint)]


class Graph:
    """What `calls()` enqueues, captured; launch() replays it on the library's stream."""

    def __init__(self, calls):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.stream = ctypes.c_void_p(rocm.load().deers_rocm_stream())
        self.graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()
        assert self.hip.hipStreamBeginCapture(self.stream, 2) == 0  # hipStreamCaptureModeRelaxed
        try:
            calls()
        finally:
            assert self.hip.hipStreamEndCapture(self.stream, ctypes.byref(self.graph)) == 0
        assert self.hip.hipGraphInstantiate(ctypes.byref(self.exec), self.graph, None, None, ctypes.c_size_t(0)) == 0

    def threads(self):
        """Threads per workgroup of every kernel node."""
        count = ctypes.c_size_t()
        assert self.hip.hipGraphGetNodes(self.graph, None, ctypes.byref(count)) == 0
        nodes = (ctypes.c_void_p * count.value)()
        assert self.hip.hipGraphGetNodes(self.graph, nodes, ctypes.byref(count)) == 0
        out = []
        for node in nodes:
            params = _KernelNodeParams()
            assert self.hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(params)) == 0
            out.append(params.block[0] * params.block[1] * params.block[2])
        return out

    def launch(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        rocm.sync()
        self.hip.hipGraphExecDestroy(self.exec)
        self.hip.hipGraphDestroy(self.graph)
