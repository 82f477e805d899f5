"""Capture of a library call into a HIP graph, for tests that look at its launches or replay it."""
import ctypes as C

from pentago_amd import hip


class Dim3(C.Structure):
    _fields_ = [("x", C.c_uint32), ("y", C.c_uint32), ("z", C.c_uint32)]


class KernelNodeParams(C.Structure):   # hipKernelNodeParams
    _fields_ = [("block", Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", Dim3),
                ("params", C.c_void_p), ("shared", C.c_uint32)]


THREAD_LOCAL, KERNEL_NODE = 1, 0


class Captured:
    """call(stream address) captured on a stream of its own."""

    def __init__(self, call):
        self.stream, self.graph, self.exec = hip.Stream(), C.c_void_p(), C.c_void_p()
        s = C.c_void_p(self.stream.ptr)
        hip.check(hip.hip().hipStreamBeginCapture(s, THREAD_LOCAL), "hipStreamBeginCapture")
        try:
            call(self.stream.ptr)
        finally:
            code = hip.hip().hipStreamEndCapture(s, C.byref(self.graph))
        hip.check(code, "hipStreamEndCapture")

    def kernels(self):
        """(grid, block) of every kernel of the graph."""
        n = C.c_size_t()
        hip.check(hip.hip().hipGraphGetNodes(self.graph, None, C.byref(n)), "hipGraphGetNodes")
        nodes = (C.c_void_p * n.value)()
        hip.check(hip.hip().hipGraphGetNodes(self.graph, nodes, C.byref(n)), "hipGraphGetNodes")
        out = []
        for node in nodes:
            kind, p = C.c_int(), KernelNodeParams()
            hip.check(hip.hip().hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)), "hipGraphNodeGetType")
            if kind.value == KERNEL_NODE:
                hip.check(hip.hip().hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)),
                          "hipGraphKernelNodeGetParams")
                out.append((p.grid.x, p.block.x))
        return out

    def replay(self):
        if not self.exec:
            hip.check(hip.hip().hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)),
                      "hipGraphInstantiate")
        hip.check(hip.hip().hipGraphLaunch(self.exec, C.c_void_p(self.stream.ptr)), "hipGraphLaunch")

    def close(self):
        self.stream.synchronize()
        if self.exec:
            hip.hip().hipGraphExecDestroy(self.exec)
        hip.hip().hipGraphDestroy(self.graph)
        self.graph = self.exec = C.c_void_p()
