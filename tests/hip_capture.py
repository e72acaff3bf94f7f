"""HIP stream capture by a caller of the library, through ctypes: the graphs
that entry points record, and the grids of their kernels."""
import ctypes as C

import aiehlc_amd as mi

NON_BLOCKING, THREAD_LOCAL, RELAXED = 1, 1, 2  # hipStreamNonBlocking, hipStreamCaptureMode*


class _Dim3(C.Structure):
    _fields_ = [("x", C.c_uint), ("y", C.c_uint), ("z", C.c_uint)]


class _KernelNodeParams(C.Structure):  # hipKernelNodeParams
    _fields_ = [("blockDim", _Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("gridDim", _Dim3),
                ("kernelParams", C.c_void_p), ("sharedMemBytes", C.c_uint)]


class Capture:
    """A context on a stream of the caller's, and a second stream for replays."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.streams = [C.c_void_p(), C.c_void_p()]
        for s in self.streams:
            self.ok(self.hip.hipStreamCreateWithFlags(C.byref(s), NON_BLOCKING))
        self.ctx = mi.Context(0, stream=self.streams[0].value)

    def ok(self, rc):
        assert rc == 0, rc

    def record(self, call):
        """(graph executable, grid of each kernel node)"""
        hip, graph, exe, n = self.hip, C.c_void_p(), C.c_void_p(), C.c_size_t()
        self.ok(hip.hipStreamBeginCapture(self.streams[0], THREAD_LOCAL))
        try:
            call()
        finally:
            rc = hip.hipStreamEndCapture(self.streams[0], C.byref(graph))
        self.ok(rc)
        self.ok(hip.hipGraphGetNodes(graph, None, C.byref(n)))
        nodes = (C.c_void_p * n.value)()
        self.ok(hip.hipGraphGetNodes(graph, nodes, C.byref(n)))
        grids = []
        for node in nodes:
            p = _KernelNodeParams()
            self.ok(hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)))
            grids.append((p.gridDim.x, p.gridDim.y, p.gridDim.z))
        self.ok(hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0))
        self.ok(hip.hipGraphDestroy(graph))
        return exe, grids

    def replay(self, exe):
        self.ok(self.hip.hipGraphLaunch(exe, self.streams[1]))

    def sync(self):
        for s in self.streams:
            self.ok(self.hip.hipStreamSynchronize(s))

    def close(self):
        self.sync()
        self.ctx.close()
        for s in self.streams:
            self.ok(self.hip.hipStreamDestroy(s))
