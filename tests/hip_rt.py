"""The HIP runtime libqpx runs on, by ctypes: streams, device memory and
graphs for the tests that enqueue device calls themselves."""
from __future__ import annotations

import ctypes as C

import numpy as np

NON_BLOCKING = 1
CAPTURE_GLOBAL, CAPTURE_THREAD_LOCAL = 0, 1


class Hip:
    def __init__(self):
        self.lib = C.CDLL("libamdhip64.so")
        self.lib.hipGetErrorString.restype = C.c_char_p

    def call(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, f"{name}: {self.lib.hipGetErrorString(rc).decode()}"

    def sync(self):
        self.call("hipDeviceSynchronize")

    def free_bytes(self) -> int:
        free, total = C.c_size_t(0), C.c_size_t(0)
        self.call("hipMemGetInfo", C.byref(free), C.byref(total))
        return free.value

    def stream(self):
        s = C.c_void_p()
        self.call("hipStreamCreateWithFlags", C.byref(s), C.c_uint(NON_BLOCKING))
        return s

    def capture(self, stream, enqueue, mode=CAPTURE_GLOBAL):
        """The executable graph of what enqueue() puts on the stream."""
        self.call("hipStreamBeginCapture", stream, C.c_int(mode))
        graph, ex = C.c_void_p(), C.c_void_p()
        try:
            enqueue()
        finally:
            rc = self.lib.hipStreamEndCapture(stream, C.byref(graph))
        assert rc == 0, "the capture was invalidated"
        self.call("hipGraphInstantiateWithFlags", C.byref(ex), graph, C.c_ulonglong(0))
        self.call("hipGraphDestroy", graph)
        return ex

    def replay(self, ex, stream):
        self.call("hipGraphLaunch", ex, stream)

    def drop(self, ex):
        self.call("hipGraphExecDestroy", ex)


class Arr:
    """A device copy of a numpy array."""

    def __init__(self, hip, a):
        self.hip, self.shape, self.dtype, self.nbytes = hip, a.shape, a.dtype, a.nbytes
        self.p = C.c_void_p()
        hip.call("hipMalloc", C.byref(self.p), C.c_size_t(max(a.nbytes, 1)))
        self.put(a)

    def put(self, a):
        a = np.ascontiguousarray(a, dtype=self.dtype)
        self.hip.call("hipMemcpy", self.p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), C.c_int(1))

    def get(self):
        a = np.empty(self.shape, dtype=self.dtype)
        self.hip.call("hipMemcpy", a.ctypes.data_as(C.c_void_p), self.p, C.c_size_t(a.nbytes), C.c_int(2))
        return a

    def free(self):
        self.hip.call("hipFree", self.p)
