"""HIP graphs of library calls for the GPU tests: capture on a stream of their own, count the nodes, replay."""
import ctypes as C

from metaltile_amd import _lib
from metaltile_amd.runtime import _ensure_init


class Graph:
    """with Graph() as g: <library calls>; then g.nodes and g.replay(). close() gives the library its own stream back."""

    def __init__(self):
        self.lib = _ensure_init()
        self.hip = C.CDLL("libamdhip64.so")
        for name, args in (("hipStreamCreate", [C.POINTER(C.c_void_p)]), ("hipStreamBeginCapture", [C.c_void_p, C.c_int]),
                           ("hipStreamEndCapture", [C.c_void_p, C.POINTER(C.c_void_p)]), ("hipGraphGetNodes", [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)]),
                           ("hipGraphInstantiate", [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]),
                           ("hipGraphLaunch", [C.c_void_p, C.c_void_p]), ("hipStreamSynchronize", [C.c_void_p]), ("hipGraphExecDestroy", [C.c_void_p]),
                           ("hipGraphDestroy", [C.c_void_p]), ("hipStreamDestroy", [C.c_void_p])):
            getattr(self.hip, name).argtypes = args
        self.stream, self.graph, self.exec = C.c_void_p(), C.c_void_p(), C.c_void_p()
        self._do("hipStreamCreate", C.byref(self.stream))
        _lib.check(self.lib.mtq_set_stream(self.stream))

    def _do(self, name, *a):
        rc = getattr(self.hip, name)(*a)
        assert rc == 0, f"{name}: {rc}"

    def __enter__(self):
        self._do("hipStreamBeginCapture", self.stream, 0)   # the global mode, the strictest
        return self

    def __exit__(self, kind, *_):
        rc = self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph))
        if kind is None:
            assert rc == 0, f"hipStreamEndCapture: {rc}"
            n = C.c_size_t()
            self._do("hipGraphGetNodes", self.graph, None, C.byref(n))
            self.nodes = n.value
            self._do("hipGraphInstantiate", C.byref(self.exec), self.graph, None, None, 0)

    def replay(self):
        self._do("hipGraphLaunch", self.exec, self.stream)
        self._do("hipStreamSynchronize", self.stream)

    def close(self):
        _lib.check(self.lib.mtq_sync())
        _lib.check(self.lib.mtq_set_stream(None))
        if self.exec:
            self._do("hipGraphExecDestroy", self.exec)
        if self.graph:
            self._do("hipGraphDestroy", self.graph)
        self._do("hipStreamDestroy", self.stream)
