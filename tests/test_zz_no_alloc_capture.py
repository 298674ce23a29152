"""eik_solve_noalloc under HIP graph capture: the captured solve is replayed several times, with other
sources written into its seed buffer and eager solves of another mesh in between, and every replay gives
what an eager solve gives (2e-6 relative, the tolerance of the batch tests)."""
import ctypes

import numpy as np
import pytest

from conftest import lognormal_mult

pytestmark = pytest.mark.gpu

TOL = 2e-6


class _Hip:
    """The HIP runtime that the library links."""

    def __init__(self):
        self.h = ctypes.CDLL("libamdhip64.so.7")

    def __getattr__(self, name):
        f = getattr(self.h, name)

        def call(*a):
            rc = f(*a)
            assert rc == 0, "%s: %d" % (name, rc)
        return call


def _ptr(x):
    return ctypes.c_void_p(x)


@pytest.mark.parametrize("kind,size", [("tets", 16), ("triangles", 5), ("triangles", 7)])
def test_replays_equal_eager_solves(E, kind, size):
    if kind == "tets":
        m = E.Mesh.kuhn_cube(size, 0.2, seed=4)
        m.set_speed(lognormal_mult(m.info()["nelem"], 4))
    else:
        m = E.Mesh.icosphere(size)
    m.partition(64)
    m.upload()
    other = E.Mesh.kuhn_cube(12, 0.2, seed=5)
    other.partition(64)
    other.upload()
    hip = _Hip()
    seeds, out, out2, stream, graph, ex = (ctypes.c_void_p() for _ in range(6))
    hip.hipMalloc(ctypes.byref(seeds), ctypes.c_size_t(4))
    hip.hipMalloc(ctypes.byref(out), ctypes.c_size_t(4 * m.nv))
    hip.hipMalloc(ctypes.byref(out2), ctypes.c_size_t(4 * other.nv))
    hip.hipStreamCreateWithFlags(ctypes.byref(stream), ctypes.c_uint(1))

    def put(p, a):
        hip.hipMemcpy(p, _ptr(a.ctypes.data), ctypes.c_size_t(a.nbytes), ctypes.c_int(1))

    def get(p, n):
        a = np.empty(n, np.float32)
        hip.hipMemcpy(_ptr(a.ctypes.data), p, ctypes.c_size_t(a.nbytes), ctypes.c_int(2))
        return a

    put(seeds, np.zeros(1, np.int32))
    m.solve_noalloc(seeds.value, 1, out.value, stream.value)  # (the first call looks up the scratch array)
    hip.hipStreamSynchronize(stream)
    hip.hipStreamBeginCapture(stream, ctypes.c_int(1))
    m.solve_noalloc(seeds.value, 1, out.value, stream.value)
    hip.hipStreamEndCapture(stream, ctypes.byref(graph))
    hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0))
    try:
        for k, v in enumerate((0, m.nv - 1, m.nv // 3, 7, 0)):
            put(seeds, np.array([v], np.int32))
            put(out, np.full(m.nv, -1.0, np.float32))
            hip.hipGraphLaunch(ex, stream)
            hip.hipStreamSynchronize(stream)
            T = get(out, m.nv)
            ref, _ = m.solve([v])
            err = np.max(np.abs(T - ref) / np.maximum(ref, 1e-3))
            print("%s %d, replay %d: max rel diff %.3e" % (kind, size, k, err), flush=True)
            assert err <= TOL
            other.solve_noalloc(seeds.value, 1, out2.value, stream.value)  # leaves its state in the scratch array
            hip.hipStreamSynchronize(stream)
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)
        for p in (seeds, out, out2):
            hip.hipFree(p)
