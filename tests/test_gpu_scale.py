"""The pruning of local solves does not depend on the mesh's scale: register-resident visits hold a tet's
corner heights in 16 bits, in units taken from the block's own heights.  The same jittered cube with its
edges (or, in a batch, a solve's factors) scaled over 16 orders of magnitude: as many local solves of the
one-launch-per-iteration solve as at scale 1, within 5% (rounding moves single times, and with them single
solves; a height rounded to 11 bits prunes 1 in 2,000 solves less), of the persistent solve and a batch within
35% (their visits vary from run to run by up to 15%; without pruning there are 3 times as many).  Times equal
those at scale 1 times the scale, at 1e-4 relative (fp32 coordinates of the scaled mesh are rounded anew)."""
import numpy as np
import pytest

from conftest import lognormal_mult

pytestmark = pytest.mark.gpu

N = 16


def _cube(E, scale):
    m = E.Mesh.kuhn_cube(N, 0.2, seed=9)
    xyz, t = m.vertices(), m.elements()
    m = E.Mesh.tet((xyz * np.float32(scale)).astype(np.float32), t)
    m.set_speed(lognormal_mult(len(t), 9))
    m.partition(64)
    return m


@pytest.mark.parametrize("sched,slack", [(0, 1.05), (1, 1.35)])
def test_local_solves_at_any_scale(E, sched, slack):
    ref, st = _cube(E, 1.0).solve([0], scheduler=sched)
    for scale in (1e-9, 1e-7, 3e-6, 1e-4, 1e3, 3e5, 1e7):
        T, s = _cube(E, scale).solve([0], scheduler=sched)
        print("scale %g: %d local solves, %d at scale 1" % (scale, s["local_solves"], st["local_solves"]), flush=True)
        assert s["local_solves"] <= slack * st["local_solves"]
        assert np.max(np.abs(T / scale - ref)) <= 1e-4 * ref.max()


def test_local_solves_with_any_factors(E):
    m = _cube(E, 1.0)
    f = np.ones(m.info()["nelem"], np.float32)
    b = E.Batch([m])
    Ts, st = b.solve([[0]])
    for scale in (1e-8, 1e-6, 1e-3, 1e4, 1e7):
        b.set_factors(0, f * np.float32(scale) ** 2)
        T, s = b.solve([[0]])
        print("factors %g^2: %d local solves, %d without" % (scale, s["local_solves"], st["local_solves"]), flush=True)
        assert s["local_solves"] <= 1.35 * st["local_solves"]
        assert np.max(np.abs(T[0] / scale - Ts[0])) <= 1e-4 * Ts[0].max()
    b.close()
