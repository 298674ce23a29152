"""Where a block visit of the persistent single solve has its element data (stage_records): in registers
where the blocks fit them, staged in LDS, and read from memory, at block sizes from one vertex to
blocks whose records do not fit the LDS.  Against the FP64 oracle at 1e-5 relative (floor: a quarter of the
shortest source-adjacent edge time), the tolerance of the parity tests."""
import numpy as np
import pytest

from conftest import center_vertex, lognormal_mult, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5
AUTO, LDS, MEMORY = 0, 1, 2


def _floor(xyz, elem, seeds, scale):
    on = np.zeros(len(xyz), bool)
    on[seeds] = True
    sel = on[elem].any(axis=1)
    t, s = elem[sel], scale[sel]
    k = elem.shape[1]
    xyz = xyz.astype(np.float64)
    return 0.25 * min(float((s * np.linalg.norm(xyz[t[:, i]] - xyz[t[:, j]], axis=1)).min())
                      for i in range(k) for j in range(i + 1, k))


@pytest.mark.parametrize("stage", [AUTO, LDS, MEMORY])
@pytest.mark.parametrize("vpb", [1, 30, 64, 192, 420, 1200])
def test_tets(E, O, vpb, stage):
    n = 14
    m = E.Mesh.kuhn_cube(n, 0.2, seed=vpb)
    xyz, t = m.vertices(), m.elements()
    mult = lognormal_mult(len(t), vpb)
    m.set_speed(mult)
    m.partition(vpb)
    seeds = np.array([center_vertex(n), 3], np.int32)
    T, st = m.solve(seeds, stage_records=stage)
    with O.exact():
        ref, _ = O.fim3d(xyz.astype(np.float64), t, seeds, M6=O.tet_metric(len(t), mult.astype(np.float64)))
    err = rel_err(T, ref, _floor(xyz, t, seeds, np.sqrt(mult.astype(np.float64))))
    print("vpb %d, stage %d: largest block %d tets, visits %d, max rel err %.3e"
          % (vpb, stage, m.info()["max_block_elems"], st["block_visits"], err), flush=True)
    assert err <= TOL


@pytest.mark.parametrize("stage", [AUTO, LDS, MEMORY])
@pytest.mark.parametrize("vpb", [1, 40, 64, 300, 700, 2600])
def test_triangles(E, O, vpb, stage):
    m = E.Mesh.icosphere(5)
    xyz, f = m.vertices(), m.elements()
    m.partition(vpb)
    seeds = np.array([5, 1300], np.int32)
    T, st = m.solve(seeds, stage_records=stage)
    ref, _ = O.fim2d(xyz.astype(np.float64), f, seeds, np.ones(len(f)), 0)
    err = rel_err(T, ref, _floor(xyz, f, seeds, np.ones(len(f))))
    print("vpb %d, stage %d: largest block %d faces, visits %d, max rel err %.3e"
          % (vpb, stage, m.info()["max_block_elems"], st["block_visits"], err), flush=True)
    assert err <= TOL
