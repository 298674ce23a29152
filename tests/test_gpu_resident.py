"""The register-resident visits of the persistent single solve (a block's items or elements held
in registers), at the block sizes where their shape changes: blocks just inside and beyond what N
items or elements per thread cover, one vertex per block, a ragged last block and a relative
convergence threshold.  Against the FP64 oracle at
1e-5 relative (floor: a quarter of the shortest source-adjacent edge time), the tolerance of the
parity tests.
"""
import numpy as np
import pytest

from conftest import center_vertex, lognormal_mult, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _edge_floor(xyz, elem, seeds, scale):
    xyz = np.asarray(xyz, np.float64)
    on = np.zeros(len(xyz), bool)
    on[np.atleast_1d(seeds)] = True
    sel = on[elem].any(axis=1)
    t, s = elem[sel], scale[sel]
    k = elem.shape[1]
    return 0.25 * min(float((s * np.linalg.norm(xyz[t[:, i]] - xyz[t[:, j]], axis=1)).min())
                      for i in range(k) for j in range(i + 1, k))


# (vertices per block): 2 x 256 items up to 85 or so, 4 x 256 up to 170, 4 x 512 up to 340, the
# general kernel beyond
@pytest.mark.parametrize("vpb", [1, 7, 64, 90, 140, 180, 300, 420])
def test_triangle_shapes(E, O, vpb):
    m = E.Mesh.icosphere(4)
    xyz, f = m.vertices(), m.elements()
    rng = np.random.default_rng(vpb)
    th, k = rng.uniform(0, np.pi, len(f)), rng.uniform(1, 10, len(f))
    M = np.stack([np.cos(th) ** 2 + k * np.sin(th) ** 2, (1 - k) * np.cos(th) * np.sin(th),
                  np.sin(th) ** 2 + k * np.cos(th) ** 2], 1).astype(np.float32)
    m.set_metric_tri(M)
    m.partition(vpb)
    seeds = np.array([5, 1300], np.int32)
    T, st = m.solve(seeds)
    G = O.tri_gram(xyz, f, metric=M.astype(np.float64))
    ref, _ = O.fim2d(xyz.astype(np.float64), f, seeds, G, 1)
    err = rel_err(T, ref, _edge_floor(xyz, f, seeds, np.ones(len(f))))
    print("vpb %d: %d blocks, visits %d, max rel err %.3e"
          % (vpb, m.info()["nblocks"], st["block_visits"], err), flush=True)
    assert err <= TOL


# 4 x 256 elements up to 85 or so vertices per block, 4 x 512 up to 200, the general kernel beyond
@pytest.mark.parametrize("vpb", [1, 7, 64, 84, 100, 180, 260])
@pytest.mark.parametrize("eps", [0.0, 1e-7])
def test_tet_shapes(E, O, vpb, eps):
    n = 11
    m = E.Mesh.kuhn_cube(n, 0.2, seed=vpb)
    xyz, t = m.vertices(), m.elements()
    mult = lognormal_mult(len(t), vpb)
    m.set_speed(mult)
    m.partition(vpb)
    seeds = np.array([center_vertex(n), 3], np.int32)
    T, st = m.solve(seeds, eps=eps)
    with O.exact():
        ref, _ = O.fim3d(xyz.astype(np.float64), t, seeds,
                         M6=O.tet_metric(len(t), mult.astype(np.float64)))
    err = rel_err(T, ref, _edge_floor(xyz, t, seeds, np.sqrt(mult.astype(np.float64))))
    print("vpb %d eps %g: largest block %d tets, visits %d, max rel err %.3e"
          % (vpb, eps, m.info()["max_block_elems"], st["block_visits"], err), flush=True)
    assert err <= TOL

