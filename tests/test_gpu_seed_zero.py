"""A source that starts at -0 starts at 0: the field equals that of the default start times, with both
schedulers, in multi-solve launches, and beside a source that starts later.  Both solves end at the same
fixed point: 2e-6 relative, the tolerance of the batch tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _mesh(E, kind):
    m = E.Mesh.kuhn_cube(12, 0.2, seed=7) if kind == "tets" else E.Mesh.icosphere(4)
    m.partition(64)
    return m


def _same(T, ref):
    assert np.max(np.abs(T - ref) / np.maximum(ref, 1e-3)) <= TOL


@pytest.mark.parametrize("kind", ["tets", "triangles"])
@pytest.mark.parametrize("vals", [[-0.0], [-0.0, 0.25]])
def test_single(E, kind, vals):
    m = _mesh(E, kind)
    seeds = [3, m.nv // 2][:len(vals)]
    ref, _ = m.solve(seeds, seed_vals=np.abs(vals))
    for sched in (0, 1):
        _same(m.solve(seeds, seed_vals=vals, scheduler=sched)[0], ref)


def test_batch(E):
    ms = [_mesh(E, "tets"), _mesh(E, "triangles")]
    seeds = [[3, 40], [5]]
    b = E.Batch(ms)
    out, _ = b.solve(seeds, seed_vals=[[-0.0, 0.25], [-0.0]])
    for m, s, v, T in zip(ms, seeds, [[0.0, 0.25], [0.0]], out):
        _same(T, m.solve(s, seed_vals=v)[0])
