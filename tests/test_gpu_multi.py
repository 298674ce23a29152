"""The visits of a multi-solve launch at the sizes where their shape changes: register-resident blocks
of each workgroup size, launches of both element kinds in one kernel, one and few workgroups, a
kind whose blocks do not fit, and so many tet blocks that the launch reads its records from
memory.  Every solve equals the same mesh solved alone with its speeds set directly, at the tolerance
of the other batch tests (2e-6 relative)."""
import numpy as np
import pytest

from conftest import center_vertex, lognormal_mult

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _metrics(nf, seed):
    rng = np.random.default_rng(seed)
    th, k = rng.uniform(0, np.pi, nf), rng.uniform(1, 10, nf)
    return np.stack([np.cos(th) ** 2 + k * np.sin(th) ** 2, (1 - k) * np.cos(th) * np.sin(th),
                     np.sin(th) ** 2 + k * np.cos(th) ** 2], 1).astype(np.float32)


def _same(T, ref):
    err = np.max(np.abs(T - ref) / np.maximum(ref, 1e-3))
    print("  max rel diff vs alone %.3e" % err, flush=True)
    assert err <= TOL


# vertices per block: workgroups of 256 threads, 512, 1,024 (the larger of the two kinds), and beyond
# what a tet block may have; workgroups 0: as many as fit
@pytest.mark.parametrize("vpb,workgroups", [(1, 0), (64, 0), (64, 1), (64, 3), (150, 0), (190, 2),
                                            (260, 0), (420, 1)])
@pytest.mark.parametrize("kinds", ["both", "tets", "triangles"])
def test_shapes_with_factors(E, vpb, workgroups, kinds):
    n = 11
    tets = lambda: E.Mesh.kuhn_cube(n, 0.2, seed=vpb)
    metric = _metrics(E.Mesh.icosphere(4).info()["nelem"], vpb)
    meshes, seeds, refs, factors = [], [], [], []
    if kinds != "triangles":
        m, c = tets(), tets()
        f = lognormal_mult(m.info()["nelem"], vpb + 1)
        c.set_speed(f)
        meshes += [m, m]
        refs += [m, c]
        factors += [None, f]
        seeds += [[center_vertex(n)], [0, m.nv - 1]]
    if kinds != "tets":
        t, c = E.Mesh.icosphere(4), E.Mesh.icosphere(4)
        f = lognormal_mult(t.info()["nelem"], vpb + 2)
        t.set_metric_tri(metric)
        c.set_metric_tri((metric * f[:, None]).astype(np.float32))
        meshes += [t, t]
        refs += [t, c]
        factors += [None, f]
        seeds += [[7], [5, 1300]]
    for m in meshes + refs:
        if m.info()["nblocks"] == 0:
            m.partition(vpb)
    b = E.Batch(meshes)
    for i, f in enumerate(factors):
        if f is not None:
            b.set_factors(i, f)
    print("%s, %d vertices per block, %s" % (kinds, vpb, b.info()), flush=True)
    for rep in range(2):  # the second from the captured graph
        Ts, _ = b.solve(seeds, workgroups=workgroups)
        for T, m, s in zip(Ts, refs, seeds):
            _same(T, m.solve(s)[0])


def test_busy_launch(E):
    """More than 24 one-vertex (too small to fill a CU) tet blocks for each of the at most 1,024 workgroups of 256 threads that
    are resident: records read from memory; one solve fewer than that: register-resident."""
    m = E.Mesh.kuhn_cube(11, 0.2, seed=3)
    m.partition(1)
    most = 24 * 1024 // m.nv + 1
    for solves in (most - 1, most):
        seeds = [[(37 * i) % m.nv] for i in range(solves)]
        b = E.Batch([m] * solves)
        print("%d solves, %s" % (solves, b.info()), flush=True)
        Ts, _ = b.solve(seeds)
        for i in (0, solves // 2, solves - 1):
            _same(Ts[i], m.solve(seeds[i])[0])


@pytest.mark.parametrize("vpb", [188, 192])
def test_full_queue(E, vpb):
    """Blocks whose queue holds fewer pairs than they have, so that two fit a CU, with every vertex a
    source: the first sweep selects most pairs of a block.  As many pairs as a queue turns away are
    selected again.  Against the synchronous scheduler, whose queue holds them all."""
    m = E.Mesh.kuhn_cube(24, 0.2, seed=vpb)
    m.partition(vpb)
    rng = np.random.default_rng(vpb)
    seeds = np.arange(m.nv, dtype=np.int32)
    values = rng.uniform(0.0, 4.0, m.nv).astype(np.float32)
    ref, _ = m.solve(seeds, values, scheduler=E.SCHED_SYNC)
    T, _ = m.solve(seeds, values)
    _same(T, ref)
    Ts, _ = E.Batch([m, m]).solve([seeds, seeds], [values, values])
    _same(Ts[0], ref)
    _same(Ts[1], ref)
