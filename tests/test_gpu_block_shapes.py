"""Every workgroup shape of the register-resident visits, each reached by a block size that the layout is
checked to belong to: persistent and one-launch-per-iteration single solves and batches, against the same
solve with the records read from memory (the general kernel, itself compared with the oracle), at 2e-6
relative, the tolerance of the batch tests; and visits whose work-item queue is too small for what a sweep
selects."""
import numpy as np
import pytest

from conftest import center_vertex, lognormal_mult

pytestmark = pytest.mark.gpu

TOL = 2e-6
MEMORY = 2
CUS = 256


def _same(T, ref, what):
    err = np.max(np.abs(T - ref) / np.maximum(ref, 1e-3))
    print("  %s: max rel diff %.3e" % (what, err), flush=True)
    assert err <= TOL


def _items(lay):
    """Per block: (element, corner) pairs that a visit may update (owned corners, of a virtual face the first)."""
    b, e = lay["blocks"], lay["elems"]
    out = []
    for d in b:
        r = e[d[5]:d[5] + d[6]]
        own = r["v"] < d[1]
        if lay["dim"] == 2:
            own &= ((r["mask"][:, None] >> np.arange(3)) & 1).astype(bool)
        out.append(int(own.sum()))
    return np.array(out)


def _shape(lay):
    """(items or elements per thread, threads) of the resident visits of a single solve; None: too large."""
    own, elem, nb = lay["blocks"][:, 1].max(), lay["blocks"][:, 6].max(), lay["nblocks"]
    if lay["dim"] == 3:
        shapes, need = [(2, 512), (4, 256), (6, 256), (6, 512), (4, 1024)], elem
        if nb > 2 * CUS:
            shapes = shapes[1:]
    else:
        shapes, need = [(1, 256), (1, 512), (2, 512), (4, 512), (4, 1024)], _items(lay).max()
        if lay["max_local"] > 1024:
            return None
    for n, bt in shapes:
        if need <= n * bt and own <= bt:
            lds = 12 * ((lay["max_local"] + 3) & ~3)
            if lay["dim"] == 3:  # (a queue for all pairs; in 512 threads it may be smaller)
                lds += 32 * int(elem) + 2 * int(_items(lay).max())
            return (n, bt) if lds <= 163840 - 1024 else None
    return None


def _queue_bound(lay):
    """No queue of a tet block in 512 threads holds more pairs, where two workgroups are to share a CU."""
    stride = (lay["max_local"] + 3) & ~3
    return (163840 // 2 - 12 * stride - 32 * int(lay["blocks"][:, 6].max())) // 2


@pytest.mark.parametrize("n,vpb,shape", [(11, 64, (2, 512)), (34, 64, (4, 256)), (11, 192, (6, 256)),
                                         (24, 192, (6, 512)), (24, 300, (6, 512)), (20, 420, (4, 1024)),
                                         (24, 450, None), (24, 600, None)])
def test_tets(E, n, vpb, shape):
    m = E.Mesh.kuhn_cube(n, 0.2, seed=1)
    mult = lognormal_mult(m.info()["nelem"], vpb)
    m.set_speed(mult)
    m.partition(vpb)
    lay = m.layout()
    print("%d^3, %d vertices per block: %d blocks, up to %d tets" % (n, vpb, lay["nblocks"],
                                                                    lay["blocks"][:, 6].max()), flush=True)
    assert _shape(lay) == shape
    seeds = [center_vertex(n), 0]
    ref, _ = m.solve(seeds, stage_records=MEMORY)
    T, st = m.solve(seeds)
    _same(T, ref, "persistent")
    # a re-run reads no element data where it stays on the CU; records beyond the LDS stay only in registers
    if 48 * lay["blocks"][:, 6].max() > 163840:
        assert (st["algo_bytes_loaded"] < st["algo_bytes"]) == (shape is not None)
    _same(m.solve(seeds, scheduler=E.SCHED_SYNC)[0], ref, "per iteration")
    b = E.Batch([m, m])
    for T in b.solve([seeds, seeds])[0]:
        _same(T, ref, "batch")
    b.close()


@pytest.mark.parametrize("vpb,shape", [(30, (1, 256)), (64, (1, 512)), (130, (2, 512)), (300, (4, 512)),
                                       (600, (4, 1024)), (800, None)])
def test_triangles(E, vpb, shape):
    m = E.Mesh.icosphere(5)
    rng = np.random.default_rng(vpb)
    m.set_speed(np.exp(rng.normal(0.0, 0.5, m.info()["nelem"])).astype(np.float32))
    m.partition(vpb)
    lay = m.layout()
    print("%d vertices per block: %d blocks, up to %d corners" % (vpb, lay["nblocks"], _items(lay).max()), flush=True)
    assert _shape(lay) == shape
    seeds = [5, 1300]
    ref, _ = m.solve(seeds, stage_records=MEMORY)
    _same(m.solve(seeds)[0], ref, "persistent")
    _same(m.solve(seeds, scheduler=E.SCHED_SYNC)[0], ref, "per iteration")
    b = E.Batch([m, m])
    for T in b.solve([seeds, seeds])[0]:
        _same(T, ref, "batch")
    b.close()


@pytest.mark.parametrize("vpb", [200, 205])
def test_sweeps_that_select_more_than_the_queue_holds(E, vpb):
    """Every vertex a source with a time of its own: the first sweep of a block selects most of its pairs."""
    m = E.Mesh.kuhn_cube(28, 0.2, seed=1)
    m.partition(vpb)
    lay = m.layout()
    assert _shape(lay) == (6, 512)
    rng = np.random.default_rng(vpb)
    values = rng.uniform(0.0, 4.0, m.nv).astype(np.float32)
    # what the first sweep of each block selects: owned corners above the smallest other time plus their height
    T = values[lay["perm"]]
    most = 0
    for d in lay["blocks"]:
        r = lay["elems"][d[5]:d[5] + d[6]]
        ids = np.concatenate([np.arange(d[0], d[0] + d[1]), lay["halo"][d[3]:d[3] + d[4]]])
        t = T[ids[r["v"]]]
        least = np.stack([np.delete(t, k, 1).min(1) for k in range(4)], 1)
        most = max(most, int(((r["v"] < d[1]) & (t > 1.001 * (least + r["H"]))).sum()))
    bound, items = _queue_bound(lay), int(_items(lay).max())
    print("%d vertices per block: %d pairs, %d selected, a queue of at most %d" % (vpb, items, most, bound), flush=True)
    assert lay["blocks"][:, 6].max() <= bound < most <= items
    seeds = np.arange(m.nv, dtype=np.int32)
    ref, _ = m.solve(seeds, values, stage_records=MEMORY)
    _same(m.solve(seeds, values)[0], ref, "persistent")
    _same(m.solve(seeds, values, scheduler=E.SCHED_SYNC)[0], ref, "per iteration")
    b = E.Batch([m, m])
    for T in b.solve([seeds, seeds], [values, values])[0]:
        _same(T, ref, "batch")
    b.close()
