"""The synchronous scheduler's visits at the block sizes where their shape changes (items or elements per
thread, workgroups of 256, 512 and 1,024 threads, blocks too large for registers), its lists of
active blocks and its history: the converged times equal the persistent scheduler's (2e-6 relative, the
tolerance of the batch tests: both end in the same fixed point), the last snapshot is the result,
and every snapshot is at most the one before."""
import numpy as np
import pytest

from conftest import center_vertex, lognormal_mult

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.mark.parametrize("vpb", [1, 7, 64, 100, 150, 190, 300, 420])
@pytest.mark.parametrize("kind", ["tets", "triangles"])
def test_shapes_and_history(E, kind, vpb):
    if kind == "tets":
        m = E.Mesh.kuhn_cube(11, 0.2, seed=vpb)
        m.set_speed(lognormal_mult(m.info()["nelem"], vpb))
        seeds = np.array([center_vertex(11), 0], np.int32)
    else:
        m = E.Mesh.icosphere(4)
        m.set_speed(lognormal_mult(m.info()["nelem"], vpb))
        seeds = np.array([5, 1300], np.int32)
    m.partition(vpb)
    print("%s, %d vertices per block, %d blocks" % (kind, vpb, m.info()["nblocks"]), flush=True)
    ref, _ = m.solve(seeds)
    for stage in (0, 2):  # element data in registers where the blocks fit; records read from memory
        T, st = m.solve(seeds, scheduler=E.SCHED_SYNC, record_history=1, stage_records=stage)
        err = np.max(np.abs(T - ref) / np.maximum(ref, 1e-3))
        print("  stage %d: %d iterations, max rel diff %.3e" % (stage, st["outer_iterations"], err), flush=True)
        assert err <= TOL
        assert st["history_len"] == st["outer_iterations"] > 0
        before = np.full(m.nv, np.inf, np.float32)
        for k in range(st["history_len"]):
            snap = m.history(k)
            assert np.all(snap <= before)
            before = snap
        np.testing.assert_array_equal(before, T)
    # a cap on the iterations ends the solve there
    _, st = m.solve(seeds, scheduler=E.SCHED_SYNC, record_history=1, max_iterations=2)
    assert 1 <= st["outer_iterations"] <= 2 and st["history_len"] == st["outer_iterations"]
