"""A solve some of whose workgroups gave up waiting (wait_limit_us), but which reached its end, returns every
time.  Before each such solve the same mesh is solved from other sources, so that a stretch of the output
that no workgroup wrote holds wrong times.  Small results (copied through pinned memory) and larger ones,
both element kinds, one and several workgroups per block.  Both solves end at the same fixed point: 2e-6
relative, the tolerance of the batch tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.mark.parametrize("kind,size,stage", [("tets", 20, 0), ("tets", 44, 0), ("tets", 20, 2),
                                             ("triangles", 5, 0), ("triangles", 7, 0), ("triangles", 5, 2)])
def test_complete_after_workgroups_gave_up(E, kind, size, stage):
    m = E.Mesh.kuhn_cube(size, 0.2, seed=5) if kind == "tets" else E.Mesh.icosphere(size)
    m.partition(64)
    seeds, others = [0, m.nv // 2], [m.nv - 1]
    m.solve(seeds, stage_records=stage)
    ref, st = m.solve(seeds, stage_records=stage)
    short = 0
    for part in np.linspace(0.05, 0.75, 15):  # of the solve's own time
        limit = max(1, int(1e3 * part * st["visit_ms"]))
        for rep in range(3):
            m.solve(others, stage_records=stage)
            try:
                T, s = m.solve(seeds, stage_records=stage, wait_limit_us=limit)
            except E.EikError as e:
                assert e.code == E.EIK_ERR_TIMEOUT
                continue
            short += s["abandoned_waits"] > 0
            err = np.max(np.abs(T - ref) / np.maximum(ref, 1e-3))
            assert err <= TOL, "limit %d us: %d waits given up, max rel diff %.3e" % (
                limit, s["abandoned_waits"], err)
    print("%s %d, stage %d: %d of 45 solves ended without some of their workgroups" % (kind, size, stage, short),
          flush=True)
    assert short > 0
