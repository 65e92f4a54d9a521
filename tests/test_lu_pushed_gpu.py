"""LU's padded sweeps (points hand on their blocks' products) at the sizes
where their geometry changes: rows of the hand-off that end on, just past and
far past a lane's entries, workgroups of every width, steps that do not fill
the load ring, a last workgroup with one row.

Each case runs three iterations against the hyperplane launches, whose points
form the blocks and read their neighbours' rsd and u from global memory.  Both
are FMA arithmetic with sums in another order: a point's value differs by a
few ulp and the sweeps are contractions, so 1e-13 relative to the largest
value bounds both u and rsd with a wide margin (they differ by under 1e-15)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(P, dims, knobs, mode="batched", npb=True):
    N = P.native
    nx, ny, nz = dims
    zones = P.zone_setup(2, 2, 2 * nx, 2 * ny, nz, 1.0, use_round=True)
    ctx = P.Context("LU", zones, 1.0, omega=1.2, npb_exchange=npb)
    for k, v in knobs.items():
        ctx.set_schedule(getattr(N, "SCHED_" + k), v)
    desc = ctx.describe()
    ctx.init_exact()
    ctx.step(3, mode)
    out = ctx.get_all(N.FIELD_U), ctx.get_all(N.FIELD_RHS)
    ctx.close()
    return out, desc


TILES = dict(LU_SWEEP=2)
CASES = [
    # nx, ny, nz, knobs, what describe must show
    ((7, 52, 17), dict(TILES, LU_TILES=4), "groups=8"),      # SJ 51: 255 of 256 entries
    ((6, 53, 16), dict(TILES, LU_TILES=4), "pipelined"),     # SJ 52: 8 entries a lane
    ((5, 104, 9), dict(TILES, LU_TILES=8), "pipelined"),     # SJ 103: past 8 a lane
    ((5, 129, 7), dict(TILES, LU_TILES=3), "pipelined"),     # 128: 10 a lane, exactly
    ((6, 130, 6), dict(TILES, LU_TILES=2), "pipelined"),     # 129: 20
    ((5, 257, 6), dict(TILES, LU_TILES=5), "pipelined"),     # 256: 20, exactly
    ((7, 258, 5), dict(TILES, LU_TILES=4), "pipelined"),     # 257: a batch past them
    ((5, 359, 6), dict(TILES, LU_TILES=2), "pipelined"),     # 358: the longest of one batch
    ((6, 360, 5), dict(TILES, LU_TILES=4), "pipelined"),     # 359: two
    ((5, 449, 5), dict(TILES, LU_TILES=4), "pipelined"),     # 448: the longest row
    ((5, 131, 12), dict(TILES, LU_TILES=4), "pipelined"),    # one row over 128 slots
    ((5, 225, 8), dict(TILES, LU_TILES=7), "nt=256"),        # 224-slot rows
    ((9, 32, 16), dict(TILES, LU_TILES=2), "groups=4"),
    ((10, 32, 17), dict(TILES, LU_TILES=5), "pipelined"),    # 16 rows in 5 tiles
    ((11, 18, 34), dict(TILES, LU_TILES=1), "pipelined"),    # one tile, several workgroups
    ((12, 6, 5), dict(TILES, LU_TILES=8), "pipelined"),      # one row each
    ((5, 5, 5), dict(TILES, LU_TILES=1), "groups=1"),        # the smallest zone
    ((8, 17, 9), dict(LU_SWEEP=1, LU_THREADS=128), "lds-halo"),  # 128 slots in 128 threads
    ((9, 17, 17), dict(LU_SWEEP=1, LU_THREADS=256), "lds-halo"),
    ((6, 33, 17), dict(LU_SWEEP=1, LU_THREADS=512), "lds-halo"),
    ((7, 5, 5), dict(LU_SWEEP=1, LU_THREADS=512), "lds-halo"),   # 16 of 512 threads
]


@pytest.mark.parametrize("dims,knobs,want", CASES)
def test_padded_sweeps_match_hyperplane_launches(gpu, dims, knobs, want):
    (u, r), desc = _run(gpu, dims, knobs)
    assert want in desc, desc
    (u0, r0), _ = _run(gpu, dims, dict(LU_SWEEP=0))
    assert np.abs(u - u0).max() <= 1e-13 * np.abs(u0).max()
    assert np.abs(r - r0).max() <= 1e-13 * np.abs(r0).max()


@pytest.mark.parametrize("dims", [(7, 52, 17), (5, 104, 9), (11, 18, 34), (6, 200, 6), (5, 370, 6)])
def test_handoff_forms_and_modes_agree_bitwise(gpu, dims):
    """Agent-scope and XCD-local hand-offs, per-zone launches and graph
    replays, and both exchanges' planes per form: the same values move."""
    knobs = dict(TILES, LU_TILES=4)
    for npb in (False, True):
        ref, desc = _run(gpu, dims, knobs, npb=npb)
        assert "handoff=xcd-local" in desc, desc
        for kw in (dict(knobs, LU_HANDOFF=0), dict(knobs, LU_TILE_BATCH=1), dict(knobs, LU_TILES=8)):
            got, desc = _run(gpu, dims, kw, mode="graph" if "LU_TILE_BATCH" in kw else "perzone", npb=npb)
            assert ("handoff=agent" if "LU_HANDOFF" in kw else "handoff=xcd-local") in desc, desc
            assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1]), (kw, npb)


@pytest.mark.parametrize("dims", [(12, 145, 26), (12, 216, 6), (60, 257, 10), (60, 301, 6)])
def test_long_rows_are_handed_on_without_a_wait_for_each_entry(gpu, dims):
    """Default schedules of zones with long slot rows are tiles, and take less
    time than the hyperplane launches do (0.4-0.7 of it; 1.02-1.9 with the
    entries past the first 8 a lane loaded one after another)."""
    N = gpu.native
    nx, ny, nz = dims
    best = []
    for knobs in ({}, dict(LU_SWEEP=0)):
        ctx = gpu.Context("LU", gpu.zone_setup(1, 1, nx, ny, nz, 1.0, use_round=True), 1.0, omega=1.2)
        for k, v in knobs.items():
            ctx.set_schedule(getattr(N, "SCHED_" + k), v)
        assert ("pipelined" in ctx.describe()) == (not knobs), ctx.describe()
        ctx.init_exact()
        ctx.step(3, "graph")
        best.append(min(ctx.step(3, "graph") for _ in range(5)))
        ctx.close()
    assert best[0] < best[1], best


def test_rows_too_long_for_one_batch_keep_the_other_sweeps(gpu):
    for ny, tiles in ((359, True), (360, False), (520, False)):
        ctx = gpu.Context("LU", gpu.zone_setup(1, 1, 60, ny, 6, 1.0, use_round=True), 1.0, omega=1.2)
        assert ("pipelined" in ctx.describe()) == tiles, ctx.describe()
        ctx.close()
