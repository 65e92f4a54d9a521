"""BT's columns line solve against the two-sided one-lane-per-line solve, at
the half lengths where its rows move between registers (4), LDS (7 more) and
the spill, with even and odd rows (an odd line's lower half starts on a dummy
row), partial tasks, and every launch form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (grid, zones, ratio): lines of 5 (the shortest), 8-13, 23-27 and 60 points
# in each direction, one line more or less than a task's five, uneven zones
GRIDS = [
    ((5, 5, 5), (1, 1), 1.0),
    ((8, 9, 10), (1, 1), 1.0),
    ((11, 12, 13), (1, 1), 1.0),
    ((13, 24, 23), (1, 1), 1.0),
    ((25, 13, 26), (1, 1), 1.0),
    ((27, 60, 8), (1, 1), 1.0),
    ((60, 8, 27), (1, 1), 1.0),
    ((9, 8, 60), (1, 1), 1.0),
    ((75, 53, 11), (3, 2), 2.5),
]


@pytest.mark.parametrize("grid,zones,ratio", GRIDS)
def test_columns_solve_tracks_the_two_sided_one(gpu, grid, zones, ratio):
    """Five steps from a disturbed state.  The eliminations differ in order
    only: a step's update changes by some ulps of the update's size, so u by
    well under 1e-14 of its own."""
    N = gpu.native
    out = {}
    for cols, mode, size in ((0, "graph", 0), (7, "graph", 0), (7, "perzone", 0), (7, "batched", 3)):
        ctx = gpu.Context("BT", gpu.zone_setup(*zones, *grid, ratio), 0.0003)
        ctx.set_schedule(N.SCHED_SOLVE_TWIST, 7)
        ctx.set_schedule(N.SCHED_SOLVE_ROWS, 0)
        ctx.set_schedule(N.SCHED_SOLVE_COLS, cols)
        ctx.set_schedule(N.SCHED_SOLVE_GRID, size)
        ctx.init_exact()
        u = ctx.get_all(0)
        rng = np.random.default_rng(5)
        ctx.put_all(0, u * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, u.size)))
        ctx.step(5, mode)
        out[cols, mode] = ctx.get_all(0)
        ctx.close()
    ref = out[0, "graph"]
    assert np.isfinite(ref).all()
    assert np.abs(out[7, "graph"] - ref).max() <= 1e-14 * np.abs(ref).max()
    # a line's result does not depend on the launch or the task it falls in
    assert np.array_equal(out[7, "graph"], out[7, "perzone"])
    assert np.array_equal(out[7, "graph"], out[7, "batched"])


def test_dummy_rows_drop_the_boundary_rhs(gpu):
    """The dummy row of an odd line reads the boundary's rhs and drops it:
    NaN there reaches nothing."""
    N = gpu.native
    res = []
    for poison in (False, True):
        ctx = gpu.Context("BT", gpu.zone_setup(1, 1, 9, 11, 13, 1.0), 0.0003)
        ctx.init_exact()
        if poison:
            r = np.zeros((13, 11, 9, 5))
            r[[0, -1]] = r[:, [0, -1]] = r[:, :, [0, -1]] = np.nan
            ctx.put_dense(0, N.FIELD_RHS, r)
        ctx.step(2, "graph")
        res.append(ctx.get_all(0))
        ctx.close()
    assert np.isfinite(res[0]).all() and np.array_equal(res[0], res[1])


def test_columns_knob_is_validated_and_rows_replaces_it(gpu):
    N = gpu.native
    ctx = gpu.Context("BT", gpu.zone_setup(1, 1, 9, 11, 13, 1.0), 0.0003)
    assert "cols=7" in ctx.describe()
    with pytest.raises(gpu.NpbmzError, match="columns"):
        ctx.set_schedule(N.SCHED_SOLVE_COLS, 8)
    ctx.set_schedule(N.SCHED_SOLVE_ROWS, 7)
    assert "cols=0" in ctx.describe()
    ctx.close()
    ctx = gpu.Context("SP", gpu.zone_setup(1, 1, 9, 11, 13, 1.0), 0.0003)
    with pytest.raises(gpu.NpbmzError):
        ctx.set_schedule(N.SCHED_SOLVE_COLS, 7)
    ctx.close()


@pytest.mark.parametrize("grid,zones,ratio", GRIDS)
def test_columns_adjoint_tracks_the_two_sided_one(gpu, grid, zones, ratio):
    """Gradients of a weighted sum of squares through three steps, forward
    and transposed solves by columns against both two-sided: 1e-12 of the
    gradient's size, a hundred times the forward's bound for the
    cancellations of the reverse pass."""
    N = gpu.native
    out = []
    for cols, size in ((0, 0), (7, 0), (7, 3)):
        ctx = gpu.Context("BT", gpu.zone_setup(*zones, *grid, ratio), 0.0003)
        ctx.set_schedule(N.SCHED_SOLVE_ROWS, 0)
        ctx.set_schedule(N.SCHED_SOLVE_COLS, cols)
        ctx.set_schedule(N.SCHED_SOLVE_GRID, size)
        ctx.init_exact()
        u = ctx.get_all(0)
        rng = np.random.default_rng(5)
        ctx.put_all(0, u * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, u.size)))
        out.append(ctx.adjoint(3, 2, np.random.default_rng(3).random(ctx.size)))
        ctx.close()
    a, b, c = out
    assert abs(b["loss"] / a["loss"] - 1.0) <= 1e-13
    for k in ("grad_u0", "grad_forcing"):
        assert np.isfinite(a[k]).all()
        assert np.abs(a[k] - b[k]).max() <= 1e-12 * np.abs(a[k]).max(), k
        assert np.array_equal(b[k], c[k]), k


# (grid, zones, ratio), the directions solved by columns (bit d) forward and
# transposed: the classes and a grid between them; just over one round of
# columns waves along x, within one of rows waves, with lines of one length
# and uneven ones; long lines whose spill
# leaves the last-level cache; the same along x only, short lines along y, and
# many medium ones along z
ROUTES = [
    ("S", 7, 7), ("A", 7, 7), ("B", 7, 7), ("C", 7, 7),
    (((131, 97, 23), (3, 2), 2.2), 7, 7),
    (((80, 112, 112), (1, 1), 1.0), 6, 7),
    (((154, 233, 27), (2, 8), 4.43), 7, 7),
    (((200, 200, 200), (1, 1), 1.0), 0, 1),
    (((400, 40, 64), (1, 1), 1.0), 6, 3),
]


@pytest.mark.parametrize("problem,forward,transposed", ROUTES)
def test_columns_where_they_are_the_faster_ones(gpu, problem, forward, transposed):
    if isinstance(problem, str):
        z = gpu.zones_for("BT", problem)[0]
    else:
        grid, zones, ratio = problem
        z = gpu.zone_setup(*zones, *grid, ratio)
    ctx = gpu.Context("BT", z, 0.0003)
    assert "cols=%d/%d" % (forward, transposed) in ctx.describe(), ctx.describe()
    ctx.close()
    ctx = gpu.Context("BT", z, 0.0003, strict=True)
    assert "cols=0/0" in ctx.describe()
    ctx.close()


def test_directions_on_different_solves_agree(gpu):
    """A default schedule with rows along x and columns along y and z, and
    with columns and the two-sided solve transposed, against the two-sided
    solve in all (the bounds of the tests above; a step small enough that
    noise on 400 points along x decays)."""
    N = gpu.native
    for grid in ((80, 112, 112), (400, 40, 64)):
        u, g = [], []
        for default in (False, True):
            ctx = gpu.Context("BT", gpu.zone_setup(1, 1, *grid, 1.0), 0.00003)
            if not default:
                ctx.set_schedule(N.SCHED_SOLVE_ROWS, 0)
            ctx.init_exact()
            u0 = ctx.get_all(0)
            rng = np.random.default_rng(5)
            ctx.put_all(0, u0 * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, u0.size)))
            g.append(ctx.adjoint(2, 1, np.random.default_rng(3).random(ctx.size)))
            ctx.step(3, "graph")
            u.append(ctx.get_all(0))
            ctx.close()
        assert np.abs(u[1] - u[0]).max() <= 1e-14 * np.abs(u[0]).max()
        for k in ("grad_u0", "grad_forcing"):
            assert np.abs(g[1][k] - g[0][k]).max() <= 1e-12 * np.abs(g[0][k]).max(), k
