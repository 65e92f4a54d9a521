"""SP's line solves staged in LDS: forward steps and gradients against the
one-wave solves, at line counts that leave partial tasks, at the shortest
lines the two-sided elimination takes, and at both sides of the longest that
fit a workgroup's LDS (310 points; longer ones keep the two-wave solve).  And
where they are taken: along y and z long lines leave few waves on a CU, and
from some number of tasks on the other kernels are faster."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (grid, zones, ratio): every direction's shortest lines; uneven odd zones;
# the longest staged lines along x, y and z; lines too long to stage along
# each; staged along x only, transposed in all three
GRIDS = [
    ((6, 6, 6), (1, 1), 1.0),
    ((31, 25, 7), (2, 3), 1.6),
    ((77, 40, 13), (3, 2), 2.5),
    ((310, 7, 6), (1, 1), 1.0),
    ((8, 620, 6), (1, 2), 1.0),
    ((6, 7, 310), (1, 1), 1.0),
    ((311, 7, 6), (1, 1), 1.0),
    ((6, 311, 7), (1, 1), 1.0),
    ((7, 6, 311), (1, 1), 1.0),
    ((84, 160, 84), (1, 1), 1.0),
]


def _context(gpu, grid, zones, ratio, twist, grid_size=0):
    N = gpu.native
    z = gpu.zone_setup(*zones, *grid, ratio)
    ctx = gpu.Context("SP", z, 0.0007)
    ctx.set_schedule(N.SCHED_SOLVE_TWIST, twist)
    ctx.set_schedule(N.SCHED_SOLVE_GRID, grid_size)
    ctx.init_exact()
    u = ctx.get_all(0)
    rng = np.random.default_rng(5)
    ctx.put_all(0, u * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, u.size)))
    return ctx


@pytest.mark.parametrize("grid,zones,ratio", GRIDS)
def test_staged_solves_track_the_one_wave_ones(gpu, grid, zones, ratio):
    """Five steps from a disturbed state.  The eliminations differ in order
    only: a step's update changes by a few ulps of the update's size, so u by
    well under 1e-14 of its own."""
    out = {}
    for twist, mode, size in ((0, "graph", 0), (7, "graph", 0), (7, "perzone", 0), (7, "batched", 3)):
        ctx = _context(gpu, grid, zones, ratio, twist, size)
        ctx.step(5, mode)
        out[twist, mode] = ctx.get_all(0)
        ctx.close()
    ref = out[0, "graph"]
    assert np.isfinite(ref).all()
    assert np.abs(out[7, "graph"] - ref).max() <= 1e-14 * np.abs(ref).max()
    # a line's result does not depend on the launch or the task it falls in
    assert np.array_equal(out[7, "graph"], out[7, "perzone"])
    assert np.array_equal(out[7, "graph"], out[7, "batched"])


@pytest.mark.parametrize("grid,zones,ratio", GRIDS)
def test_staged_adjoint_tracks_the_one_wave_one(gpu, grid, zones, ratio):
    """Gradients of a weighted sum of squares through three steps: 1e-12 of
    the gradient's size, a hundred times the forward's bound for the
    cancellations of the reverse pass."""
    out = []
    for twist in (0, 7):
        ctx = _context(gpu, grid, zones, ratio, twist)
        w = np.random.default_rng(3).random(ctx.size)
        out.append(ctx.adjoint(3, 2, w))
        ctx.close()
    a, b = out
    assert abs(b["loss"] / a["loss"] - 1.0) <= 1e-13
    for k in ("grad_u0", "grad_forcing"):
        assert np.isfinite(a[k]).all()
        assert np.abs(a[k] - b[k]).max() <= 1e-12 * np.abs(a[k]).max(), k


# (grid, zones, ratio), the directions staged (bit d) forward and transposed:
# the classes; long lines with few tasks; one wave per CU and over 4 tasks
# each along y (1121), z's 3 waves and over 8 (2160); the same with over 5
# along y and z; two waves and tasks over 25 per CU; lines too long
ROUTES = [
    ((128, 128, 16), (4, 4), 1.0, 7, 7),
    ((304, 208, 17), (8, 8), 1.0, 7, 7),
    ((310, 7, 6), (1, 1), 1.0, 7, 7),
    ((6, 7, 310), (1, 1), 1.0, 7, 7),
    ((84, 160, 84), (1, 1), 1.0, 1, 7),
    ((100, 160, 160), (1, 1), 1.0, 1, 1),
    ((160, 128, 160), (2, 2), 1.0, 3, 3),
    ((140, 300, 140), (2, 2), 1.0, 7, 3),
    ((6, 311, 7), (1, 1), 1.0, 5, 5),
]


@pytest.mark.parametrize("grid,zones,ratio,forward,transposed", ROUTES)
def test_staged_where_it_is_the_faster_one(gpu, grid, zones, ratio, forward, transposed):
    z = gpu.zone_setup(*zones, *grid, ratio)
    ctx = gpu.Context("SP", z, 0.0007)
    assert "staged=%d/%d" % (forward, transposed) in ctx.describe(), ctx.describe()
    ctx.close()
    ctx = gpu.Context("SP", z, 0.0007, strict=True)
    assert "staged=0/0" in ctx.describe()
    ctx.close()
