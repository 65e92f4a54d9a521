"""Field transfers in each of their forms: the zone's own shape (one block),
rows of contiguous points inside a padded array, and points whose components
lie apart.  Every form moves the same values and leaves the padding alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bench", ["SP", "LU"])
@pytest.mark.parametrize(
    "order,pads",
    [  # elements below and above the grid on the axes m, i, j, k
        (0, ((0, 0), (0, 0), (0, 0), (0, 0))),
        (0, ((0, 0), (2, 1), (0, 3), (1, 0))),
        (0, ((0, 0), (0, 0), (0, 0), (0, 2))),
        (0, ((1, 2), (0, 0), (1, 0), (0, 0))),
        (1, ((0, 0), (0, 0), (0, 0), (0, 0))),
        (1, ((2, 1), (1, 2), (0, 1), (3, 0))),
    ],
)
def test_every_transfer_form_moves_the_same_values(gpu, bench, order, pads):
    zones = gpu.zone_setup(2, 1, 20, 9, 7, 1.0, use_round=bench == "LU")
    org = 1 if bench == "LU" else 0
    with gpu.Context(bench, zones, 0.001, omega=1.2) as ctx:
        z = 1
        nx, ny, nz = (int(a[z]) for a in (zones.nx, zones.ny, zones.nz))
        vals = np.random.default_rng(1).standard_normal((nz, ny, nx, 5))
        # bounds of the axes m, i, j, k, then in the order they are stored
        first, count = (1, org, org, org), (5, nx, ny, nz)
        lo = [f - p for f, (p, _) in zip(first, pads)]
        hi = [f + n - 1 + p for f, n, (_, p) in zip(first, count, pads)]
        perm = [0, 1, 2, 3] if order == 0 else [1, 2, 3, 0]
        shape = [hi[a] - lo[a] + 1 for a in perm][::-1]
        inner = tuple(slice(pads[a][0], pads[a][0] + count[a]) for a in perm)[::-1]
        body = vals if order == 0 else np.moveaxis(vals, -1, 0)
        host = np.full(shape, 7.0)
        host[inner] = body
        lo, hi = [lo[a] for a in perm], [hi[a] for a in perm]
        ctx.put_field(z, 0, host, lo, hi, order)
        assert np.array_equal(ctx.get_all(0)[-vals.size:], vals.ravel())
        back = np.full(shape, -3.0)
        ctx.get_field(z, 0, back, lo, hi, order)
        assert np.array_equal(back[inner], body)
        back[inner] = -3.0
        assert (back == -3.0).all()
