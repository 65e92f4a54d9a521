"""A closed context gives its device memory back: free memory is the same
before and after many contexts were made, used and closed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("bench", ["BT", "SP", "LU"])
def test_closed_contexts_leave_no_device_memory(gpu, bench):
    """Class B contexts, whose task tables alone take some 100 KB each; the
    first ones warm up what the runtime keeps (code objects, pools)."""
    zones, p = gpu.zones_for(bench, "B")

    def use():
        with gpu.Context(bench, zones, p.dt, omega=1.2) as ctx:
            ctx.init_exact()
            ctx.step(1, "graph")
        with gpu.Context(bench, gpu.zone_setup(2, 2, 24, 24, 8, 1.0), p.dt, omega=1.2) as ctx:
            ctx.init_exact()
            ctx.adjoint(1, 1, np.ones(ctx.size))

    for _ in range(3):
        use()
    before = _free_bytes()
    for _ in range(40):
        use()
    assert before - _free_bytes() < 1 << 20
