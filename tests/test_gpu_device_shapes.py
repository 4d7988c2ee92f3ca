"""Mixed results do not depend on the number of compute units of the device.
The context's count (the second int of pmx_ctx) is set to that of a smaller
and of a larger device before the system is made; the launches then have
other grids, on the same device."""
import ctypes as C

import numpy as np
import pytest

from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(192, 180, 8), (128, 128, 16), (64, 72, 64)])
def test_mixed_results_do_not_depend_on_the_compute_units(grid):
    s = systems.water_box(n_side=5, box=15.5, seed=3)
    spec = pmx.ForceSpec(5.0, lj=(pmx.SW_C2, 5.0, 7.0), pme=dict(rc=7.0, grid=grid, order=4, alpha=0.4))
    out = []
    for cus in (None, 32, 128, 512):
        ctx = pmx.Context(0)
        try:
            words = (C.c_int * 2).from_address(ctx.h.value)
            assert words[0] == 0 and 32 <= words[1] <= 256
            words[1] = cus or words[1]
            sy = pmx.System(ctx, s, spec, pmx.MIXED)
            out.append(sy.evaluate(s.pos))
            sy.close()
        finally:
            ctx.close()
    for f, ec, elj in out[1:]:
        assert np.array_equal(f, out[0][0]) and (ec, elj) == out[0][1:]
