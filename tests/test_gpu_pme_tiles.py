"""The PME passes at the edges of their launch shapes: grids smaller than a
tile and its stencil window, odd lines, every radix, lines longer than a block
of 256 threads holds, planes in one block and planes in lines, wide tiles."""
import numpy as np
import pytest

from oracle import oracle as O
from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu

GRIDS = [
    ((4, 5, 6), 4),        # grid as small as the stencil
    ((8, 6, 9), 6),        # the stencil window wraps onto itself
    ((9, 15, 25), 4),      # odd lines, odd number of line pairs
    ((27, 50, 45), 8),     # radices 9, 10 and 5, a plane in one block
    ((64, 64, 72), 4),     # the largest plane in one block
    ((72, 81, 12), 6),     # planes in lines
    ((8, 6, 1500), 6),     # a z line of more than 256 threads' points
    ((1800, 8, 10), 4),    # an x line of that length
    ((6, 2048, 8), 4),     # a y line of that length
    ((192, 180, 8), 4),    # 8 x 4 tiles
]


@pytest.mark.parametrize("grid,order", GRIDS)
@pytest.mark.parametrize("precision,tol", [(pmx.FP64, 1e-9), (pmx.MIXED, 1e-5)])
def test_reciprocal_forces_on_edge_grids(grid, order, precision, tol):
    s = systems.water_box(n_side=5, box=15.5, seed=3)
    lj = (pmx.SW_C2, 5.0, 7.0)
    pme = dict(rc=7.0, grid=grid, order=order, alpha=0.4)
    f_ref, ec_ref, elj_ref = O.evaluate(s, O.make_spec(5.0, lj=lj, pme=pme))
    ctx = pmx.Context(0)
    try:
        for spread2 in (0, 1):  # the spread's tiles differ
            sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, lj=lj, pme=pme), precision)
            sy.set_tuning(pmx.TUNE_SPREAD_STREAM, spread2)
            f, ec, elj = sy.evaluate(s.pos)
            sy.close()
            rms = np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1)) / np.mean(np.sum(f_ref ** 2, 1)))
            assert rms <= tol
            assert abs(ec - ec_ref) <= (1e-9 if precision == pmx.FP64 else 3e-5) * abs(ec_ref)
    finally:
        ctx.close()
