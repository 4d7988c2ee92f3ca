"""The FP64 pair kernel at the edges of test_gpu_pair_edges: partial clusters,
unequal cutoffs, LJ tables in LDS and beyond it, every kind of Coulomb."""
import numpy as np
import pytest
from test_gpu_pair_edges import _gas

from oracle import oracle as O
from protomol3_amd import pmx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,ntypes,lj_rc,c_rc", [
    (1, 16.0, 1, 7.0, 7.0), (2, 16.0, 2, 7.0, 7.0), (7, 12.0, 3, 5.9, 5.9), (9, 12.0, 16, 5.0, 5.9),
    (63, 14.0, 16, 6.5, 6.5), (64, 14.0, 4, 6.9, 5.0), (65, 14.1, 17, 6.5, 6.5), (130, 15.0, 40, 6.0, 7.4),
    (517, 24.0, 16, 8.0, 8.0), (1801, 32.0, 2, 9.0, 7.0)])
@pytest.mark.parametrize("coul", ["pme", "c1", "c2"])
def test_fp64_forces_at_pair_kernel_edges(n, box, ntypes, lj_rc, c_rc, coul):
    s = _gas(n, box, ntypes, n)
    kw = dict(lj=(pmx.SW_C2, lj_rc - 2.0, lj_rc))
    if coul == "pme":
        kw["pme"] = dict(rc=c_rc, grid=(16, 16, 18), order=4, alpha=0.4, terms=pmx.PME_REAL, recip=False, corr=False)
    else:
        kw["coul"] = (pmx.SW_C1 if coul == "c1" else pmx.SW_C2, c_rc - 1.5, c_rc)
    f_ref, ec_ref, elj_ref = O.evaluate(s, O.make_spec(5.0, **kw))
    # some tens of roundings (1e-16) a pair, and sums over hundreds of pairs
    # that cancel to a hundredth or less of their size: 1e-11
    scale = np.sqrt(np.mean(np.sum(f_ref ** 2, 1)))
    size = np.abs(s.charge).sum() ** 2 / max(n, 1) + abs(ec_ref) + abs(elj_ref) + 1.0
    ctx = pmx.Context(0)
    try:
        for prune in (1, 0):
            sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, **kw), pmx.FP64)
            sy.set_tuning(pmx.TUNE_LIST_PRUNE, prune)
            f, ec, elj = sy.evaluate(s.pos)
            sy.close()
            assert np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1))) <= 1e-11 * scale
            assert abs(ec - ec_ref) <= 1e-11 * size and abs(elj - elj_ref) <= 1e-11 * size
    finally:
        ctx.close()
