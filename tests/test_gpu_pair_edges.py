"""The mixed pair kernel at its edges: less than one cluster, partly filled
superclusters, one and unequal cutoffs, LJ tables in LDS and beyond it,
excluded and scaled pairs, a box in which entries need the per-pair image."""
import numpy as np
import pytest

from oracle import oracle as O
from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu


def _gas(n, box, ntypes, seed):
    """n atoms no closer than 1.8 A, random types and charges, every 5th pair
    of neighbours in the list excluded, every 7th scaled."""
    rng = np.random.default_rng(seed)
    pos = []
    while len(pos) < n:
        p = rng.uniform(0, box, 3)
        if pos:
            d = np.array(pos) - p
            d -= box * np.rint(d / box)
            if np.min(np.sum(d * d, 1)) < 1.8 ** 2:
                continue
        pos.append(p)
    eps, rmin2 = rng.uniform(0.05, 0.2, ntypes), rng.uniform(0.6, 1.0, ntypes)
    pairs = [(a, a + 1, 1) for a in range(0, n - 1, 5)] + [(a, a + 2, 2) for a in range(0, n - 2, 7)]
    return systems.MolSystem(
        name="gas", pos=np.array(pos), charge=rng.uniform(-9, 9, n), atype=rng.integers(0, ntypes, n).astype(np.int32),
        molecule=np.zeros(n, np.int32), mass=np.ones(n),
        lj=systems.charmm_table(list(eps), list(rmin2), list(0.5 * eps), list(0.9 * rmin2)), box=np.array([box] * 3),
        origin=np.zeros(3), bonds=np.zeros((0, 2), np.int32), bond_par=np.zeros((0, 2)),
        angles=np.zeros((0, 3), np.int32), angle_par=np.zeros((0, 2)),
        exclusions=np.array(sorted(set(pairs)), np.int32).reshape(-1, 3), csf=0.4)


@pytest.mark.parametrize("n,box,ntypes,lj_rc,c_rc", [
    (1, 16.0, 1, 7.0, 7.0), (2, 16.0, 2, 7.0, 7.0), (7, 12.0, 3, 5.9, 5.9), (9, 12.0, 16, 5.0, 5.9),
    (63, 14.0, 16, 6.5, 6.5), (64, 14.0, 4, 6.9, 5.0), (65, 14.1, 17, 6.5, 6.5), (130, 15.0, 40, 6.0, 7.4),
    (517, 24.0, 16, 8.0, 8.0), (1801, 32.0, 2, 9.0, 7.0)])
@pytest.mark.parametrize("coul", ["pme", "c1", "c2"])
def test_mixed_forces_at_pair_kernel_edges(n, box, ntypes, lj_rc, c_rc, coul):
    s = _gas(n, box, ntypes, n)
    kw = dict(lj=(pmx.SW_C2, lj_rc - 2.0, lj_rc))
    if coul == "pme":
        # the real-space part: the grid's FP32 error on charges this large is another matter
        kw["pme"] = dict(rc=c_rc, grid=(16, 16, 18), order=4, alpha=0.4, terms=pmx.PME_REAL, recip=False, corr=False)
    else:
        kw["coul"] = (pmx.SW_C1 if coul == "c1" else pmx.SW_C2, c_rc - 1.5, c_rc)
    f_ref, ec_ref, elj_ref = O.evaluate(s, O.make_spec(5.0, **kw))
    ctx = pmx.Context(0)
    try:
        for prune in (1, 0):
            sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, **kw), pmx.MIXED)
            sy.set_tuning(pmx.TUNE_LIST_PRUNE, prune)
            f, ec, elj = sy.evaluate(s.pos)
            sy.close()
            scale = np.sqrt(np.mean(np.sum(f_ref ** 2, 1)))
            assert np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1))) <= 1e-5 * scale + 1e-9
            size = np.abs(s.charge).sum() ** 2 / max(n, 1) + 1.0  # of single terms; FP32 keeps 1e-6 of them
            assert abs(ec - ec_ref) <= 1e-6 * size + 3e-5 * abs(ec_ref)
            assert abs(elj - elj_ref) <= 1e-6 * size + 3e-5 * abs(elj_ref)
    finally:
        ctx.close()
