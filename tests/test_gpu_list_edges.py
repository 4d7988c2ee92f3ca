"""The list at its edges: a drop in a large box (cell bins of many atoms that
continue from one supercluster to the next), more masked entries of a
supercluster than are made together, an atom with excluded partners beyond
those its threads hold, empty space between, atoms in any input order."""
import numpy as np
import pytest

from oracle import oracle as O
from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu


def _drop(n, box, spread, hub, seed):
    """n atoms on a jittered grid in one corner region, in random order; each
    excluded from the next `spread`, the first from `hub` others."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = rng.permutation(2.0 * g + rng.uniform(-0.3, 0.3, (n, 3)) + box - 9.0)  # across the boundary
    ex = {(a, b): 1 + (a + b) % 2 for a in range(n) for b in range(a + 1, min(n, a + 1 + spread))}
    ex.update({(0, b): 1 for b in range(1, min(n, hub + 1))})
    return systems.MolSystem(
        name="drop", pos=pos, charge=rng.uniform(-5, 5, n), atype=np.zeros(n, np.int32),
        molecule=np.zeros(n, np.int32), mass=np.ones(n),
        lj=systems.charmm_table([0.1], [0.8], [0.05], [0.7]), box=np.array([box] * 3), origin=np.zeros(3),
        bonds=np.zeros((0, 2), np.int32), bond_par=np.zeros((0, 2)), angles=np.zeros((0, 3), np.int32),
        angle_par=np.zeros((0, 2)),
        exclusions=np.array([(*p, c) for p, c in sorted(ex.items())], np.int32).reshape(-1, 3), csf=0.4)


@pytest.mark.parametrize("precision", [pmx.FP64, pmx.MIXED])
@pytest.mark.parametrize("n,box,spread,hub", [(1, 20.0, 0, 0), (5, 20.0, 4, 4), (65, 24.0, 9, 0), (343, 90.0, 0, 342),
                                              (700, 60.0, 30, 0), (1331, 30.0, 2, 900), (1500, 120.0, 12, 40)])
def test_pairs_and_forces_at_list_edges(n, box, spread, hub, precision):
    s = _drop(n, box, spread, hub, n)
    kw = dict(lj=(pmx.SW_C2, 6.0, 7.5), coul=(pmx.SW_C1, 0.0, 7.5))
    f_ref, ec_ref, elj_ref = O.evaluate(s, O.make_spec(5.0, **kw))
    ref = O.pairs_bruteforce(s, 7.5)
    ctx = pmx.Context(0)
    try:
        sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, **kw), precision)
        f, ec, elj = sy.evaluate(s.pos, flags=pmx.EVAL_PAIRSTATS)
        npairs, phash = sy.pair_stats()
        sy.close()
    finally:
        ctx.close()
    assert npairs == len(ref) and phash == pmx.pair_hash_set(ref)
    rel = 1e-12 if precision == pmx.FP64 else 1e-5  # FP64 sums of at most 200 terms; FP32 pair terms
    scale = np.sqrt(np.mean(np.sum(f_ref ** 2, 1)))
    assert np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1))) <= rel * scale + 1e-9
    size = np.abs(s.charge).sum() ** 2 / n + 1.0
    assert abs(ec - ec_ref) <= rel * size + 3 * rel * abs(ec_ref)
    assert abs(elj - elj_ref) <= rel * size + 3 * rel * abs(elj_ref)
