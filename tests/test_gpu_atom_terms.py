"""Bonded terms and exclusion corrections at the edges of their per-atom sums:
atoms without a term, an atom in many, terms listed twice and in either order,
less than a supercluster and just more than whole ones."""
import numpy as np
import pytest

from oracle import md
from oracle import oracle as O
from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu


def _molecules(n, seed, star):
    """n atoms on a jittered grid of 1.9 A, bonds of random order between
    neighbours in the first two thirds, one star, every bonded pair excluded."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    box = max(12.0, 1.9 * m)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = 1.9 * g + rng.uniform(-0.2, 0.2, (n, 3))
    k = max(1, 2 * n // 3)
    bonds = [(a, a + 1) if a % 3 else (a + 1, a) for a in range(k - 1)]
    bonds += bonds[:2] + [(0, j) for j in range(2, min(n, star + 2))]
    angles = [(a, a + 1, a + 2) if a % 2 else (a + 2, a + 1, a) for a in range(max(0, k - 2))]
    angles += angles[:1] + [(j, 0, j + 1) for j in range(2, min(n - 1, star + 1))]
    ex = {(min(b), max(b)): 1 for b in bonds}
    for a, _, c in angles:
        ex.setdefault((min(a, c), max(a, c)), 2)
    return systems.MolSystem(
        name="chain", pos=pos, charge=rng.uniform(-5, 5, n), atype=np.zeros(n, np.int32),
        molecule=np.zeros(n, np.int32), mass=rng.uniform(1, 16, n),
        lj=systems.charmm_table([0.1], [0.8], [0.05], [0.7]), box=np.array([box] * 3), origin=np.zeros(3),
        bonds=np.array(bonds, np.int32).reshape(-1, 2), bond_par=rng.uniform(1, 3, (len(bonds), 2)),
        angles=np.array(angles, np.int32).reshape(-1, 3), angle_par=rng.uniform(1, 3, (len(angles), 2)),
        exclusions=np.array([(*p, c) for p, c in sorted(ex.items())], np.int32).reshape(-1, 3), csf=0.4)


# FP64: every term and sum carries a few units of 1e-16 of forces up to 1e3;
# mixed: pair forces in FP32 (6e-8 of sums of terms up to 1e3), forces in 2^-32
@pytest.mark.parametrize("precision,rel", [(pmx.FP64, 1e-11), (pmx.MIXED, 3e-5)])
@pytest.mark.parametrize("n,star", [(1, 0), (2, 0), (3, 0), (64, 0), (65, 40), (200, 150), (513, 7)])
def test_terms_summed_by_atom(n, star, precision, rel):
    s = _molecules(n, 100 + n, star)
    kw = dict(lj=(pmx.SW_C2, 4.0, 5.9), pme=dict(rc=5.9, grid=(16, 16, 18), order=4, alpha=0.4))
    f_ref, e_ref = md.total_forces(s, O.make_spec(5.0, **kw), s.pos)
    ctx = pmx.Context(0)
    try:
        sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, **kw), precision)
        sy.md_init(s, 1.0, skin=0.0)
        sy.md_set_state(s.pos, np.zeros_like(s.pos))
        _, _, e = sy.md_get_state()
        f = sy.get_forces()[0]
        sy.close()
    finally:
        ctx.close()
    scale = np.sqrt(np.mean(np.sum(f_ref ** 2, 1))) + 1.0
    assert np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1))) <= rel * scale
    size = sum(abs(v) for v in e_ref.values()) + np.abs(s.charge).sum() ** 2 + 1.0
    for key, ref in e_ref.items():
        assert abs(e[key] - ref) <= rel * size, key
