"""Arrays to and from the host at the sizes where they no longer go in one
piece: forces, positions and velocities below and above the 4 MB that a
system stages at once, with a remainder."""
import numpy as np
import pytest

from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu


# 648 atoms a cell: 16,848 atoms (all in one piece), 168,480 (forces in one
# piece, state in chunks), 174,960 (both in chunks of 1 MB and a remainder)
@pytest.mark.parametrize("cells", [(2, 1, 13), (2, 10, 13), (5, 6, 9)])
def test_forces_and_state_in_chunks(cells):
    base = systems.water_box(n_side=6, box=18.6, seed=3)
    assert base.n == 648
    kw = dict(lj=(pmx.SW_C2, 4.0, 6.0), coul=(pmx.SW_C1, 0.0, 6.0))
    s = systems.tiled(base, cells)
    ctx = pmx.Context(0)
    try:
        one = pmx.System(ctx, base, pmx.ForceSpec(6.0, **kw), pmx.FP64)
        f0, _, _ = one.evaluate(base.pos)
        one.close()
        sy = pmx.System(ctx, s, pmx.ForceSpec(6.0, **kw), pmx.FP64)
        f, _, _ = sy.evaluate(s.pos)
        rng = np.random.default_rng(1)
        v = rng.normal(0, 1e-3, (s.n, 3))
        sy.md_init(s, 1.0, skin=0.5)
        sy.md_set_state(s.pos, v)
        x1, v1, e = sy.md_get_state()
        f1, _, _ = sy.get_forces()
        sy.close()
    finally:
        ctx.close()
    # every cell has the base cell's forces: sums of the same terms in another
    # order, on coordinates up to 200 A (1e-14 of them)
    scale = np.sqrt(np.mean(np.sum(f0 ** 2, 1)))
    tiled = np.tile(f0, (s.n // base.n, 1))
    assert np.abs(f - tiled).max() <= 1e-10 * scale * 100
    assert np.array_equal(x1, s.pos) and np.array_equal(v1, v)
    assert np.isfinite(f1).all() and f1.shape == f.shape
    assert abs(e["kinetic"] - 0.5 * np.sum(s.mass[:, None] * v ** 2)) <= 1e-9 * e["kinetic"]
