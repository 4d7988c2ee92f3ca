"""PME grids with an axis of more than 4,096 points, whose passes hold more
points per thread: up to 10,125 in the mixed form and 5,120 in FP64, on every
axis, alone and in batched launches beside ordinary systems."""
import numpy as np
import pytest

from oracle import oracle as O
from protomol3_amd import pmx, systems

pytestmark = pytest.mark.gpu
LJ = (pmx.SW_C2, 5.0, 7.0)


def _pme(axis, n, order=4):
    grid = [8, 6, 10]
    grid[axis] = n
    if order > 6:
        grid = [max(g, order) for g in grid]
    return dict(rc=7.0, grid=tuple(grid), order=order, alpha=0.4)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("precision,n,order", [(pmx.MIXED, 4320, 6), (pmx.MIXED, 10125, 8), (pmx.FP64, 4320, 2),
                                               (pmx.FP64, 5120, 8)])
def test_forces_on_grids_with_a_long_axis(precision, n, order, axis):
    s = systems.water_box(n_side=5, box=15.5, seed=3)
    pme = _pme(axis, n, order)
    f_ref, ec_ref, _ = O.evaluate(s, O.make_spec(5.0, lj=LJ, pme=pme))
    # mixed: forces are differences of neighbouring points of an FP32
    # potential (2^-24 of its size each), whose number an angstrom grows with n
    tol = 1e-9 if precision == pmx.FP64 else 1e-8 * n
    ctx = pmx.Context(0)
    try:
        for spread2 in (0, 1):
            sy = pmx.System(ctx, s, pmx.ForceSpec(5.0, lj=LJ, pme=pme), precision)
            sy.set_tuning(pmx.TUNE_SPREAD_STREAM, spread2)
            f, ec, _ = sy.evaluate(s.pos)
            sy.close()
            assert np.sqrt(np.mean(np.sum((f - f_ref) ** 2, 1)) / np.mean(np.sum(f_ref ** 2, 1))) <= tol
            assert abs(ec - ec_ref) <= (1e-9 if precision == pmx.FP64 else 3e-5) * abs(ec_ref)
    finally:
        ctx.close()


def test_longer_axes_are_refused():
    s = systems.water_box(n_side=5, box=15.5, seed=3)
    ctx = pmx.Context(0)
    try:
        for precision, n in ((pmx.MIXED, 10240), (pmx.FP64, 5184)):
            for axis in range(3):
                with pytest.raises(pmx.PmxError) as e:
                    pmx.System(ctx, s, pmx.ForceSpec(5.0, lj=LJ, pme=_pme(axis, n)), precision)
                assert e.value.code == -4
    finally:
        ctx.close()


@pytest.mark.parametrize("precision", [pmx.MIXED, pmx.FP64])
def test_long_axes_in_a_batch(precision):
    """Systems with a long axis beside an ordinary one: the forces of each are
    those of a batch of its own (mixed to the last bit), and of an evaluation
    alone; a batched run follows the run in batches of one."""
    s = systems.water_box(n_side=5, box=15.5, seed=3).with_velocities(300.0, seed=5)
    specs = [pmx.ForceSpec(5.0, lj=LJ, pme=_pme(axis, 4320)) for axis in range(3)]
    specs.append(pmx.ForceSpec(5.0, lj=LJ, pme=dict(rc=7.0, grid=(16, 15, 18), order=4, alpha=0.4)))
    exact = precision == pmx.MIXED

    def close(a, b, tol):
        return np.array_equal(a, b) if exact else np.abs(a - b).max() <= tol * np.abs(b).max()

    ctx = pmx.Context(0)
    out = []
    try:
        for together in (True, False):
            sys_ = [pmx.System(ctx, s, sp, precision) for sp in specs]
            groups = [sys_] if together else [[sy] for sy in sys_]
            f = [r for g in groups for r in pmx.evaluate_batch(g, [s.pos] * len(g))]
            alone = [sy.evaluate(s.pos) for sy in sys_]
            for sy in sys_:
                sy.md_init(s, 0.5, skin=0.4)
                sy.md_set_state(s.pos, s.vel)
            for g in groups:
                pmx.run_batch(g, 10)
            out.append((f, alone, [sy.md_get_state()[0] for sy in sys_]))
            for sy in sys_:
                sy.close()
    finally:
        ctx.close()
    for f, g, alone in zip(out[0][0], out[1][0], out[0][1]):
        assert close(f[0], g[0], 1e-12) and abs(f[1] - g[1]) <= (0.0 if exact else 1e-9 * abs(g[1]))
        assert np.abs(f[0] - alone[0]).max() <= (1e-4 if exact else 1e-9) * np.abs(alone[0]).max()
    for x, y in zip(out[0][2], out[1][2]):
        assert close(x, y, 1e-10)
