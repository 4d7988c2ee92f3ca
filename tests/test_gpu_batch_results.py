"""What pmx_sys_get_forces returns after batched passes and runs in turn: the
forces of the last pass, whatever brought them about."""
import numpy as np
import pytest

from protomol3_amd import pmx, serve, systems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = pmx.Context(0)
    yield c
    c.close()


def _make(ctx, n, seed, precision=pmx.FP64, **kw):
    s = systems.replica_box(n, seed).with_velocities(300.0, seed=seed + 1)
    sy = pmx.System(ctx, s, serve.request_spec(s), precision)
    sy.md_init(s, **{**dict(timestep_fs=0.2, skin=2.0), **kw})
    sy.md_set_state(s.pos, s.vel)
    return sy


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("how", ["batch", "run"])
def test_forces_of_a_run_after_a_batched_evaluation(ctx, how, graphs):
    """Run, batched evaluation at the positions reached, run again: the forces
    are those of the last step, as without the evaluation (the FP64 form: the
    lists' builds, which the evaluation adds to, change only the order of
    sums).  Runs of 16 steps whose chunks are replays of one graph."""
    out = {}
    for evaluated in (False, True):
        sys_ = [_make(ctx, n, 20 + n, graphs=graphs) for n in (600, 1500)]
        try:
            def run():
                if how == "batch":
                    pmx.run_batch(sys_, 16)
                else:
                    for sy in sys_:
                        sy.md_run(16)
            run()
            run()
            f_before = [sy.get_forces()[0] for sy in sys_]
            if evaluated:
                pmx.evaluate_batch(sys_, [sy.md_get_state()[0] for sy in sys_])
            run()
            out[evaluated] = f_before, [sy.get_forces()[0] for sy in sys_]
        finally:
            for sy in sys_:
                sy.close()
    for f_old, f, g in zip(out[False][0], out[False][1], out[True][1]):
        scale = np.abs(f).max()
        assert np.abs(f - f_old).max() > 1e-3 * scale
        assert np.abs(f - g).max() <= 1e-8 * scale


@pytest.mark.parametrize("precision", [pmx.MIXED, pmx.FP64])
@pytest.mark.parametrize("how", ["batch", "run"])
def test_energies_of_the_state_under_new_launch_shapes(ctx, how, precision):
    """The energies of the state at hand do not change with the launch shapes
    set after the run (the list is cut into other runs, the x pass into other
    blocks), nor with a force pass that keeps its partials elsewhere."""
    sys_ = [_make(ctx, n, 40 + n, precision) for n in (900, 4000)]
    try:
        if how == "batch":
            pmx.run_batch(sys_, 16)
        else:
            for sy in sys_:
                sy.md_run(16)
        for sy, first in zip(sys_, (False, True)):
            e0 = sy.md_get_state()[2] if first else None
            for knob, value in ((pmx.TUNE_PAIR_BLOCKS_PER_CU, 1), (pmx.TUNE_FFT_PLANES, 0), (pmx.TUNE_FFT_LINES, 1),
                                (pmx.TUNE_FFT_PLANES, 1)):
                sy.set_tuning(knob, value)
                e = sy.md_get_state()[2]
                if e0 is None:
                    e0 = e
                assert e == e0, (knob, value)
            x, _, _ = sy.md_get_state()
            _, ec, elj = sy.evaluate(x)
            # FP32 pair energies summed over other runs: 1e-6 of their magnitudes
            tol = 1e-9 if precision == pmx.FP64 else 1e-6
            size = abs(ec) + abs(elj)
            assert abs(e0["coulomb"] - ec) <= tol * size + (1e-3 if precision == pmx.MIXED else 0.0)
            assert abs(e0["lj"] - elj) <= tol * size + (1e-3 if precision == pmx.MIXED else 0.0)
        if how == "batch":
            pmx.run_batch(sys_, 16)
        for sy in sys_:
            if how == "run":
                sy.md_run(16)
            sy.compute_noalloc()
            e = sy.md_get_state()[2]
            _, ec, elj = sy.evaluate(sy.md_get_state()[0])
            size = abs(ec) + abs(elj)
            tol = (1e-9 if precision == pmx.FP64 else 1e-6) * size + (1e-3 if precision == pmx.MIXED else 0.0)
            assert abs(e["coulomb"] - ec) <= tol and abs(e["lj"] - elj) <= tol
    finally:
        for sy in sys_:
            sy.close()


def _droplet(n, seed):
    """A water droplet in a box of four times its edge: its lists outgrow the
    capacity set for the box's mean density."""
    s = systems.replica_box(n, seed).with_velocities(300.0, seed=seed + 1)
    first = s.pos[np.searchsorted(s.molecule, s.molecule)]
    s.pos = s.pos - s.box * np.rint((s.pos - first) / s.box)
    edge = float(s.box[0])
    s.box = np.array([4 * edge] * 3)
    spec = pmx.ForceSpec(4.5, lj=(pmx.SW_C2, 7.0, 9.0), pme=dict(rc=9.0, grid=(48, 48, 48), order=4, alpha=0.35))
    return s, spec


def _mixed(ctx, s, spec):
    sy = pmx.System(ctx, s, spec, pmx.MIXED)
    sy.md_init(s, 1.0, skin=1.0)
    sy.md_set_state(s.pos, s.vel)
    return sy


def _states(sys_):
    return [sy.md_get_state() for sy in sys_]


def _equal(a, b):
    return np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]


def test_batched_results_where_a_list_outgrows_its_buffers(ctx):
    """The first batched run or evaluation of a droplet, in which its buffers
    grow, gives the results of the second, in which they fit."""
    other = systems.replica_box(900, 3).with_velocities(300.0, seed=4)
    drop = _droplet(3000, 8)
    sys_ = [_mixed(ctx, *drop), _mixed(ctx, other, serve.request_spec(other))]
    ev = [pmx.System(ctx, *drop, pmx.MIXED), pmx.System(ctx, other, serve.request_spec(other), pmx.MIXED)]
    try:
        before = ev[0].device_bytes()
        e1 = pmx.evaluate_batch(ev, [drop[0].pos, other.pos])
        assert ev[0].device_bytes() > before
        e2 = pmx.evaluate_batch(ev, [drop[0].pos, other.pos])
        pmx.run_batch(sys_, 20)
        r1 = _states(sys_)
        for sy, s in zip(sys_, (drop[0], other)):
            sy.md_set_state(s.pos, s.vel)
        pmx.run_batch(sys_, 20)
        r2 = _states(sys_)
    finally:
        for sy in sys_ + ev:
            sy.close()
    for a, b in zip(e1, e2):
        assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]
    for a, b in zip(r1, r2):
        assert _equal(a, b)


@pytest.mark.parametrize("how", ["batch", "run"])
def test_a_run_leaves_the_energies_of_the_last_evaluation(ctx, how):
    """pmx_sys_get_forces gives the last step's forces and the energies and
    pair statistics of the last evaluation, in either kind of run."""
    s = systems.replica_box(900, 13).with_velocities(300.0, seed=14)
    sy = _mixed(ctx, s, serve.request_spec(s))
    try:
        _, ec, elj = sy.evaluate(s.pos + 0.05 * np.sin(np.arange(3 * s.n).reshape(-1, 3)), pmx.EVAL_PAIRSTATS)
        stats = sy.pair_stats()
        sy.md_set_state(s.pos, s.vel)
        if how == "batch":
            pmx.run_batch([sy], 10)
        else:
            sy.md_run(10)
        _, ec2, elj2 = sy.get_forces()
        assert (ec2, elj2) == (ec, elj) and sy.pair_stats() == stats
    finally:
        sy.close()


def test_first_forces_do_not_depend_on_the_partners(ctx):
    """A new system's batched run is the same, to the last bit in the mixed
    form, in a batch of its own, with new partners and with partners that
    continue an earlier run."""
    s, t = (systems.replica_box(n, seed).with_velocities(300.0, seed=seed + 1) for n, seed in ((1500, 31), (2400, 33)))
    out = []
    for partner in (None, "new", "continued"):
        sys_ = [_mixed(ctx, s, serve.request_spec(s))]
        try:
            if partner:
                sys_.append(_mixed(ctx, t, serve.request_spec(t)))
            if partner == "continued":
                pmx.run_batch(sys_[1:], 5)
            pmx.run_batch(sys_, 12)
            out.append(_states(sys_[:1])[0] + (sys_[0].md_stats(),))
        finally:
            for sy in sys_:
                sy.close()
    for o in out[1:]:
        assert _equal(o, out[0]) and o[3] == out[0][3]


@pytest.mark.parametrize("how", ["batch", "run"])
def test_launch_shapes_leave_the_energies_of_the_last_evaluation(ctx, how):
    """Shapes set after a run change neither what pmx_sys_get_forces gives
    (the last evaluation's energies and pair statistics) nor the energies of
    the state."""
    s = systems.replica_box(900, 13).with_velocities(300.0, seed=14)
    sy, twin = _mixed(ctx, s, serve.request_spec(s)), _mixed(ctx, s, serve.request_spec(s))
    try:
        for t in (sy, twin):
            _, ec, elj = t.evaluate(s.pos + 0.05 * np.sin(np.arange(3 * s.n).reshape(-1, 3)), pmx.EVAL_PAIRSTATS)
            t.md_set_state(s.pos, s.vel)
            if how == "batch":
                pmx.run_batch([t], 10)
            else:
                t.md_run(10)
        stats = sy.pair_stats()
        for knob, value in ((pmx.TUNE_PAIR_BLOCKS_PER_CU, 1), (pmx.TUNE_FFT_PLANES, 0)):
            sy.set_tuning(knob, value)
            _, ec2, elj2 = sy.get_forces()
            assert (ec2, elj2) == (ec, elj) and sy.pair_stats() == stats
        assert sy.md_get_state()[2] == twin.md_get_state()[2]
    finally:
        sy.close()
        twin.close()
