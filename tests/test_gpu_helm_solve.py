"""The Helmholtz right-hand sides in r segments and the partitioned radial
solves against the oracle, at the line lengths where their shapes change:
one segment, a ragged last one, the ends of each row capacity (72, 256, 400,
800 rows) and one past the longest, and for factors that exchange rows.
Planes of 180 lines: no multiple of 64, and one partial theta tile.
Tolerance: the 1e-10 relative L2 of the workload contract."""
import numpy as np
import pytest

from helpers import compare_fields, load_both, random_state, rel_l2, small_params, start_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("defer", ["0", "2"])
@pytest.mark.parametrize("nrm", [3, 8, 9, 16, 72, 73, 256, 257, 400, 401, 800, 801])
def test_step_at_row_capacities(tc, oracle, monkeypatch, nrm, defer):
    monkeypatch.setenv("TC_DEFER_CORRECTION", defer)
    p = small_params(tc, 20, 9, nrm, ntst=1000, dtmin=1e-4, dtmax=1e-4, sizepert=0.1,
                     omegapert=0.5, virotext=-0.3)
    dev, orc = start_pair(tc, oracle, p, 11, 1e-2)
    for n in range(2):
        assert dev.step(n)[0] == orc.step(n)[0] == 0
    compare_fields(dev, orc, nrm, 1e-10)


@pytest.mark.parametrize("nrm", [17, 100, 300, 500])
def test_slip_walls_on_both_cylinders(tc, oracle, nrm):
    """Masks that differ from line to line, on the outer wall too, through
    the routine entries (which keep the masks they are given)."""
    p = small_params(tc, 20, 9, nrm, ren=500.0)
    _implicit(tc, oracle, p, 1e-4, nrm)


@pytest.mark.parametrize("nrm,dt", [(9, 2.0), (33, 0.3)])
def test_factors_with_row_exchanges(tc, oracle, nrm, dt):
    """A free-slip outer wall at a dt whose last matrix row is larger off the
    diagonal than on it: dgttrf exchanges the last two rows."""
    p = small_params(tc, 20, 9, nrm, ren=50.0)
    am = tc.grid_vector(p, "am1j")[nrm - 1]
    assert am * 0.5 * dt / p["ren"] * 8.0 / 15.0 > 1.0
    _implicit(tc, oracle, p, dt, nrm)


def _implicit(tc, oracle, p, dt, nrm):
    dev, orc = tc.Solver(p), oracle.Oracle(p)
    rng = np.random.default_rng(nrm)
    masks = [rng.integers(0, 2, (p["nzm"], p["nthm"])).astype(np.int32) for _ in range(2)]
    load_both(dev, orc, random_state(p, 5))
    for s in (dev, orc):
        s.set_time(0.3, dt)
        s.begin_step()
        s.set_masks(*masks)
        s.set_substep(1)
    for a, b in (("ImplicitAndUpdateQT", "implicit_and_update_qt"), ("ImplicitAndUpdateQR", "implicit_and_update_qr"),
                 ("ImplicitAndUpdateQZ", "implicit_and_update_qz")):
        getattr(dev, a)()
        orc.call(b)
    for f, sl in (("qt", slice(0, nrm)), ("qr", slice(0, nrm + 1)), ("qz", slice(0, nrm))):
        assert rel_l2(dev.get(f)[sl], orc.get(f)[sl]) < 1e-10, f


def test_masks_set_between_steps_are_replaced(tc):
    """A step forms SlipBCs' masks again after others were set, also where
    the pattern has not moved since the last step."""
    p = small_params(tc, 48, 40, 17, minstrz=3, multmin=1)
    s = tc.Solver(p)
    s.set_time(0.0, 1e-3)
    s.begin_step()
    want = s.masks()
    ones = np.ones_like(want[0])
    assert want[0].min() == 0
    s.set_masks(ones, ones)
    s.begin_step()
    got = s.masks()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("defer", ["0", "2"])
@pytest.mark.parametrize("nrm", [1025, 1601])
def test_step_with_lines_in_chunks(tc, oracle, monkeypatch, nrm, defer):
    """Lines past the 800 rows that a block holds: a first chunk of 225 rows,
    and three chunks of which the first is one row (for q_r two full ones)."""
    monkeypatch.setenv("TC_DEFER_CORRECTION", defer)
    p = small_params(tc, 20, 9, nrm, ntst=1000, dtmin=1e-4, dtmax=1e-4, sizepert=0.1,
                     omegapert=0.5, virotext=-0.3)
    dev, orc = start_pair(tc, oracle, p, 11, 1e-2)
    for n in range(2):
        assert dev.step(n)[0] == orc.step(n)[0] == 0
    compare_fields(dev, orc, nrm, 1e-10)


@pytest.mark.parametrize("nrm", [801, 1030])
def test_slip_walls_with_lines_in_chunks(tc, oracle, nrm):
    p = small_params(tc, 20, 9, nrm, ren=500.0)
    _implicit(tc, oracle, p, 1e-6, nrm)


def test_batched_lines_in_chunks_equal_the_single_run(tc):
    p = small_params(tc, 20, 9, 801, idtv=0, ntst=1000, dtmin=1e-4, dtmax=1e-4, limitcfl=1e30)
    f = tc.init_perturbed_couette(p, 3, 1e-2)
    s = tc.Solver(p)
    with tc.Batch() as b:
        ids = [b.add(p) for _ in range(2)]
        for t in [s] + [b.solver(i) for i in ids]:
            for n, a in zip(("qt", "qr", "qz"), f):
                t.set(n, a)
            t.project()
        s.run(0, 3)
        b.advance(3)
        for i in ids:
            for n in ("qt", "qr", "qz", "pr"):
                assert np.array_equal(b.solver(i).get(n), s.get(n)), n


@pytest.mark.parametrize("nrm", [200, 201])
def test_step_where_the_rows_a_wave_change(tc, oracle, nrm):
    """Eight waves of 25 rows, and the first length with 50 a wave."""
    p = small_params(tc, 20, 9, nrm, ntst=1000, dtmin=1e-4, dtmax=1e-4)
    dev, orc = start_pair(tc, oracle, p, 11, 1e-2)
    assert dev.step(0)[0] == orc.step(0)[0] == 0
    compare_fields(dev, orc, nrm, 1e-10)


def _slip_implicit(tc, p, dt, masks, between=None):
    """Fields after one substep's implicit updates under `masks`, with other
    masks set and taken back before where `between` gives them."""
    s = tc.Solver(p)
    for name, a in random_state(p, 5).items():
        s.set(name, a)
    s.set_time(0.3, dt)
    s.begin_step()
    if between is not None:
        s.set_masks(*between)
    s.set_masks(*masks)
    s.set_substep(1)
    s.ImplicitAndUpdateQT(), s.ImplicitAndUpdateQR(), s.ImplicitAndUpdateQZ()
    return {f: s.get(f) for f in ("qt", "qr", "qz")}


def test_row_exchanges_of_other_lines_change_nothing(tc):
    """A free-slip outer wall exchanges rows of q_theta here.  No other
    component, no pattern without such lines and no later one without them
    may be solved differently because of it."""
    p = small_params(tc, 20, 9, 33, ren=50.0)
    am = tc.grid_vector(p, "am1j")[32]
    assert am * 0.5 * 0.3 / p["ren"] * 8.0 / 15.0 > 1.0
    ones = np.ones((p["nzm"], p["nthm"]), np.int32)
    half = ones.copy()
    half[:, ::2] = 0
    plain = _slip_implicit(tc, p, 0.3, (ones, ones))
    after = _slip_implicit(tc, p, 0.3, (ones, ones), between=(half, half))
    inner = _slip_implicit(tc, p, 0.3, (half, ones))
    outer = _slip_implicit(tc, p, 0.3, (ones, half))
    for f in ("qt", "qr", "qz"):
        assert np.array_equal(after[f], plain[f]), f
    for masked in (inner, outer):
        assert np.array_equal(masked["qr"], plain["qr"])


@pytest.mark.parametrize("strength", [1.5, 3.5])
def test_folded_solve_does_not_amplify_its_rounding(tc, strength):
    """One AB2 step of a flow that is 1 in the inner half and 2 in the outer,
    whose explicit terms vanish: the fused step folds q into the radial
    solve, the routines add the solution to q.  Powers of two make every
    product of the right-hand side exact, so both solve for the same one (in
    general they contract its products differently, which alone is 6e-15 of q
    on the clustered rows) and differ by what the fold rounds.  On rows
    clustered so that beta*ac is some tens and some ten thousands a fold that
    cancels loses 2e-16 and 4e-15 of q (a model of the same systems against
    extended precision); three roundings of q's size and the solve's own give
    3e-16 at either.  Bound: three times that."""
    p = small_params(tc, 16, 12, 385, nsst=1, ntst=1000, ren=1e3, str=strength, dtmin=1e-2, dtmax=1e-2,
                     virotext=0.5)
    out = []
    for fused in (True, False):
        d = tc.Solver(p)
        d.set_fused(fused)
        q = np.zeros(d.shape, order="F")
        q[:192], q[192:385] = 1.0, 2.0
        d.set("qt", q), d.set("qz", q)
        d.set_time(0.0, p["dtmax"])
        d.TimeMarcher()
        out.append({f: d.get(f)[:385] for f in ("qt", "qz")})
    for f in ("qt", "qz"):
        assert rel_l2(out[0][f], out[1][f]) <= 9e-16, f


def test_a_line_keeps_its_bits_beside_other_lines(tc):
    """No-slip lines beside grooves of the inner wall, where each lane reads
    its own table, and among themselves, where a block shares one."""
    p = small_params(tc, 20, 9, 33, ren=50.0)
    ones = np.ones((p["nzm"], p["nthm"]), np.int32)
    half = ones.copy()
    half[:, ::2] = 0
    plain = _slip_implicit(tc, p, 0.3, (ones, ones))
    inner = _slip_implicit(tc, p, 0.3, (half, ones))
    for f in ("qt", "qr", "qz"):
        assert np.array_equal(inner[f][:, :, 1::2], plain[f][:, :, 1::2]), f
