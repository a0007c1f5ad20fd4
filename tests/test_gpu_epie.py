"""ePIE iteration on the GPU against the FP64 oracle (same state, same position order).

Frames of 64^2 and more are shared by a team of workgroups; 16^2 and 32^2 frames run on one
workgroup with the exit waves staged through LDS.
Both are checked, with and without texture-weight quantisation, with a second (unused) probe mode
whose intensities enter the probe maximum, and in the modal form."""
import numpy as np
import pytest

from conftest import rel_err
from problems import make_problem

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _engine_for(p, quant=0):
    from ptychopy_amd._engine import Engine
    e = Engine(p["n"], p["m"], p["shape"], n_modes=p["k"], tex_quantize=quant)
    e.set_frames(p["amp"])
    e.set_positions(p["pos"])
    e.clear_object()
    e.init_probe(beam_size=60e-9, dx_s=5e-9)
    return e


def _flags(i, rms=False):
    from ptychopy_amd import _engine as E
    f = E.FLAG_RMS if rms else 0
    if i <= 1:
        f |= E.FLAG_PHASE_CONSTRAINT
    if i >= 10:
        f |= E.FLAG_UPDATE_PROBE
    return f


def _check(e, orc, p, amp, order, flags, quant=0, k_use=1, modal=False):
    from ptychopy_amd import _engine as E
    o0, p0 = e.get_object(), e.get_probe()
    sc = e.get_scalars()
    st = orc.EpieState(o0, p0, sc[E.SCAL_OBJ_MAX], sc[E.SCAL_PROBE_MAX])
    err_g = e.epie_iteration(order, flags)
    err_o = orc.epie_iteration(st, amp, p["pos"], order, k_use=k_use, modal=modal,
                               phase_constraint=bool(flags & E.FLAG_PHASE_CONSTRAINT),
                               update_probe=bool(flags & E.FLAG_UPDATE_PROBE), rms=bool(flags & E.FLAG_RMS),
                               quantize=quant)
    errs = dict(obj=rel_err(e.get_object(), st.obj), probe=rel_err(e.get_probe(), st.probe))
    print("epie step errors", errs)
    assert errs["obj"] < TOL and errs["probe"] < TOL, errs
    sc1 = e.get_scalars()
    assert sc1[E.SCAL_OBJ_MAX] == pytest.approx(st.scal[0], rel=1e-5)
    assert sc1[E.SCAL_PROBE_MAX] == pytest.approx(st.scal[1], rel=1e-5)
    if flags & E.FLAG_RMS:
        assert err_g == pytest.approx(err_o, rel=1e-4)
    return errs


@pytest.mark.parametrize("m,n_side,seed,quant", [(32, 4, 0, 0), (64, 4, 1, 0), (128, 3, 2, 1), (16, 5, 3, 0),
                                                   (128, 4, 4, 0), (64, 3, 5, 1)])
def test_epie_iterations_match_oracle(gpu, orc, m, n_side, seed, quant):
    p = make_problem(m=m, n_side=n_side, seed=seed)
    rng = np.random.default_rng(seed)
    with _engine_for(p, quant) as e:
        amp = e.get_frames().astype(np.float64)
        for i in range(1, 12):
            order = rng.permutation(p["n"])
            if i in (1, 2, 10, 11):
                _check(e, orc, p, amp, order, _flags(i, rms=(i == 2)), quant)
            else:
                e.epie_iteration(order, _flags(i))


def test_epie_is_bitwise_deterministic(gpu):
    p = make_problem(m=64, n_side=3, seed=7)
    outs = []
    for _ in range(2):
        rng = np.random.default_rng(0)
        with _engine_for(p) as e:
            for i in range(1, 12):
                e.epie_iteration(rng.permutation(p["n"]), _flags(i))
            outs.append((e.get_object(), e.get_probe()))
    for a, b in zip(outs[0], outs[1]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_epie_with_an_unused_second_mode_matches_oracle(gpu, orc):
    """Single-mode updates with K = 2 stored modes: the probe maximum also runs over mode 2."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=128, n_side=3, seed=6, modes=2)
    rng = np.random.default_rng(6)
    with _engine_for(p) as e:
        pr = e.get_probe()
        pr[1] = 1.2 * pr[0].T  # brighter than mode 1 somewhere, so it sets the maximum at first
        e.set_probe(pr)
        e.refresh_maxima()
        amp = e.get_frames().astype(np.float64)
        for i in (1, 10, 11):
            _check(e, orc, p, amp, rng.permutation(p["n"]), _flags(i, rms=(i == 11)))


@pytest.mark.parametrize("m,seed", [(32, 8), (128, 9)])
def test_modal_epie_matches_oracle(gpu, orc, m, seed):
    """Modal ePIE (all modes updated against the summed intensity) after the modes are formed."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=m, n_side=3, seed=seed, modes=2)
    rng = np.random.default_rng(seed)
    with _engine_for(p) as e:
        amp = e.get_frames().astype(np.float64)
        for i in range(1, 4):
            e.epie_iteration(rng.permutation(p["n"]), _flags(i))
        modal = E.FLAG_UPDATE_MODES | E.FLAG_UPDATE_PROBE
        e.epie_iteration(rng.permutation(p["n"]), modal)  # forms the modes (from the base probe)
        assert np.abs(e.get_probe()[1]).max() > 0
        for rms in (False, True):
            _check(e, orc, p, amp, rng.permutation(p["n"]), modal | (E.FLAG_RMS if rms else 0), k_use=2, modal=True)


def _near_engine(p, amp=None):
    """An engine a few steps from the truth (spectra well above rounding wherever counts are)."""
    from ptychopy_amd import _engine as E
    rng = np.random.default_rng(3)
    e = E.Engine(p["n"], p["m"], p["shape"], n_modes=p["k"])
    e.set_frames(p["amp"] if amp is None else amp)
    e.set_positions(p["pos"])
    e.set_object((0.95 * p["obj"]).astype(np.complex64))
    modes = [p["probe"]] + [0.4 * p["probe"] * (rng.standard_normal(p["probe"].shape) + 1j) for _ in range(p["k"] - 1)]
    modes = np.array(modes) * np.exp(0.5j * rng.standard_normal(p["probe"].shape))
    if p["k"] > 1:
        e.set_probe(modes)
        e.begin_modal()
    e.set_probe(modes)
    e.refresh_maxima()
    s = e.get_scalars()
    s[E.SCAL_PROBE_MAX] = float((np.abs(e.get_probe().astype(np.complex128)) ** 2).sum(axis=0).max())
    e.set_scalars(s)
    return e


def _flat_counts(p):
    """Amplitudes without dark pixels: the model's own spectrum is nowhere decided by rounding alone."""
    return (p["amp"] + 0.05 * p["amp"].mean(axis=(1, 2), keepdims=True) + 1.0).astype(np.float32)


@pytest.mark.parametrize("m,n_side,step,modes,rms,pc", [
    (64, 1, 5.0, 1, True, False),     # one position: the canvas is hardly larger than the ROI
    (64, 3, 150.3, 2, False, True),   # canvas rows and columns far beyond the ROI
    (128, 2, 331.7, 3, True, False),
    (256, 2, 40.2, 1, True, True),
    (256, 2, 21.9, 4, True, False),
    (512, 2, 33.3, 1, False, False),
    (512, 2, 27.1, 3, True, False),
])
def test_team_iterations_match_oracle(gpu, orc, m, n_side, step, modes, rms, pc):
    """Frames shared by a team of workgroups: sizes, modes in and out of LDS, small and wide canvases."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=m, n_side=n_side, step=step, seed=m + modes, modes=modes, photons=100.0 * m * m)
    rng = np.random.default_rng(m)
    flags = E.FLAG_UPDATE_PROBE | (E.FLAG_RMS if rms else 0) | (E.FLAG_UPDATE_MODES if modes > 1 else 0)
    with _near_engine(p, _flat_counts(p)) as e:
        amp = e.get_frames().astype(np.float64)
        kw = dict(k_use=modes, modal=modes > 1)
        _check(e, orc, p, amp, rng.permutation(p["n"]), flags, **kw)
        _check(e, orc, p, amp, rng.permutation(p["n"]),
               (flags & ~E.FLAG_UPDATE_PROBE) | (E.FLAG_PHASE_CONSTRAINT if pc else 0), **kw)
        _check(e, orc, p, amp, rng.permutation(p["n"]), flags, **kw)


def test_teams_of_several_threads_give_their_own_results(gpu):
    """More teams at once than the device holds: each handle's result is the one it gives alone."""
    import threading
    from ptychopy_amd import _engine as E
    p = make_problem(m=256, n_side=2, step=30.0, seed=5)
    orders = [np.random.default_rng(i).permutation(p["n"]) for i in range(6)]

    def go(out, i):
        with _near_engine(p) as e:
            for _ in range(3):
                e.epie_iteration(orders[i], E.FLAG_UPDATE_PROBE)
            out[i] = (e.get_object(), e.get_probe())

    alone, together = {}, {}
    for i in range(6):
        go(alone, i)
    ts = [threading.Thread(target=go, args=(together, i)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in range(6):
        for a, b in zip(alone[i], together[i]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _wide_problem(cols, n, seed, m=64, rows=100, modes=1):
    """Frames scattered over a canvas many times as wide as they are, some of them overlapping and two at
    its left and right ends."""
    import oracle
    from ptychopy_amd import sim
    rng = np.random.default_rng(seed)
    pos = np.stack([rng.uniform(0, rows - m, n), rng.uniform(0, cols - m, n)], axis=1).astype(np.float32)
    pos[:2, 1] = 0, cols - m
    pos[2:n // 2, 1] = (pos[0, 1] + rng.uniform(0, 1.5 * m, n // 2 - 2)).astype(np.float32)
    obj = sim.random_field_object((rows, cols), rng, phase_std=0.5)
    probe = sim.gaussian_probe(m, fwhm=m / 3, defocus_edge=2.0)
    amp = sim.poisson_amplitudes(oracle.simulate(obj, probe, pos, squared=True), 100.0 * m * m, rng)
    return dict(pos=pos, obj=obj, probe=probe, amp=amp, shape=(rows, cols), m=m, n=n, k=modes)


@pytest.mark.parametrize("m,cols,modes", [(64, 2200, 1), (64, 4173, 2), (128, 2500, 1)])
def test_teams_on_wide_canvases_match_oracle(gpu, orc, m, cols, modes):
    """A long row of |O|^2 beside the frame: the maximum of the whole canvas enters every probe update,
    whatever a workgroup is at when the others announce theirs."""
    from ptychopy_amd import _engine as E
    p = _wide_problem(cols, 12, cols, m=m, rows=m + 36, modes=modes)
    rng = np.random.default_rng(cols)
    flags = E.FLAG_UPDATE_PROBE | (E.FLAG_UPDATE_MODES if modes > 1 else 0)
    with _near_engine(p, _flat_counts(p)) as e:
        amp = e.get_frames().astype(np.float64)
        for f in (flags | E.FLAG_RMS, flags & ~E.FLAG_UPDATE_PROBE, flags):
            _check(e, orc, p, amp, rng.permutation(p["n"]), f, k_use=modes, modal=modes > 1)


def test_teams_on_wide_canvases_repeat_bitwise(gpu):
    """The same iterations from the same state give the same bits, run after run."""
    from ptychopy_amd import _engine as E
    p = _wide_problem(2200, 24, 11)
    orders = [np.random.default_rng(i).permutation(p["n"]) for i in range(4)]
    first = None
    with _near_engine(p) as e:
        state = e.get_object(), e.get_probe(), e.get_scalars()
        for _ in range(25):
            e.set_object(state[0])
            e.set_probe(state[1])
            e.refresh_maxima()
            e.set_scalars(state[2])
            for o in orders:
                e.epie_iteration(o, E.FLAG_UPDATE_PROBE)
            out = [a.view(np.uint32) for a in (e.get_object(), e.get_probe())] + [e.get_scalars().view(np.uint64)]
            first = first or out
            for a, b in zip(first, out):
                assert np.array_equal(a, b)


@pytest.mark.parametrize("m,rows,cols,at", [
    (64, 64, 64, (0, 0)),        # nothing beside the frame
    (64, 70, 128, (3, 64)),      # whole segments on both sides
    (64, 66, 129, (1, 1)),       # one pixel on each side, a last segment of one column
    (64, 200, 200, (70, 63)),
    (64, 1100, 333, (1000, 65)),
    (64, 71, 9000, (2, 4500)),   # more segments than a thread reads at once
    (128, 130, 383, (2, 127)),
    (256, 257, 700, (0, 300)),
    (512, 513, 1100, (1, 500)),
])
def test_canvas_maximum_wherever_it_lies(gpu, orc, m, rows, cols, at):
    """The probe step divides by max |O|^2 of the canvas: one bright pixel at the edges of the frame, of
    its segments and of the canvas has to be seen (it makes the step 4 times shorter)."""
    import oracle
    from ptychopy_amd import _engine as E
    from ptychopy_amd import sim
    rng = np.random.default_rng(cols)
    pos = np.array([at, (rows - m, cols - m)], np.float32)
    obj = sim.random_field_object((rows, cols), rng, phase_std=0.5)
    probe = sim.gaussian_probe(m, fwhm=m / 3, defocus_edge=2.0)
    amp = sim.poisson_amplitudes(oracle.simulate(obj, probe, pos, squared=True), 100.0 * m * m, rng)
    p = dict(pos=pos, obj=obj, probe=probe, amp=amp, shape=(rows, cols), m=m, n=2, k=1)
    r, c = at
    lo, hi = c // 64 * 64, (c + m + 63) // 64 * 64
    spots = {(y, x) for y in (r, r + m - 1) for x in (0, lo - 1, lo, c - 1, c + m, hi - 1, hi, cols - 1)}
    spots |= {(y, x) for y in (0, r - 1, r + m, rows - 1) for x in (c, cols - 1)}
    with _near_engine(p, _flat_counts(p)) as e:
        a64 = e.get_frames().astype(np.float64)
        for y, x in sorted(s for s in spots if 0 <= s[0] < rows and 0 <= s[1] < cols):
            o = (0.95 * obj).astype(np.complex64)
            o[y, x] *= 2.0 * np.abs(o).max() / abs(o[y, x])
            e.set_object(o)
            e.set_probe(probe * np.exp(0.3j * rng.standard_normal(probe.shape)))
            e.refresh_maxima()
            _check(e, orc, p, a64, [0, 1], E.FLAG_UPDATE_PROBE)


@pytest.mark.parametrize("m,modes,most", [(64, 3, 1), (128, 4, 2), (256, 14, 0), (512, 7, 0)])
def test_modes_beyond_lds_match_oracle(gpu, orc, m, modes, most):
    """More modes than a workgroup's LDS holds (or is let hold): the others' spectra wait in the exchange
    buffer, with an even and an odd number of transform stages."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=m, n_side=2, step=27.1, seed=m + modes, modes=modes, photons=100.0 * m * m)
    rng = np.random.default_rng(m)
    flags = E.FLAG_UPDATE_PROBE | E.FLAG_UPDATE_MODES
    with _near_engine(p, _flat_counts(p)) as e:
        e.set_tuning(E.TUNE_EPIE_RESIDENT, most)
        assert 0 < e.get_tuning(E.TUNE_EPIE_RESIDENT) < modes
        amp = e.get_frames().astype(np.float64)
        for f in (flags, flags | E.FLAG_RMS):
            _check(e, orc, p, amp, rng.permutation(p["n"]), f, k_use=modes, modal=True)


@pytest.mark.parametrize("m,modes", [(64, 1), (64, 2), (128, 1), (128, 3), (256, 1), (256, 2), (512, 1), (512, 2)])
def test_one_workgroup_matches_oracle(gpu, orc, m, modes):
    """The form without a team (devices that cannot hold one), at the sizes that have a team."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=m, n_side=2, step=27.1, seed=m + modes, modes=modes, photons=100.0 * m * m)
    rng = np.random.default_rng(m)
    flags = E.FLAG_UPDATE_PROBE | (E.FLAG_UPDATE_MODES if modes > 1 else 0)
    with _near_engine(p, _flat_counts(p)) as e:
        assert e.get_tuning(E.TUNE_EPIE_TEAM) > 0
        e.set_tuning(E.TUNE_EPIE_TEAM, 0)
        assert e.get_tuning(E.TUNE_EPIE_TEAM) == 0
        amp = e.get_frames().astype(np.float64)
        for f in (flags, (flags & ~E.FLAG_UPDATE_PROBE) | E.FLAG_PHASE_CONSTRAINT, flags | E.FLAG_RMS):
            _check(e, orc, p, amp, rng.permutation(p["n"]), f, k_use=modes, modal=modes > 1)


@pytest.mark.parametrize("m,modes", [(64, 1), (128, 2), (256, 1), (512, 1)])
def test_a_team_that_does_not_come_together(gpu, m, modes):
    """A team whose workgroups do not wait for one another gives up at once: one workgroup takes the
    iteration, with its own result to the bit, and the next team starts as if nothing had been."""
    from ptychopy_amd import _engine as E
    p = make_problem(m=m, n_side=2, step=27.1, seed=m, modes=modes)
    order = np.random.default_rng(m).permutation(p["n"])
    flags = E.FLAG_UPDATE_PROBE | E.FLAG_RMS | (E.FLAG_UPDATE_MODES if modes > 1 else 0)

    def states(*tuning):
        out = []
        with _near_engine(p) as e:
            for t in tuning:
                for key, value in t.items():
                    e.set_tuning(key, value)
                err = e.epie_iteration(order, flags)
                out.append([e.get_object().view(np.uint32), e.get_probe().view(np.uint32),
                            e.get_scalars().view(np.uint64), np.float64(err).view(np.uint64)])
        return out

    one, team = {E.TUNE_EPIE_TEAM: 0}, {E.TUNE_EPIE_TEAM: 1, E.TUNE_EPIE_TEAM_WAIT: 250}
    want = states(one, one, team, team)
    got = states({E.TUNE_EPIE_TEAM_WAIT: 0}, {}, team, team)
    for a, b in zip(want, got):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
