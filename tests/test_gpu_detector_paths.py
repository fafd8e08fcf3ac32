"""The detector response's device paths at the sizes where they can go wrong:
escape peaks against a channel-by-channel restatement of
src/xmi_detector_f.F90:582-809 (odd channel counts, more orders than one pass
takes, several elements, axes that cover part of the spectrum, tables larger
than one launch takes, lines that land in their own channel, axes that only
the host routine takes), and the pile-up's channel search against its
statistics with contents in few channels."""
import ctypes as C

import numpy as np
import pytest

from xmimsim_amd import api, lines, workloads

pytestmark = pytest.mark.gpu


def _opts(**kw):
    return api.default_options(use_escape_peaks=1, use_sum_peaks=0, use_poisson=0, use_default_seeds=1, **kw)


def _ratios(Zs, fe, ci, co, rng, self_line):
    fluo = np.zeros((len(fe), 109, len(Zs)))
    for j in range(len(Zs)):
        for line in (2, 3, 5, 60, 90):
            fluo[:, line - 1, j] = 0.01 * rng.uniform(0.5, 1.5, len(fe))
        if self_line:  # an absent line: energy 0, lands in its own channel
            fluo[:, 24 - 1, j] = 0.003
            fluo[:, 28 - 1, j] = 0.002
    comp = 1e-3 * rng.random((len(co), len(ci)))
    Z = (C.c_int * len(Zs))(*Zs)
    keep = [np.ascontiguousarray(a, np.float64) for a in (fluo, fe, comp, ci, co)] + [Z]
    P = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    er = api.xmi_escape_ratios(len(Zs), len(fe), len(ci), len(co), C.cast(Z, C.POINTER(C.c_int)), P(keep[0]),
                               P(keep[1]), P(keep[2]), P(keep[3]), P(keep[4]), None)
    return er, keep


def _findpos(a, x):
    if abs(x - a[0]) < 1e-10:
        return 0
    above = np.flatnonzero(x <= a)
    return int(above[0]) - 1 if above.size else -1


def _restated(ch, gain, Zs, fluo, fe, comp, ci, co):
    ch = ch.copy()
    nch = ch.size
    atoms = [lines.atom(z) for z in Zs]
    e_all = (np.arange(nch) + 0.5) * gain
    for i in range(nch):
        e, s = e_all[i], 0.0
        if fe[0] <= e < fe[-1]:
            p = _findpos(fe, e)
            for j, a in enumerate(atoms):
                for sh, (lo, hi) in enumerate(zip((1, 32, 60, 86), (29, 58, 85, 109))):
                    for line in range(lo, hi + 1):
                        el = a["line_energy"][line]
                        if not e > a["edge"][sh] or not e - el >= 0.5 * gain:
                            continue
                        r0, r1 = fluo[p, line - 1, j], fluo[p + 1, line - 1, j]
                        r = r0 + (r1 - r0) * (e - fe[p]) / (fe[p + 1] - fe[p])
                        s += r
                        k = int((e - el) / gain)
                        if 0 <= k < nch:
                            ch[k] += r * ch[i]
        if ci[0] <= e < ci[-1] and i:
            p1 = _findpos(ci, e)
            d = e - e_all[:i]
            ok = np.flatnonzero((d >= co[0]) & (d < co[-1]))
            p2 = np.array([_findpos(co, x) for x in d[ok]], int)
            if ok.size:
                den = (ci[p1 + 1] - ci[p1]) * (co[p2 + 1] - co[p2])
                v = ((ci[p1 + 1] - e) * (co[p2 + 1] - d[ok]) * comp[p2, p1]
                     + (e - ci[p1]) * (co[p2 + 1] - d[ok]) * comp[p2, p1 + 1]
                     + (ci[p1 + 1] - e) * (d[ok] - co[p2]) * comp[p2 + 1, p1]
                     + (e - ci[p1]) * (d[ok] - co[p2]) * comp[p2 + 1, p1 + 1]) / den
                r = v * gain / (co[1] - co[0])
                ch[ok] += r * ch[i]
                s += r.sum()
        ch[i] *= 1.0 - s
    return ch


# (channels, orders, crystal, points of the three axes, axes' ends, self lines)
CASES = [(65, 1, [14], (40, 30, 30), 24.0, False), (257, 5, [14, 32], (90, 70, 81), 24.0, False),
         (300, 2, [32], (50, 40, 40), 9.0, True), (200, 3, [14], (60, 1500, 1600), 24.0, False),
         (128, 1, [14], (2, 2, 2), 24.0, False)]


@pytest.mark.parametrize("nch,n_int,Zs,n_axes,top,self_line", CASES)
def test_escape_peaks_on_the_device(orc, nch, n_int, Zs, n_axes, top, self_line):
    rng = np.random.default_rng(nch)
    gain = 24.0 / nch
    inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=n_int)
    inp.nchannels, inp.gain, inp.det_absorbers, inp.crystal = nch, gain, [], []
    prep = api.Prepared(inp)
    fe = np.linspace(1.0, top, n_axes[0])
    ci = np.linspace(0.7, top, n_axes[1])
    co = np.linspace(0.1, top, n_axes[2])
    er, keep = _ratios(Zs, fe, ci, co, rng, self_line)
    ch = np.zeros((n_int + 1, nch))
    ch[1:] = np.exp(rng.uniform(0.0, 8.0, (n_int, nch)))
    ch[1:, rng.integers(0, nch, nch // 3)] = 0.0
    print("escape peaks", nch, n_int, flush=True)
    out = api.detector_response(prep, ch, escape_ratios=er, options=_opts())
    again = api.detector_response_noalloc(prep, ch, escape_ratios=er, options=_opts())
    assert np.array_equal(out, again)
    for n in range(1, n_int + 1):
        ref = orc.detector_convolute(prep, _restated(ch[n], gain, Zs, *[keep[k] for k in (0, 1, 2, 3, 4)]))
        # sums of at most 4 nch terms of one sign, each of a few roundings, and
        # 1 - sum with sums below one half: 1e-12 is some 20 times the bound
        assert np.abs(out[n] - ref).max() <= 1e-12 * np.abs(ref).max(), n
    prep.close()


def test_axes_that_do_not_increase_take_the_host_routine(orc):
    """An axis with a repeated value is searched as the reference does, on the host."""
    rng = np.random.default_rng(3)
    nch, gain = 96, 0.25
    inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=1)
    inp.nchannels, inp.gain, inp.det_absorbers, inp.crystal = nch, gain, [], []
    prep = api.Prepared(inp)
    fe, ci = np.linspace(1.0, 24.0, 30), np.linspace(1.0, 24.0, 30)
    co = np.linspace(0.1, 24.0, 30)
    co[20] = co[19]
    er, keep = _ratios([14], fe, ci, co, rng, False)
    ch = np.zeros((2, nch))
    ch[1] = rng.uniform(1.0, 100.0, nch)
    out = api.detector_response(prep, ch, escape_ratios=er, options=_opts())
    ref = orc.detector_convolute(prep, _restated(ch[1], gain, [14], *keep[:5]))
    assert np.abs(out[1] - ref).max() <= 1e-12 * np.abs(ref).max()
    prep.close()


def test_workspaces_are_given_back():
    """What a response keeps for the next call goes with the release, whose
    repetition finds nothing; a response after it gives the same."""
    rng = np.random.default_rng(12)
    inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=4)
    inp.nchannels, inp.gain = 4096, 0.01
    prep = api.Prepared(inp)
    ch = np.zeros((5, 4096))
    ch[1:] = rng.uniform(0.0, 100.0, (4, 4096))
    opts = api.default_options(use_escape_peaks=0, use_sum_peaks=1, use_poisson=1, use_default_seeds=1)
    er, keep = _ratios([14], *(np.linspace(0.1, 24.0, 200) for _ in range(3)), rng, False)
    api.release_detector_workspaces()
    a = api.detector_response(prep, ch, escape_ratios=er, options=_opts())  # 8 MB of tables
    b = api.detector_response(prep, ch, options=opts)
    # one workspace (the calls came one after another): the tables on both sides, and the spectra
    assert 2 * (8 << 20) < api.release_detector_workspaces() <= 128 << 20
    assert api.release_detector_workspaces() == 0
    assert np.array_equal(api.detector_response(prep, ch, escape_ratios=er, options=_opts()), a)
    assert np.array_equal(api.detector_response(prep, ch, options=opts), b)
    prep.close()


@pytest.mark.parametrize("ne", [618, 619])
def test_many_escape_elements(ne):
    """Escape ratios of as many elements as the device's line buffer holds,
    and of one more (the host routine): only the first element's ratios are
    not zero, so both give what it gives alone."""
    rng = np.random.default_rng(6)
    inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=1)
    inp.nchannels, inp.gain, inp.det_absorbers, inp.crystal = 64, 0.375, [], []
    prep = api.Prepared(inp)
    ax = np.array([1.0, 12.0, 24.0])
    one, keep1 = _ratios([14], ax, ax, ax, rng, False)
    many, keep = _ratios([14] * ne, ax, ax, ax, rng, False)
    keep[0][:] = 0.0
    keep[0][:, :, 0] = keep1[0][:, :, 0]
    keep[2][:] = keep1[2]
    ch = np.zeros((2, 64))
    ch[1] = rng.uniform(1.0, 100.0, 64)
    ref = api.detector_response(prep, ch, escape_ratios=one, options=_opts())
    for respond in (api.detector_response, api.detector_response_noalloc):
        out = respond(prep, ch, escape_ratios=many, options=_opts())
        # sums of the same terms in another order
        assert np.abs(out - ref).max() <= 1e-12 * ref.max()
    prep.close()


@pytest.mark.parametrize("respond", [api.detector_response, api.detector_response_noalloc])
def test_no_order_leaves_nothing_under_way(respond):
    """Calls without an order (only the net-line histories get the detector's
    absorption) between calls with orders: another detector's tables of a call
    that has returned must not reach the next one's."""
    rng = np.random.default_rng(8)
    preps = []
    for k, thick in enumerate((0.002, 0.2)):
        inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=2)
        inp.nchannels, inp.gain = 128, 0.2
        inp.det_absorbers = [api.Layer([4 + 9 * k], [1.0], 1.85, thick)]
        preps.append(api.Prepared(inp))
    ch = np.zeros((3, 128))
    ch[1:] = rng.uniform(0.0, 100.0, (2, 128))
    vr = np.zeros((100, 385, 2))
    vr[25, 2] = vr[28, 1] = (1e4, 1e3)
    opts = api.default_options(use_escape_peaks=0, use_sum_peaks=0, use_poisson=0, use_default_seeds=1)
    v_ref = [vr.copy(), vr.copy()]
    ref = [respond(p, ch, v, options=opts) for p, v in zip(preps, v_ref)]
    assert np.abs(ref[0] - ref[1]).max() > 1e-3 * ref[0].max()
    for k in (0, 1, 1, 0):
        v = vr.copy()
        none = respond(preps[1 - k], np.full((1, 128), 7.0), v, options=opts)
        assert none.shape == (1, 128) and not none.any()
        assert np.array_equal(v, v_ref[1 - k])
        assert np.array_equal(respond(preps[k], ch, options=opts), ref[k])
    for p in preps:
        p.close()


@pytest.mark.parametrize("nch", [200, 4096, 5000])
def test_pileup_keeps_the_spectrum_without_pulses_in_time(nch):
    """A pulse width of 1e-12 s: every pulse is its own train, so the counts
    are a multinomial of the contents (channels between empty ones, the first
    and the last among them), on tables in LDS and beyond."""
    inp = workloads.single_layer_steel(n_photons_line=10, n_interactions=2)
    inp.nchannels, inp.gain, inp.noise, inp.fano = nch, 100.0 / nch, 1e-3, 1e-9
    inp.det_absorbers, inp.crystal, inp.pulse_width = [], [], 1e-12
    prep = api.Prepared(inp)
    lo = int(np.ceil(60.0 / inp.gain))  # above 50 keV: Gaussian response, here narrower than a channel
    at = np.array([lo, lo + 1, lo + 7, nch - 101, nch - 1])
    ch = np.zeros((3, nch))
    ch[1, at] = [4e5, 1e3, 2e5, 5.0, 1e5]
    ch[2, at] = [1e3, 3e5, 10.0, 4e5, 2e3]
    opts = api.default_options(use_escape_peaks=0, use_sum_peaks=1, use_poisson=0, use_default_seeds=1)
    out = api.detector_response(prep, ch, options=opts)
    for n in (1, 2):
        N = int(ch[n].sum())
        assert out[n].sum() == pytest.approx(N, abs=1e-6 * N)
        p = ch[n, at] / ch[n].sum()
        # five standard deviations of a binomial count
        assert np.all(np.abs(out[n, at] - N * p) <= 5.0 * np.sqrt(N * p * (1 - p)) + 1.0), (n, out[n, at])
    prep.close()
