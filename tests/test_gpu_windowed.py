"""The windowed 1D transforms against the pruned ones and the CPU oracle at
the edges of their range: every grid size that has a window, both coarse
sizes (a narrow dataset moves the kept spectrum from one to the other and
past both) and walkers of each in one batch, split over 1, 2 and 4 workgroups,
two-signed beams, and nodes so dense that no window is used."""
import os

import numpy as np
import pytest

from conftest import REFDATA
from oracle_side import build_oracle, check_exact_parity
from pofd_affine_amd import fitsio, synth, workload

pytestmark = pytest.mark.gpu


def _window(ctx, walker=0):
    """The window that a walker's transforms took (0: the pruned ones, the
    only ones that keep rows)."""
    dbg = ctx.get_debug(walker)
    assert (dbg["nrows"] == 0) == (dbg["window"] > 0)
    return int(dbg["window"])


@pytest.mark.parametrize("nflux,ninterp,sigma,window", [
    # below 2^16 there is no window
    (32768, 512, 0.0025, 0), (65536, 400, 0.0025, 1),
    (65536, 1023, 0.0025, 1), (131072, 2048, 0.0025, 1),
    (262144, 2048, 0.0025, 1),
    # kept spectra above 1024 (the second window) and above 2048 (none)
    (65536, 512, 0.0006, 2), (131072, 2048, 0.0006, 2),
    (65536, 512, 0.0003, 0)])
def test_windowed_against_exact(nflux, ninterp, sigma, window):
    print("[gpu-window-case] %d %d %g" % (nflux, ninterp, sigma), flush=True)
    inp = dict(workload.make_inputs(npix_side=120, seed=9, sigma=sigma))
    th = synth.walker_thetas(3, seed=21)
    ctx = workload.build_context(inp, nflux, ninterp, binned=True)
    lls = []
    for parts in (1, 2, 4):
        ctx.set_parts(parts)
        ll, st = ctx.loglike_batch(th)
        assert np.all(st == 0), st
        lls.append(ll)
        assert _window(ctx) == window
    assert np.array_equal(lls[0], lls[1]) and np.array_equal(lls[0], lls[2])
    L = build_oracle(inp, nflux, ninterp, True, th[0])
    # the contract of every 1D path: 1e-6 of the exact-math value
    check_exact_parity(ctx, L, th, lls[2], tol=1e-6, nthreads=3)


@pytest.mark.parametrize("sigma,cut,window", [
    # the default keeps some 290 spectral indices at 2.5 mJy, 1200 at 0.6 mJy
    (0.0025, 746.0, 2), (0.0025, 12.0, 1),
    (0.0006, 746.0, 0), (0.0006, 12.0, 2)])
def test_other_spectral_cuts(sigma, cut, window):
    """A cut that keeps more of the spectrum takes the next window, or none;
    one that keeps half of it must not take a smaller one than the noise
    allows.  The kept spectrum is the default cut's, and the P(D) is the plain
    inverse transform of what is kept times the noise factor."""
    print("[gpu-window-case] cut %g %g" % (sigma, cut), flush=True)
    nflux = 65536
    inp = dict(workload.make_inputs(npix_side=120, seed=9, sigma=sigma))
    th = synth.walker_thetas(3, seed=22)
    ref = workload.build_context(inp, nflux, 512, binned=True)
    ctx = workload.build_context(inp, nflux, 512, binned=True,
                                 spectral_cut=cut)
    a, sa = ref.loglike_batch(th)
    b, sb = ctx.loglike_batch(th)
    assert np.all(sa == 0) and np.all(sb == 0)
    # e^-12 of the DC term is left out at the lower cut, so only the higher
    # cut's likelihood is the default one's
    if cut > 64:
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-8)
    iflux = 2.0 * np.pi / (nflux * ctx.beamset_info(0)["dflux"])
    for w in range(len(th)):
        assert _window(ctx, w) == window
        kept, full = ctx.get_spectrum(w), ref.get_spectrum(w)
        n = min(kept.size, full.size)
        assert kept.size == int(ctx.get_debug(w)["kmax_beamset"]) + 1
        # |spectrum| <= 1, its exponent's roundings some 1e-14
        np.testing.assert_allclose(kept[:n], full[:n], rtol=0, atol=1e-12)
        x = np.zeros(nflux // 2 + 1, dtype=complex)
        x[:kept.size] = kept
        x *= np.exp(-0.5 * (sigma * iflux * np.arange(x.size)) ** 2)
        x[0] = 1.0
        pd = np.maximum(np.fft.irfft(x) * nflux, 0.0)
        raw = ctx.get_pd(w, is_log="raw")[0]
        # the transforms' roundings: log2(n) of 1e-16 of the peak
        assert np.max(np.abs(raw - pd)) < 1e-14 * pd.max()


@pytest.mark.parametrize("binned", [True, False])
def test_walkers_of_every_window_in_one_batch(binned):
    """The window is each walker's own, by its noise multiplier: walkers of
    both windows and of none beside each other, whole and split, have the bits
    that they have alone."""
    print("[gpu-window-case] mixed %s" % binned, flush=True)
    inp = dict(workload.make_inputs(npix_side=120, seed=9))
    th = synth.walker_thetas(9, seed=23)
    th[:, len(inp["knots"])] = [1.0, 0.25, 0.1, 0.3, 0.0, 2.0, 0.1, 0.26, 1.1]
    want = [1, 2, 0, 1, 0, 1, 0, 2, 1]
    ctx = workload.build_context(inp, 65536, 512, binned=binned)
    alone = [ctx.loglike_batch(th[w:w + 1]) for w in range(len(th))]
    for parts in (0, 1, 2, 4):
        ctx.set_parts(parts)
        ll, st = ctx.loglike_batch(th)
        for w in range(len(th)):
            assert _window(ctx, w) == want[w]
            assert st[w] == alone[w][1][0] == 0
            assert ll[w] == alone[w][0][0]


def test_nodes_too_dense_for_windows():
    """A beam of small values between knots a factor of ten apart puts 2048
    nodes less than six grid points apart at point 2048, past the table of
    single points: eight points then lie in more than two node intervals, and
    the walkers keep the pruned transforms."""
    print("[gpu-window-case] dense nodes", flush=True)
    g, ps = synth.gaussian_beam()
    sigma, nflux, ninterp = 2e-5, 65536, 2048
    d = np.random.default_rng(3).normal(0.0, 1.3 * sigma, 3000)
    inp = dict(beam=(1.5e-4 * g).ravel(), pixsize=ps, data=d, sigma=sigma,
               minbeamval=1e-8, nbeamhist=120, nbins=200,
               knots=np.geomspace(0.1, 1.0, 5))
    th = np.array([[4.0, 3.5, 3.0, 2.5, 2.0, 1.0, 0, 0],
                   [4.1, 3.6, 3.1, 2.6, 2.1, 1.0, 0, 0]], dtype=np.float32)
    ctx = workload.build_context(inp, nflux, ninterp, binned=True)
    ctx.loglike_batch(th)
    x = ctx.get_rinterp(0)[0] / ctx.beamset_info(0)["dflux"]
    assert 2 < np.diff(x[x > 2048.0])[0] < 6
    L = build_oracle(inp, nflux, ninterp, True, th[0])
    for parts in (1, 2, 4):
        ctx.set_parts(parts)
        ll, st = ctx.loglike_batch(th)
        assert np.all(st == 0), st
        assert _window(ctx) == 0
        check_exact_parity(ctx, L, th, ll, tol=1e-6, nthreads=2)


@pytest.mark.parametrize("nflux,cut,window", [
    # 8, 16 (of both windows) and 32 points to a coarse one
    (65536, None, 1), (65536, 2.5e5, 2), (131072, None, 1), (131072, 2.5e5, 2),
    (262144, None, 1)])
def test_values_made_again_are_the_same_bits(nflux, cut, window):
    """The split search takes minima and peak from the matrix products of the
    inverse and the values beside them from sums made again: both round alike.
    The R range is some ten widths of the noise, so that the smallest value of
    the P(D) is far above rounding and not clamped."""
    print("[gpu-window-case] bits %d %s" % (nflux, cut), flush=True)
    sigma = 0.004
    inp = dict(workload.make_inputs(npix_side=40, seed=9, sigma=sigma))
    th = np.tile(synth.true_theta(), (24, 1))
    th[:, :len(inp["knots"])] -= 12.0  # hardly any sources
    th[:, len(inp["knots"])] = np.linspace(0.65, 1.0, len(th))
    ctx = workload.build_context(inp, nflux, 512, binned=True,
                                 spectral_cut=cut)
    ctx.set_rrange(0, 0.0, 10.2 * sigma)
    ll, st = ctx.loglike_batch(th)
    assert np.all(st == 0), st
    for w in range(len(th)):
        dbg = ctx.get_debug(w)
        raw = ctx.get_pd(w, is_log="raw")[0]
        assert _window(ctx, w) == window
        assert raw.max() == dbg["peak"]
        assert 0 < dbg["minval"] < 1e-5 * dbg["peak"]
        assert raw[int(dbg["minidx"])] == dbg["minval"] == raw.min()


@pytest.mark.parametrize("nflux", [65536, 131072])
def test_windowed_two_signed_beam(nflux):
    print("[gpu-window-case] negative beam %d" % nflux, flush=True)
    pix, ps = fitsio.read_beam(os.path.join(REFDATA,
                                            "band12_beam_f100.fits[0]"))
    inp = dict(workload.make_inputs(npix_side=120, seed=7), beam=pix,
               pixsize=ps)
    th = synth.walker_thetas(3, seed=13)
    ctx = workload.build_context(inp, nflux, 700, binned=False)
    lls = []
    for parts in (1, 2, 4):
        ctx.set_parts(parts)
        ll, st = ctx.loglike_batch(th)
        assert np.all(st == 0), st
        lls.append(ll)
    assert _window(ctx) == 1
    assert np.array_equal(lls[0], lls[1]) and np.array_equal(lls[0], lls[2])
    L = build_oracle(inp, nflux, 700, False, th[0])
    check_exact_parity(ctx, L, th, lls[0], tol=1e-6, nthreads=3)


@pytest.mark.parametrize("nflux,shift", [(65536, 0), (131072, 0), (65536, 3)])
def test_negative_fluxes_only_far_from_zero(nflux, shift):
    """An R range set by hand to a few mJy with 16 nodes up to 450 mJy: the
    negative node next to zero is then 170 grid points and more from it, past
    the head of the grid, and the head has no negative side.  The wrapped
    fluxes start at a multiple of eight points, so that windows are used, or
    three points on, where a group of eight has both signs and they are not.
    Against the pruned transforms, which a cut that keeps more than the
    windows hold selects.  (The reference fills no negative fluxes where the
    lowest node is below the range: its index wraps.)"""
    print("[gpu-window-case] far negative %d %d" % (nflux, shift), flush=True)
    g, ps = synth.gaussian_beam()
    sigma = 0.0005
    d = np.random.default_rng(3).normal(0.0, 1.2 * sigma, 3000)
    inp = dict(beam=np.hstack([g, -0.9 * g]).ravel(), pixsize=ps, data=d,
               sigma=sigma, minbeamval=1e-6, nbeamhist=120, nbins=200,
               knots=synth.knot_positions())
    th = synth.walker_thetas(3, seed=4)
    th[:, :len(inp["knots"])] -= 5.5
    full = 0.010
    neg = (nflux // 2 + shift + 0.5) * full / (nflux - 1)
    out = []
    for cut in (64.0, 3e5):
        ctx = workload.build_context(inp, nflux, 16, binned=True,
                                     spectral_cut=cut)
        ctx.set_rrange(0, -neg, full - neg)
        for parts in (1, 2, 4):
            ctx.set_parts(parts)
            ll, st = ctx.loglike_batch(th)
            assert np.all(st == 0), st
            assert _window(ctx) == (1 if shift == 0 and cut == 64.0 else 0)
            out.append((ll, ctx.get_debug(0)))
    ref, dref = out[-1]
    for ll, dbg in out:
        # sums of 1e4 to 1e5 positive terms, each within some 1e-16
        for key in ("mn", "var_noi", "r0"):
            assert dbg[key] == pytest.approx(dref[key], rel=1e-10), key
        np.testing.assert_allclose(ll, ref, rtol=0, atol=1e-8)


@pytest.mark.parametrize("sigmas,window", [((0.0006, 0.0025), 2),
                                           ((0.0025, 0.0006), 2),
                                           ((0.0025, 0.004), 1)])
def test_datasets_of_different_noise(sigmas, window):
    """Two datasets share the spectrum, kept up to the narrower noise's last
    index: more of them than a workgroup has threads in the second window,
    and zeros between in the other dataset's transform."""
    print("[gpu-window-case] two datasets %g %g" % sigmas, flush=True)
    nflux, ninterp = 65536, 512
    inp = dict(workload.make_inputs(npix_side=120, seed=9, sigma=sigmas[0]))
    other = dict(workload.make_inputs(npix_side=100, seed=10, sigma=sigmas[1]))
    th = synth.walker_thetas(3, seed=25)
    ctx = workload.build_context(inp, nflux, ninterp, binned=True)
    ctx.add_field(0, pix=other["data"], sigma_base=sigmas[1])
    ctx.prepare()
    L = build_oracle(inp, nflux, ninterp, True, th[0])
    L.add_field(0, pix=other["data"], sigma_base=sigmas[1])
    L.finalize(th[0])
    L.set_precise(1)
    ref, rst = L.loglike_batch(th, 3)
    assert np.all(rst == 0), rst
    lls = []
    for parts in (1, 2, 4):
        ctx.set_parts(parts)
        ll, st = ctx.loglike_batch(th)
        assert np.all(st == 0), st
        assert _window(ctx) == window
        # the contract of every 1D path, for each dataset
        np.testing.assert_allclose(ll, ref, rtol=0, atol=2e-6)
        lls.append(ll)
    assert np.array_equal(lls[0], lls[1]) and np.array_equal(lls[0], lls[2])
