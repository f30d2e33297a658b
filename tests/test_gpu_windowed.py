"""The windowed 1D transforms against the pruned ones and the CPU oracle at
the edges of their range: every grid size that has a window, both coarse
sizes (a narrow dataset moves the kept spectrum from one to the other and
past both), split over 1, 2 and 4 workgroups, a two-signed beam, and nodes
so dense that no window is used."""
import os

import numpy as np
import pytest

from conftest import REFDATA
from oracle_side import build_oracle, check_exact_parity
from pofd_affine_amd import fitsio, synth, workload

pytestmark = pytest.mark.gpu


def _nrows(ctx):
    """Kept rows of the pruned transform; 0: the windowed one ran."""
    return int(ctx.get_debug(0)["nrows"])


@pytest.mark.parametrize("nflux,ninterp,sigma,windowed", [
    # below 2^16 there is no window
    (32768, 512, 0.0025, False), (65536, 400, 0.0025, True),
    (65536, 1023, 0.0025, True), (131072, 2048, 0.0025, True),
    (262144, 2048, 0.0025, True),
    # kept spectra above 1024 (the second window) and above 2048 (none)
    (65536, 512, 0.0007, True), (131072, 2048, 0.0007, True),
    (65536, 512, 0.0003, False)])
def test_windowed_against_exact(nflux, ninterp, sigma, windowed):
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
        assert (_nrows(ctx) == 0) == windowed
    assert np.array_equal(lls[0], lls[1]) and np.array_equal(lls[0], lls[2])
    L = build_oracle(inp, nflux, ninterp, True, th[0])
    # the contract of every 1D path: 1e-6 of the exact-math value
    check_exact_parity(ctx, L, th, lls[2], tol=1e-6, nthreads=3)


@pytest.mark.parametrize("cut", [746.0, 12.0])
def test_other_spectral_cuts(cut):
    """A cut that keeps twice the spectrum takes the second window, one that
    keeps half of it must not take a smaller one than the noise allows."""
    print("[gpu-window-case] cut %g" % cut, flush=True)
    inp = dict(workload.make_inputs(npix_side=120, seed=9))
    th = synth.walker_thetas(3, seed=22)
    ref = workload.build_context(inp, 65536, 512, binned=True)
    ctx = workload.build_context(inp, 65536, 512, binned=True, spectral_cut=cut)
    a, sa = ref.loglike_batch(th)
    b, sb = ctx.loglike_batch(th)
    assert np.all(sa == 0) and np.all(sb == 0)
    # e^-12 of the DC term is left out at the lower cut: 6e-6 of the peak in
    # P(D), so only the higher cut is compared with the default one
    if cut > 64:
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-8)
    else:
        L = build_oracle(inp, 65536, 512, True, th[0])
        r, _ = L.loglike_batch(th, 3)
        assert np.all(np.isfinite(b)) and np.max(np.abs(b - r)) < 1e-2 * np.max(np.abs(r))


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
        assert dbg["window"] == window
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
    assert _nrows(ctx) == 0
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
            assert (_nrows(ctx) == 0) == (shift == 0 and cut == 64.0)
            out.append((ll, ctx.get_debug(0)))
    ref, dref = out[-1]
    for ll, dbg in out:
        # sums of 1e4 to 1e5 positive terms, each within some 1e-16
        for key in ("mn", "var_noi", "r0"):
            assert dbg[key] == pytest.approx(dref[key], rel=1e-10), key
        np.testing.assert_allclose(ll, ref, rtol=0, atol=1e-8)
