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
