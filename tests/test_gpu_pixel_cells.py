"""The unbinned 1D sum by cells of the P(D) grid against the CPU oracle and
a pixel-by-pixel sum: few pixels, repeated and equal ones, pixels on either
side of the grid, and data far beyond it (no rank table)."""
import numpy as np
import pytest

import pyoracle as O
from pofd_affine_amd import _lib, synth, workload

pytestmark = pytest.mark.gpu

NF, NI = 8192, 256


def _data(kind):
    rng = np.random.default_rng(11)
    core = rng.normal(0.0, 0.004, 700000)
    if kind.startswith("n"):
        return core[:int(kind[1:])]
    if kind == "constant":
        return np.full(5000, 0.00125)
    if kind == "repeated":  # 64 values, many pixels each
        return np.repeat(core[:64], 101)
    if kind == "dense":  # several steps of the rank table per cell
        return np.concatenate([core, rng.uniform(-0.02, 0.5, 300)])
    if kind == "wide":  # below and above every flux of the grid
        return np.concatenate([core[:3000], [-0.8, -0.3, 0.9, 2.5]])
    raise ValueError(kind)


def _pixel_sum(pd, minflux, dflux, d):
    """PD::getLogLikeUnbinned (src/PD.cc:628-677), pixel by pixel."""
    n = pd.size
    i = np.clip((d - minflux) / dflux, 0, n - 2).astype(np.int64)
    t = (d - minflux) / dflux - i
    v = (1.0 - t) * pd[i] + t * pd[i + 1]
    v = np.where(d <= minflux, pd[0], v)
    v = np.where(d >= minflux + (n - 2) * dflux, pd[-1], v)
    return np.log(2.0) * v.sum()


@pytest.mark.parametrize("kind,rmax", [
    ("n1", None), ("n2", None), ("n63", None), ("n64", None), ("n65", None),
    ("n4097", None), ("constant", None), ("repeated", None), ("dense", None),
    ("wide", None),
    # the R range set by hand: pixels beyond the grid's last flux, then data
    # that span more than four grids
    ("wide", 0.75), ("far", 0.75)])
def test_unbinned_sum_by_cells(kind, rmax):
    print("[gpu-cells-case] %s %s" % (kind, rmax), flush=True)
    d = _data("wide" if kind == "far" else kind)
    if kind == "far":
        d = np.concatenate([d, [6.0, -1.5]])
    inp = workload.make_inputs(npix_side=64, seed=3)
    th = synth.walker_thetas(3, seed=5)
    ctx = _lib.Context(0)
    ctx.configure(NF, NI, inp["knots"])
    b = ctx.add_beamset(_lib.Beam(inp["beam"], inp["pixsize"],
                                  inp["minbeamval"], inp["nbeamhist"]))
    ctx.add_field(b, pix=d, sigma_base=0.0025)
    ctx.prepare()
    if rmax:
        ctx.set_rrange(b, 0.0, rmax)
    ll, st = ctx.loglike_batch(th)
    assert np.all(st == 0), st
    # roundings of some 1e-16 of the terms, at most 60 a pixel, and of 1e-11
    # of a cell (the double fluxes' own) in each pixel's place between two
    # values that differ by less than 1
    tol = d.size * (60.0 * 1e-15 + 1e-11)
    var = 0.0025 ** 2
    off = -0.5 * d.size * (np.log(2.0 * np.pi * var) + 1.0)
    for w in range(len(th)):
        pd, mf, df = ctx.get_pd(w, is_log=True)
        assert ll[w] + off == pytest.approx(_pixel_sum(pd, mf, df, d),
                                            rel=0, abs=tol)
    # (a pixel where P(D) is nothing but a transform's rounding has no value
    # that two transforms share)
    if kind not in ("wide", "far"):
        L = O.Like(NF, NI, inp["knots"])
        bm = O.Beam(inp["beam"], inp["pixsize"], inp["minbeamval"],
                    inp["nbeamhist"])
        L.add_field(L.add_beamset(bm), pix=d, sigma_base=0.0025)
        L.finalize(th[0])
        ref, rst = L.loglike_batch(th, 1)
        assert np.all(rst == 0), rst
        np.testing.assert_allclose(ll, ref, rtol=0, atol=1e-6 + tol)
