"""The work this library is used for, as cases that can be timed and checked.

A case names one call through the public entry points: a batch of one-band
or two-band P(D) log likelihoods (the call a sampler makes for every step), a
few steps of the device-resident sampler, or one forward and backward pass of
the surrogate network.  ``prepare`` makes the data and the context a fit keeps
for its whole length, ``run`` is one call, ``work`` is what that call cannot do
without, and ``exact`` restates the likelihood in plain numpy and torch.
"""
import math

import numpy as np
import torch

from pofd_affine_amd import _lib

# ------------------------------------------------------------------ the cases


def listed():
    """One call each of the ways the library is used, smallest to largest."""
    return [
        # one getLogLike at one theta from host buffers on the 720 x 720 map,
        # what a program without a batch (or a slave of a farm) asks for
        dict(name="1d_getlike_1w", kind="like1d", nflux=131072, ninterp=2048, walkers=1,
             side=720, data="unbinned", beam="gauss", entry="host", sigma=0.0025),
        # a quick fit: short transform, few nodes, small binned map
        dict(name="1d_small_4w", kind="like1d", nflux=32768, ninterp=512, walkers=4,
             side=200, data="binned", beam="gauss", entry="host", sigma=0.0025),
        # half of a 40-walker ensemble, the reference's own chain size
        dict(name="1d_chain_half_20w", kind="like1d", nflux=131072, ninterp=2048, walkers=20,
             side=720, data="unbinned", beam="gauss", entry="device", sigma=0.0025),
        # half of a 512-walker ensemble against a binned map (the benchmark)
        dict(name="1d_binned_256w", kind="like1d", nflux=131072, ninterp=2048, walkers=256,
             side=1000, data="binned", beam="gauss", entry="device", sigma=0.0025),
        # the same against the million pixels themselves
        dict(name="1d_unbinned_256w", kind="like1d", nflux=131072, ninterp=2048, walkers=256,
             side=1000, data="unbinned", beam="gauss", entry="device", sigma=0.0025),
        # a filtered (two-signed) beam, two datasets, a sigma prior, and a
        # batch that fills no whole number of anything
        dict(name="1d_two_fields_157w", kind="like1d", nflux=65536, ninterp=1024, walkers=157,
             side=501, data="both", beam="signed", entry="device", sigma=0.003),
        # the largest transform and a four-million-pixel map
        dict(name="1d_large_96w", kind="like1d", nflux=262144, ninterp=2048, walkers=96,
             side=2000, data="unbinned", beam="gauss", entry="device", sigma=0.0018),
        # two bands: a small grid and map
        dict(name="2d_small_6w", kind="like2d", n=512, nedge=64, walkers=6, side=120,
             data="unbinned", entry="host"),
        # two bands, binned pairs, an odd batch
        dict(name="2d_binned_17w", kind="like2d", n=1024, nedge=128, walkers=17, side=500,
             data="binned", entry="device"),
        # two bands at full size (the benchmark)
        dict(name="2d_batch_32w", kind="like2d", n=2048, nedge=256, walkers=32, side=1000,
             data="unbinned", entry="device"),
        # steps of the 512-walker stretch move on the binned likelihood
        dict(name="chain_512w_4steps", kind="chain1d", nflux=131072, ninterp=2048, walkers=512,
             side=500, steps=4),
        # loss and gradient of the surrogate over one training batch
        dict(name="surrogate_grad_512", kind="mlp", nin=8, hidden=256, rows=512),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case over the ranges above."""
    kind = rng.choice(["like1d"] * 5 + ["like2d"] * 3 + ["chain1d", "mlp"])
    if kind == "like1d":
        nflux = 1 << rng.randint(13, 18)
        # walkers x transform length no more than the largest listed batch
        most = min(300, (256 * 131072) // nflux)
        walkers = int(round(_log(rng, 1, most + 0.49)))
        side = int(round(_log(rng, 150, 1000)))
        return dict(kind=kind, nflux=nflux, ninterp=rng.randint(400, 2048), walkers=walkers,
                    side=side, data=rng.choice(["binned", "unbinned", "unbinned", "both"]),
                    beam=rng.choice(["gauss", "gauss", "signed"]),
                    entry=rng.choice(["host", "device"]), sigma=rng.uniform(0.0015, 0.004))
    if kind == "like2d":
        n = 1 << rng.randint(8, 11)
        walkers = int(round(_log(rng, 1, min(48, 32 * 2048 * 2048 // (n * n)) + 0.49)))
        return dict(kind=kind, n=n, nedge=rng.randint(n // 16, n // 8), walkers=walkers,
                    side=int(round(_log(rng, 100, 1000))),
                    data=rng.choice(["binned", "unbinned"]),
                    entry=rng.choice(["host", "device"]))
    if kind == "chain1d":
        return dict(kind=kind, nflux=1 << rng.randint(15, 17), ninterp=rng.randint(400, 2048),
                    walkers=2 * rng.randint(20, 256), side=int(round(_log(rng, 150, 500))),
                    steps=rng.randint(1, 4))
    return dict(kind=kind, nin=rng.randint(4, 14), hidden=rng.choice([64, 128, 200, 256]),
                rows=int(round(_log(rng, 64, 4096))))


# ------------------------------------------------------------------- the data

KNOTS = np.array([2.0, 5.0, 10.0, 20.0, 45.0, 100.0, 200.0, 450.0]) * 1e-3
KNOTS2 = np.array([3.0, 8.0, 20.0, 50.0, 120.0, 300.0]) * 1e-3
COLOUR_POS = np.array([5.0, 30.0, 200.0]) * 1e-3
COLOUR_SIGMA = np.array([0.1, 0.2, 0.3])
COLOUR_OFFSET = np.array([-0.2, -0.05, 0.1])
SIGMA2D = (0.0025, 0.0027)
PIX = 6.0                       # arcsec
MINBEAM, NBEAMHIST = 1e-6, 120
SIGMA_PRIOR = 0.05


def _counts(s):
    """dN/dS: a power law of slope -2.2 to 20 mJy and -3.5 above."""
    s = np.asarray(s, dtype=np.float64)
    at = 5e6 * 2.0 ** -2.2
    return np.where(s <= 0.02, 5e6 * (s / 0.01) ** -2.2, at * (s / 0.02) ** -3.5)


def _sources(rng, area, smin, smax):
    """Poisson-drawn source fluxes (inverse CDF on a fine table)."""
    edge = np.geomspace(smin, smax, 4097)
    mid = np.sqrt(edge[1:] * edge[:-1])
    cum = np.concatenate([[0.0], np.cumsum(_counts(mid) * np.diff(edge))])
    return np.interp(rng.random(rng.poisson(area * cum[-1])) * cum[-1], cum, edge)


def _gauss(half, fwhm):
    y, x = np.mgrid[-half:half + 1, -half:half + 1].astype(np.float64)
    s = fwhm / (2.0 * math.sqrt(2.0 * math.log(2.0))) / PIX
    return np.exp(-0.5 * (x * x + y * y) / (s * s))


def _beam(kind):
    """A Gaussian beam cut at nine FWHM, or the same with the negative ring
    that filtering a map leaves."""
    b = _gauss(int(4.5 * 18.1 / PIX), 18.1)
    return b if kind == "gauss" else b - 0.08 * _gauss(b.shape[0] // 2, 40.0)


def _observe(rng, side, pos, flux, beam, sigma):
    img = np.bincount(pos, weights=flux, minlength=side * side).reshape(side, side)
    kern = np.zeros((side, side))
    h = beam.shape[0] // 2
    kern[:2 * h + 1, :2 * h + 1] = beam
    kern = np.roll(kern, (-h, -h), (0, 1))
    m = np.fft.irfft2(np.fft.rfft2(img) * np.fft.rfft2(kern), s=img.shape)
    d = (m + rng.normal(0.0, sigma, img.shape)).ravel()
    return d - d.mean()


def _bin1(d, n):
    lo, step = d.min(), (d.max() - d.min()) / (n - 1)
    return np.bincount(((d - lo) * (1.0 / step) + 0.5).astype(np.int64),
                       minlength=n).astype(np.uint32), lo, step


def _inputs1(case, seed):
    """Fields (data, sigma, bins or None) and walkers of a one-band case."""
    rng = np.random.default_rng(1000003 + seed)
    beam = _beam(case.get("beam", "gauss"))
    side, data = case["side"], case.get("data", "binned")
    sigma = case.get("sigma", 0.0025)
    fields = []
    for k, how in enumerate(("binned", "unbinned") if data == "both" else (data,)):
        flux = _sources(rng, (side * PIX / 3600.0) ** 2, 0.001, 0.6)
        pos = rng.integers(0, side * side, flux.size)
        d = _observe(rng, side, pos, flux, beam, sigma * (1.0 + 0.2 * k))
        fields.append((d, sigma * (1.0 + 0.2 * k), _bin1(d, 1000) if how == "binned" else None))
    th = np.zeros((case["walkers"], KNOTS.size + 3))
    th[:, :KNOTS.size] = np.log10(_counts(KNOTS)) + rng.normal(0, 0.05, (len(th), KNOTS.size))
    th[:, KNOTS.size] = 1.0 + rng.normal(0.0, 0.03, len(th))
    return beam, fields, th.astype(np.float32)


def _inputs2(case, seed):
    rng = np.random.default_rng(2000003 + seed)
    side = case["side"]
    half = int(4.5 * 25.2 / PIX)
    beams = _gauss(half, 18.1), _gauss(half, 25.2)
    s1 = _sources(rng, (side * PIX / 3600.0) ** 2, KNOTS2[0], KNOTS2[-1])
    s2 = s1 * np.exp(rng.normal(np.interp(s1, COLOUR_POS, COLOUR_OFFSET),
                                np.interp(s1, COLOUR_POS, COLOUR_SIGMA)))
    pos = rng.integers(0, side * side, s1.size)
    d = [_observe(rng, side, pos, s, b, sg) for s, b, sg in zip((s1, s2), beams, SIGMA2D)]
    base = np.concatenate([np.log10(_counts(KNOTS2)), COLOUR_SIGMA, COLOUR_OFFSET, [1.0, 1.0],
                           np.zeros(4)])
    th = np.tile(base, (case["walkers"], 1))
    th[:, :6] += rng.normal(0.0, 0.05, (len(th), 6))
    th[:, 6:12] += rng.normal(0.0, 0.01, (len(th), 6))
    th[:, 12:14] += rng.normal(0.0, 0.03, (len(th), 2))
    # the flux range of the fit: knots, colours and noise with some to spare
    rng2 = 1.1 * KNOTS2[-1] * np.array([1.0, math.exp(0.1 + 3 * 0.3)])
    hi = [max(r + 7.5 * s, x.max()) for r, s, x in zip(rng2, SIGMA2D, d)]
    return beams, d, th.astype(np.float32), hi


def _bin2(d, n):
    (i1, lo1, st1), (i2, lo2, st2) = (
        (((x - x.min()) * ((n - 1) / (x.max() - x.min())) + 0.5).astype(np.int64), x.min(),
         (x.max() - x.min()) / (n - 1)) for x in d)
    return (np.bincount(i1 * n + i2, minlength=n * n).astype(np.uint32).reshape(n, n),
            np.array([lo1, st1, lo2, st2]))


def _mlp_inputs(case, seed):
    rng = np.random.default_rng(3000003 + seed)
    nin, h = case["nin"], case["hidden"]
    x = rng.normal(0.0, 1.0, (case["rows"], nin)).astype(np.float32)
    y = -0.5 * (x.astype(np.float64) ** 2).sum(1) + 0.2 * np.sin(3.0 * x[:, 0])
    shapes = [(h, nin), (h,), (h, h), (h,), (h, h), (h,), (h,), (1,)]
    return x, y, [rng.normal(0.0, 1.0 / math.sqrt(s[-1] if len(s) > 1 else h), s)
                  .astype(np.float32) for s in shapes]


# ------------------------------------------------------------- prepare and run


def _context1(case, beam, fields):
    ctx = _lib.Context(0)
    ctx.configure(case["nflux"], case["ninterp"], KNOTS)
    b = ctx.add_beamset(_lib.Beam(beam.ravel(), PIX, MINBEAM, NBEAMHIST))
    for d, sigma, bins in fields:
        if bins is None:
            ctx.add_field(b, pix=d, sigma_base=sigma)
        else:
            ctx.add_field(b, bins=bins[0], bincent0=bins[1], bindelta=bins[2],
                          sigma_base=sigma, npix=d.size)
    if case.get("data") == "both":
        ctx.set_priors(sigma_width=SIGMA_PRIOR)
    ctx.prepare()
    return ctx


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, case=case)
    if kind == "mlp":
        x, y, w = _mlp_inputs(case, seed)
        net = _lib.Mlp(case["nin"], case["hidden"], seed=1)
        flat = np.zeros(net.nparams, dtype=np.float32)
        for o, v in zip(net.offsets, w):
            flat[o:o + v.size] = v.ravel()
        net.set_params(flat)
        return dict(st, net=net, x=x, y=y, sizes=[v.size for v in w])
    if kind == "like2d":
        beams, d, th, hi = _inputs2(case, seed)
        ctx = _lib.Context2(0)
        ctx.configure2d(case["n"], KNOTS2, COLOUR_POS, COLOUR_POS, nedge=case["nedge"])
        b = ctx.add_beamset2d(_lib.DoubleBeam(beams[0], beams[1], PIX, MINBEAM, NBEAMHIST))
        bins, info = _bin2(d, 300) if case["data"] == "binned" else (None, None)
        ctx.add_field2d(b, d[0], d[1], SIGMA2D[0], SIGMA2D[1], bins=bins, bininfo=info)
        ctx.prepare2d(th[0])
        ctx.set_rrange2d(b, [0.0, hi[0], 0.0, hi[1]])
    else:
        beam, fields, th = _inputs1(case, seed)
        ctx = _context1(case, beam, fields)
        if kind == "chain1d":
            ens = _lib.Ensemble(ctx, _lib.TARGET_1D, case["walkers"], th.shape[1], seed=seed + 1)
            # the knots are fitted; the sigma multiplier and the bonus
            # parameters are fixed
            ens.set_param_state([0] * KNOTS.size + [1] * (th.shape[1] - KNOTS.size))
            th[:, KNOTS.size] = 1.0
            return dict(st, ens=ens, theta=th)
    st.update(ctx=ctx, theta=th)
    if case["entry"] == "device":
        w = len(th)
        st.update(d_theta=torch.from_numpy(th).cuda(),
                  d_ll=torch.zeros(w, dtype=torch.float64, device="cuda"),
                  d_st=torch.zeros(w, dtype=torch.int32, device="cuda"))
    return st


def run(state):
    kind = state["kind"]
    if kind == "mlp":
        loss, g = state["net"].loss_grad(state["x"], state["y"])
        # the padding between the layers' blocks is not a result
        return dict(loss=loss, grad=[g[o:o + n] for o, n in zip(state["net"].offsets,
                                                                state["sizes"])])
    if kind == "chain1d":
        ens = state["ens"]
        ens.set_positions(state["theta"])
        ens.clear_chain()
        ens.run(state["case"]["steps"])
        th, ll, acc, _ = ens.state()
        return dict(theta=th, loglike=ll, accepted=acc.astype(np.int64))
    ctx = state["ctx"]
    two = kind == "like2d"
    if "d_theta" not in state:
        ll, s = (ctx.loglike2d_batch if two else ctx.loglike_batch)(state["theta"])
        return dict(loglike=ll, status=s)
    th, ll, s = state["d_theta"], state["d_ll"], state["d_st"]
    call = ctx.loglike2d_batch_device if two else ctx.loglike_batch_device
    call(th.data_ptr(), th.shape[0], th.shape[1], ll.data_ptr(), s.data_ptr(), 0)
    return dict(loglike=ll, status=s)


# --------------------------------------------------------- work and tolerance


def work(case):
    """Bytes: parameters, data and tables in, results out, once each.  Flops:
    R on the flux grid, one transform each way per dataset, the data sum."""
    kind = case["kind"]
    w = case.get("walkers", 0)
    if kind == "mlp":
        per = 2 * (case["nin"] * case["hidden"] + 2 * case["hidden"] ** 2 + case["hidden"])
        npar = per // 2
        return {"bytes": 4 * (case["rows"] * (case["nin"] + 2) + 2 * npar),
                "flops": 3 * case["rows"] * per}
    if kind == "like2d":
        n, npix = case["n"], case["side"] ** 2
        binned = case["data"] == "binned"
        items = 300 * 300 if binned else npix
        per = n * n * (23 * 20 + 2 * 2.5 * 2 * math.log2(n) + 10) + 12 * items
        return {"bytes": items * (4 if binned else 16) + w * 84, "flops": w * per}
    data, npix = case.get("data", "binned"), case["side"] ** 2
    nb = data in ("binned", "both")
    nu = data in ("unbinned", "both")
    n, nf = case["nflux"], 1 + (data == "both")
    per = (n * (30 + (1 + nf) * 2.5 * math.log2(n) + 6 * nf)
           + case["ninterp"] * 65 * 20 + nb * 1000 * 30 + nu * npix * 8)
    evals = w * (case["steps"] + 1) if kind == "chain1d" else w
    return {"bytes": nb * 4000 + nu * 8 * npix + w * 56 + 2 * n + 9 * 65 * case["ninterp"],
            "flops": evals * per}


def tolerance(case):
    """Double-precision log likelihoods of some 1e5 agree with the plain
    restating below to a few 1e-14 and, where a two-signed beam leaves P(D) a
    faint tail, to 2e-13; where rounding moves the split search by one index
    a walker moves by a few 1e-6, 1e-11 of it.  Two networks in bfloat16
    differ by roundings of single activations."""
    if case["kind"] == "mlp":
        return {"rel": 4e-3, "max": 0.1}
    return {"rel": 1e-11, "max": 1e-10}


# ------------------------------------------------------------- plain restating


def _spline(x, y):
    """Coefficients [4, n-1, ...] of the natural cubic spline through (x, y)."""
    n = len(x)
    h = np.diff(x)
    a = np.zeros((n, n))
    a[0, 0] = a[-1, -1] = 1.0
    i = np.arange(1, n - 1)
    a[i, i - 1], a[i, i], a[i, i + 1] = h[:-1], 2 * (h[:-1] + h[1:]), h[1:]
    hh = h.reshape((-1,) + (1,) * (y.ndim - 1))
    s = np.diff(y, axis=0) / hh
    r = np.zeros_like(y)
    r[1:-1] = 3.0 * np.diff(s, axis=0)
    c = torch.linalg.solve(torch.from_numpy(a), torch.from_numpy(
        np.ascontiguousarray(r.reshape(n, -1)))).numpy().reshape(y.shape)
    return np.stack([y[:-1], s - hh * (c[1:] + 2 * c[:-1]) / 3.0, c[:-1],
                     np.diff(c, axis=0) / (3.0 * hh)])


def _at(x, cf, v):
    k = np.clip(np.searchsorted(x, v, side="right") - 1, 0, len(x) - 2)
    d = v - x[k]
    c = cf[:, k]
    return c[0] + d * (c[1] + d * (c[2] + d * c[3]))


def _split(p, bot, top, f2):
    """findSplitPoint: where the P(D) is cut and rotated (the whole search
    range is inside the array); None where the search fails."""
    peak = p.max()
    mi = bot + int(np.argmin(p[bot:top + 1]))
    mv = p[mi]
    if mv > f2 * peak or bot >= top:
        return None
    if mi > 17:
        run = p[mi - 17:mi]
        if np.all(np.diff(run) < 0):
            return mi
        jitter = 1.1 * (run.sum() + mv) / 18.0
    else:
        jitter = 5e-14 * peak
        if mv > jitter:
            return mi
    if mv <= 0.0:
        mv = max(p[max(mi - 3, 0):min(mi + 3, top - 3)].max(initial=0.0), mv)
    if mv > 0:
        jitter = min(jitter, 5 * mv)
    if p[top] < jitter:
        return None
    low = np.nonzero(p[bot:top] < jitter)[0]
    return bot + int(low[-1]) + 1 if low.size else None


def _log2(p):
    return np.where(p > 0, np.log2(np.where(p > 0, p, 1.0)), -30.0)


def _hist1(v):
    """Beam pixels in 120 log bins: weights and inverse mean values."""
    lo, hi = np.log2(v.min()) - math.log2(1.001), np.log2(v.max()) + math.log2(1.001)
    b = ((np.log2(v) - lo) / ((hi - lo) / NBEAMHIST)).astype(np.int64)
    w = np.bincount(b, minlength=NBEAMHIST)
    s = np.bincount(b, weights=v, minlength=NBEAMHIST)
    return w[w > 0].astype(np.float64), w[w > 0] / s[w > 0]


def _exact1(case, beam, fields, th):
    n, ni = case["nflux"], case["ninterp"]
    pix = np.sort(beam.ravel())
    pos, neg = pix[pix > MINBEAM], -pix[pix < -MINBEAM]
    smax = max(f[1] for f in fields)
    lo = -1.05 * KNOTS[-1] * neg.max() if neg.size else 0.0
    hi = 1.05 * KNOTS[-1] * pos.max() + 7.5 * smax
    ranges = [(d.min(), d.max()) if b is None else (b[1], b[1] + 999 * b[2])
              for d, _, b in fields]
    hi = max(hi, max(r[1] for r in ranges))
    if neg.size:
        lo = min(lo, min(r[0] for r in ranges))
    dflux, wrap, minr = hi / (n - 1), n - 1, 0.0
    if lo < 0:
        dflux = (hi - lo) / (n - 1)
        dflux = hi / (n - math.floor(-lo / dflux) - 1.0)
        wrap = int(hi / dflux + 0.9999999999)
        minr = (wrap + 1) * dflux - n * dflux
    flux = np.arange(n) * dflux
    flux[wrap + 1:] += minr - (wrap + 1) * dflux
    lk = np.log2(KNOTS)
    cf = _spline(lk, (math.log2(10.0) * th[:, :KNOTS.size].astype(np.float64)).T.copy())
    r = np.zeros((len(th), n))
    for sgn, v in ((1, pos), (-1, neg)):
        if not v.size:
            continue
        wt, inv = _hist1(v)
        x0, x1 = KNOTS[0] * 1e-5, KNOTS[-1] * v.max()
        step = 0.001 * (x1 - x0) / (ni - 1)
        x1 -= step
        if sgn < 0:
            x0 += step
        x = x0 * 2.0 ** (np.arange(ni) * (math.log2(x1 / x0) / (ni - 1)))
        s = x[:, None] * inv
        ok = (s >= KNOTS[0]) & (s < KNOTS[-1])
        ls = np.log2(s)
        k = np.clip(np.searchsorted(lk, ls, side="right") - 1, 0, len(lk) - 2)
        d = ls - lk[k]
        at = np.empty((ni, len(th)))
        for i in range(len(th)):
            c = cf[:, :, i][:, k]
            e = np.exp2(c[0] + d * (c[1] + d * (c[2] + d * c[3])))
            at[:, i] = (np.where(ok, e, 0.0) * (wt * inv)).sum(1) * (PIX / 3600.0) ** 2
        sc = _spline(x, _log2(at))
        sel = np.nonzero((sgn * flux >= x[0]) & (sgn * flux <= x[-1]))[0]
        kk = np.clip(np.searchsorted(x, sgn * flux[sel], side="right") - 1, 0, ni - 2)
        dx = sgn * flux[sel] - x[kk]
        for i in range(len(th)):
            c = sc[:, :, i][:, kk]
            r[i, sel] = np.exp2(c[0] + dx * (c[1] + dx * (c[2] + dx * c[3]))) * dflux
    out = np.zeros(len(th))
    w = 2.0 * math.pi / (n * dflux) * np.arange(n // 2 + 1)
    data = []
    for d, sg, b in fields:
        c = np.sort(d) if b is None else b[1] + np.nonzero(b[0])[0] * b[2]
        data.append((c, 1.0 if b is None else b[0][b[0] > 0].astype(np.float64)))
    for i in range(len(th)):
        sm = float(th[i, KNOTS.size])
        wt = np.ones(n)
        wt[wrap] = 0.5
        mn = (wt * flux * r[i]).sum()
        var = (wt * flux * flux * r[i]).sum()
        if wrap < n - 1:  # the lower edge's correction, as the model makes it
            mn -= 0.5 * minr * r[i, wrap - 1]
            var -= 0.5 * minr * minr * r[i, wrap - 1]
        f = np.fft.rfft(r[i])
        # R^(k) - R^(0) as one sum, so that R's peak does not round it
        ph = f - f[0].real
        if math.sqrt(var) > dflux and abs(mn) > dflux:
            ph = ph + 1j * mn * w
        for (c, nb), (d, s0, b) in zip(data, fields):
            s = sm * s0
            g = np.maximum(np.fft.irfft(np.exp(ph - 0.5 * s * s * w * w), n), 0.0)
            sgp = math.sqrt(var + s * s)
            sgn_ = s if 9 * s * s > var else sgp
            bot = int(2.5 * sgp / dflux)
            top = wrap if 2.5 * sgp > abs(minr) else int(-(2.5 * sgn_ + minr) / dflux + wrap + 1)
            sp = _split(g, bot, top, 1e-5)
            if sp is None:
                out[i] = math.nan
                break
            g = np.roll(g, -sp)
            g /= (g.sum() - 0.5 * (g[0] + g[-1])) * dflux
            m0 = -((np.arange(n) * g).sum() - 0.5 * (n - 1) * g[-1]) * dflux * dflux
            lg = _log2(g)
            t = np.clip((c - m0) / dflux, 0.0, n - 1.0)
            j = np.minimum(t.astype(np.int64), n - 2)
            t = np.where(c > m0 + (n - 2) * dflux, 1.0, t - j)
            j = np.where(c > m0 + (n - 2) * dflux, n - 2, j)
            ll = math.log(2.0) * (nb * ((1 - t) * lg[j] + t * lg[j + 1])).sum()
            out[i] += ll + 0.5 * d.size * (math.log(2 * math.pi * s0 * s0) + 1.0)
        if case["data"] == "both":
            v = (sm - 1.0) / SIGMA_PRIOR
            out[i] -= 0.5 * math.log(2 * math.pi) + math.log(SIGMA_PRIOR) + 0.5 * v * v
    return out


def _exact2(case, beams, d, th, hi):
    n, ne = case["n"], case["nedge"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    b1, b2 = beams[0].ravel(), beams[1].ravel()
    ok = (b1 > MINBEAM) & (b2 > MINBEAM)
    b1, b2 = b1[ok], b2[ok]
    pad, idx = math.log2(1.001), []
    for b in (b1, b2):
        lo, up = np.log2(b.min()) - pad, np.log2(b.max()) + pad
        idx.append(((np.log2(b) - lo) * (NBEAMHIST / (up - lo))).astype(np.int64))
    cell = idx[0] * NBEAMHIST + idx[1]
    wt = np.bincount(cell, minlength=NBEAMHIST ** 2)
    on = wt > 0
    s1, s2 = (np.bincount(cell, weights=b, minlength=NBEAMHIST ** 2)[on] for b in (b1, b2))
    wt = wt[on].astype(np.float64)
    inv1, lratio = wt / s1, np.log(s1 / s2)
    df = [h / (n - 1) for h in hi]
    f1, f2 = np.arange(n) * df[0], np.arange(n) * df[1]
    low = 1e-9
    e1 = df[0] * low * np.exp(np.arange(ne) * (-math.log(low) / (ne - 1)))
    e2 = df[1] * low + np.arange(ne) * (df[1] * (1 - low) / (ne - 1))
    iw = [2 * math.pi / (n * x) for x in df]
    k1 = np.fft.fftfreq(n, 1.0 / n)
    k1[n // 2] = n // 2
    w1, w2 = T(iw[0] * k1)[:, None], T(iw[1] * np.arange(n // 2 + 1))[None, :]
    if case["data"] == "binned":
        bins, info = _bin2(d, 300)
        i, j = np.nonzero(bins)
        pts = T(info[0] + i * info[1]), T(info[2] + j * info[3])
        nb = T(bins[i, j].astype(np.float64))
    else:
        pts, nb = (T(d[0]), T(d[1])), 1.0
    tw = np.ones(n)
    tw[[0, -1]] = 0.5
    tw, te = T(tw), np.ones(ne)
    te[[0, -1]] = 0.5
    te, ar = T(te), T(np.arange(n, dtype=np.float64))
    F1, F2 = T(f1), T(f2)
    off = -d[0].size * (math.log(2 * math.pi * SIGMA2D[0] * SIGMA2D[1]) + 1.0)
    out = np.zeros(len(th))
    for q in range(len(th)):
        p = th[q].astype(np.float64)
        kc = _spline(np.log2(KNOTS2), math.log2(10.0) * p[:6])
        sc, oc = _spline(COLOUR_POS, p[6:9]), _spline(COLOUR_POS, p[9:12])

        def grid(a, b):
            lb = torch.log(b.clamp_min(1e-300))[None, :]
            r = torch.zeros((len(a), len(b)), dtype=torch.float64, device=dev)
            with np.errstate(divide="ignore"):
                la = np.log(a)
            for wk, ik, lr in zip(wt, inv1, lratio):
                s = a * ik
                good = (s >= KNOTS2[0]) & (s < KNOTS2[-1])
                c = np.where(good, np.exp2(_at(np.log2(KNOTS2), kc,
                                               np.log2(np.where(good, s, KNOTS2[0])))), 0.0)
                sv = np.clip(s, COLOUR_POS[0], COLOUR_POS[-1])
                sg, mu = _at(COLOUR_POS, sc, sv), _at(COLOUR_POS, oc, sv)
                m = np.where(good, la + mu - lr, 0.0)
                z = (lb - T(m)[:, None]) / T(sg)[:, None]
                r += T(wk * ik * c / sg)[:, None] * torch.exp(-0.5 * z * z)
            k = (PIX / 3600.0) ** 2 / math.sqrt(2 * math.pi)
            return torch.where(b > 0, r / b.clamp_min(1e-300), torch.zeros_like(r)) * k

        E1, E2 = T(e1), T(e2)
        x1 = -math.log(low) / (ne - 1) / (df[0] * (1 - low))
        x2 = 1.0 / (ne - 1)
        R = grid(f1, F2)
        R[0, :] = ((te * E1)[:, None] * grid(e1, F2)).sum(0) * x1
        R[:, 0] = (grid(f1, E2) * te).sum(1) * x2
        R[0, 0] = ((te * E1)[:, None] * grid(e1, E2) * te).sum() * x1 * x2
        R *= df[0] * df[1]
        m = tw[:, None] * R * tw
        mn = [float((m * F1[:, None]).sum()), float((m * F2).sum())]
        var = [float((m * F1[:, None] ** 2).sum()), float((m * F2 ** 2).sum())]
        f = torch.fft.rfft2(R)
        f = f - f[0, 0].real
        for k, ww in enumerate((w1, w2)):
            if math.sqrt(var[k]) > df[k] and abs(mn[k]) > df[k]:
                f = f + 1j * mn[k] * ww
        s = [p[12 + k] * SIGMA2D[k] for k in (0, 1)]
        noise = 0.5 * (s[0] * w1) ** 2 + 0.5 * (s[1] * w2) ** 2
        g = torch.fft.irfft2(torch.exp(f - noise), s=(n, n)).clamp_min(0.0)
        cut = []
        for k, mg in enumerate(((g * tw).sum(1), (tw[:, None] * g).sum(0))):
            sp = math.sqrt(var[k] + s[k] ** 2)
            sn = s[k] if 9 * s[k] ** 2 > var[k] else sp
            cut.append(_split(mg.cpu().numpy(), int(2.25 * sp / df[k]),
                              n - int(2.25 * sn / df[k]) - 1, 1.5e-5))
        if None in cut:
            out[q] = math.nan
            continue
        g = torch.roll(g, (-cut[0], -cut[1]), (0, 1))
        m = tw[:, None] * g * tw
        tot = float(m.sum())
        m0 = [-float((m * ar[:, None]).sum()) / tot * df[0], -float((m * ar).sum()) / tot * df[1]]
        g = g / (tot * df[0] * df[1])
        lg = torch.where(g > 0, torch.log2(g.clamp_min(5e-324)), torch.full_like(g, -30.0))
        at = [((c - a) / x) for c, a, x in zip(pts, m0, df)]
        lo, up = [t <= 0 for t in at], [t >= n - 1 for t in at]
        edge = lo[0] | lo[1] | up[0] | up[1]
        j = [t.clamp(0, n - 1).long() for t in at]
        t, u = at[0] - j[0], at[1] - j[1]
        jn = [(x + 1).clamp_max(n - 1) for x in j]
        iv = ((1 - t) * ((1 - u) * lg[j[0], j[1]] + u * lg[j[0], jn[1]])
              + t * ((1 - u) * lg[jn[0], j[1]] + u * lg[jn[0], jn[1]]))
        iv = torch.where(edge, lg[j[0], j[1]], iv)
        out[q] = math.log(2.0) * float((iv * nb).sum()) - off
    return out


def _exact_mlp(x, y, w):
    x, y = torch.from_numpy(x).double(), torch.from_numpy(y).double()
    w = [torch.from_numpy(v).double().requires_grad_() for v in w]
    for k in range(3):
        x = torch.nn.functional.gelu(x @ w[2 * k].t() + w[2 * k + 1])
    loss = ((x @ w[6] + w[7] - y) ** 2).mean()
    return dict(loss=float(loss.detach()), grad=[g.numpy().ravel()
                                                 for g in torch.autograd.grad(loss, w)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(*_mlp_inputs(case, seed))
    if kind == "like1d":
        terms = 0 if case["data"] == "binned" else case["walkers"] * case["side"] ** 2
        if case["walkers"] * case["nflux"] > 1 << 25 or terms > 1 << 28:
            return None  # half a minute and more in numpy
        return dict(loglike=_exact1(case, *_inputs1(case, seed)), status=None)
    if kind == "like2d":
        return dict(loglike=_exact2(case, *_inputs2(case, seed)), status=None)
    return None  # a chain's proposals are the library's own random numbers
