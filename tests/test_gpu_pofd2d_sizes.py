"""The two-band transforms at the grid sizes where their work divides
differently: eight short rows a workgroup (and transforms too short for the
swizzled order), four and two long ones, one column at the largest grid; odd
and even powers of two, with and without the edge integrals, and a second
dataset, against the CPU oracle."""
import threading

import numpy as np
import pytest

from oracle2d_side import build_oracle2d, make_inputs2d
from pofd_affine_amd import synth2d, workload2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nedge,edge,nwalk", [
    (64, 16, True, 3), (128, 16, False, 3), (256, 32, True, 5), (512, 64, False, 3),
    (1024, 64, True, 2), (4096, 32, True, 1)])
def test_sizes_against_oracle(n, nedge, edge, nwalk):
    print("[gpu2d-size-case] %d edge=%s" % (n, edge), flush=True)
    inp = make_inputs2d(npix_side=60, seed=5, nbins=40, nbeamhist=30)
    th0 = synth2d.true_theta()
    th = synth2d.walker_thetas(nwalk, seed=17)
    ctx = workload2d.build_context2d(inp, n, th0, nedge=nedge, edge_integ=edge)
    L = build_oracle2d(inp, n, th0, nedge=nedge, edge_integ=edge)
    ll, st = ctx.loglike2d_batch(th)
    ref, rst = L.loglike_batch(th, nwalk)
    assert np.array_equal(st, rst), (st, rst)
    ok = st == 0
    # the contract of every 2D path: 1e-6 of the oracle
    np.testing.assert_allclose(ll[ok], ref[ok], rtol=0, atol=1e-6)


@pytest.mark.parametrize("n", [64, 512, 4096])
def test_second_dataset_is_the_first(n):
    """The same pixels as the second dataset take the other column pass: the
    likelihood doubles (the stored spectrum is the first pass's)."""
    print("[gpu2d-size-case] two datasets %d" % n, flush=True)
    inp = make_inputs2d(npix_side=60, seed=5, nbins=40, nbeamhist=30)
    th0 = synth2d.true_theta()
    th = synth2d.walker_thetas(2, seed=18)
    one = workload2d.build_context2d(inp, n, th0, nedge=16)
    two = workload2d.build_context2d(inp, n, th0, nedge=16)
    two.add_field2d(0, inp["d1"], inp["d2"], synth2d.SIGMA1, synth2d.SIGMA2)
    two.prepare2d(th0)
    a, sa = one.loglike2d_batch(th)
    b, sb = two.loglike2d_batch(th)
    assert np.array_equal(sa, sb)
    ok = sa == 0
    assert np.array_equal(b[ok], a[ok] + a[ok])


@pytest.mark.parametrize("n", [64, 256, 1024])
@pytest.mark.parametrize("signed", [False, True])
def test_colour_width_of_zero_is_no_model(n, signed):
    """A colour width that is interpolated through zero makes weights of R
    infinite; where their Gaussians are zero R has no value, and the walker
    must fail as in the reference, whatever the rows in which that happens."""
    print("[gpu2d-size-case] zero width %d %s" % (n, signed), flush=True)
    inp = make_inputs2d(npix_side=60, seed=5, nbins=40, nbeamhist=30)
    if signed:
        inp["beam1"] = inp["beam1"] - 0.3 * np.roll(inp["beam1"], 5, 0)
        inp["beam2"] = inp["beam2"] - 0.2 * np.roll(inp["beam2"], 4, 1)
    th0 = synth2d.true_theta()
    th = np.tile(th0, (4, 1))
    for w in (1, 2, 3):  # the width at one of its three knots
        th[w, len(synth2d.KNOTS_MJY) + w - 1] = -0.5
    ctx = workload2d.build_context2d(inp, n, th0, edge_integ=False)
    L = build_oracle2d(inp, n, th0, edge_integ=False)
    ll, st = ctx.loglike2d_batch(th)
    ref, rst = L.loglike_batch(th, 4)
    assert np.array_equal(st, rst), (st, rst)
    assert np.any(rst[1:] != 0)
    ok = st == 0
    np.testing.assert_allclose(ll[ok], ref[ok], rtol=0, atol=1e-6)


def test_small_and_large_grids_in_two_threads():
    """A thread each for the smallest and the largest grid: what the kernels
    may use of LDS is one setting for the process, and a small grid's calls
    must not take it from a large one's."""
    print("[gpu2d-size-case] two threads", flush=True)
    inp = make_inputs2d(npix_side=60, seed=5, nbins=40, nbeamhist=30)
    th0 = synth2d.true_theta()
    th = synth2d.walker_thetas(1, seed=19)
    ctxs = {n: workload2d.build_context2d(inp, n, th0, nedge=16)
            for n in (4096, 64)}
    alone = {n: c.loglike2d_batch(th) for n, c in ctxs.items()}
    got = {n: [] for n in ctxs}

    def work(n, calls):
        got[n] += [ctxs[n].loglike2d_batch(th) for _ in range(calls)]
    threads = [threading.Thread(target=work, args=a)
               for a in ((4096, 20), (64, 100))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n, calls in ((4096, 20), (64, 100)):
        assert len(got[n]) == calls
        for ll, st in got[n]:
            assert np.array_equal(st, alone[n][1])
            assert np.array_equal(ll, alone[n][0], equal_nan=True)
