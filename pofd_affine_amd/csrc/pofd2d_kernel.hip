// 2D (two-band) P(D) log-likelihood kernels for gfx950: the work of
// calcLikeDoubleSingle::getLogLike (src/calcLikeDouble.cc:558-620) for a
// batch of walkers, one beam set at a time.  Grid layout n x n, row index i
// along band 1 (RFlux1), column index j along band 2 (RFlux2), as rvals in
// PDFactoryDouble.
//
//   prep2d        model set-up per walker: knot spline, colour sigma and
//                 offset interpolants (numberCountsDoubleLogNormal::setParams,
//                 src/numberCountsDoubleLogNormal.cc:1010-1052)
//   rpieces2d     the parts of R that depend on the row alone (getR array
//                 version, :1788-2007)
//   edge2d_*      edge integrals R[0,0], R[0,y], R[x,0] of initR
//                 (src/PDFactoryDouble.cc:376-551)
//   rowfft2d      R row by row, mean and variance along each axis (getRStats,
//                 :593-722), r2c transform, columns k2 <= K2 kept
//   rstats2d      the moments' parts combined, the shifts, R^(0)
//   colpass2d     complex transform down every kept column; spectrum
//                 exp(R^ - R^0) with the mean shifts (initPD, :1228-1340);
//                 per dataset the noise factor (getPD, :1396-1431) and the
//                 inverse transform
//   rowifft2d     c2r transform of every row, clamp, row marginal
//   colsum2d      column marginal (unwrapAndNormalizePD, :1001-1011)
//   split2d       findSplitPoint on both marginals (:784-975)
//   norm2d        rotation by the split points, integral and means
//                 (PDDouble::getIntegral / getMeans, src/PDDouble.cc:142-452)
//   like2d        binned or unbinned bilinear log likelihood
//                 (src/PDDouble.cc:976-1222)
//   combine2d     (curr - like_offset)/like_norm over datasets
//
// Spectral pruning: after the noise factor only components with
// sigma1^2 w1^2/2 <= cut and sigma2^2 w2^2/2 <= cut survive, so the forward
// column transforms run only for k2 <= K2 and the inverse only takes k1 in
// [0, K1] U [n-K1, n) and k2 <= K2 (K1, K2 from the widest dataset).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "exp2.h"
#include "internal2d.h"

namespace pofd2 {

namespace {

constexpr int kT = 256;  // threads per workgroup

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double mul_rn(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ double add_rn(double a, double b) { return __dadd_rn(a, b); }
__device__ __forceinline__ double sub_rn(double a, double b) { return __dsub_rn(a, b); }

__device__ __forceinline__ double log2_or_small(double v) {
  return (v > 0.0) ? log2(v) : -30.0;  // pofd_mcmc::smalllogval
}

__device__ double block_sum(double v, double* red) {
  const int tid = threadIdx.x;
  const int nw = blockDim.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  double s = red[0];
  for (int i = 1; i < nw; ++i) s += red[i];
  __syncthreads();
  return s;
}

__device__ double block_max(double v, double* red) {
  const int tid = threadIdx.x;
  const int nw = blockDim.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  double s = red[0];
  for (int i = 1; i < nw; ++i) s = fmax(s, red[i]);
  __syncthreads();
  return s;
}

__device__ int block_max_int(int v, int* ired) {
  const int tid = threadIdx.x;
  const int nw = blockDim.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
  __syncthreads();
  if ((tid & 63) == 0) ired[tid >> 6] = v;
  __syncthreads();
  int s = ired[0];
  for (int i = 1; i < nw; ++i) s = max(s, ired[i]);
  __syncthreads();
  return s;
}

// (value, index) minimum, the lowest index among equal values; idx < 0 is
// an empty slot
__device__ void block_argmin(double& v, int& idx, double* red, int* ired) {
  const int tid = threadIdx.x;
  const int nw = blockDim.x >> 6;
  auto better = [](double a, int ia, double b, int ib) {
    if (ib < 0) return true;
    if (ia < 0) return false;
    return (a < b) || (a == b && ia < ib);
  };
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const int oi = __shfl_xor(idx, o);
    if (!better(v, idx, ov, oi)) {
      v = ov;
      idx = oi;
    }
  }
  __syncthreads();
  if ((tid & 63) == 0) {
    red[tid >> 6] = v;
    ired[tid >> 6] = idx;
  }
  __syncthreads();
  v = red[0];
  idx = ired[0];
  for (int i = 1; i < nw; ++i)
    if (!better(v, idx, red[i], ired[i])) {
      v = red[i];
      idx = ired[i];
    }
  __syncthreads();
}

// ---- per-walker model block (doubles): [0] status, [1] sigmult1,
// [2] sigmult2, [3] K1, [4] K2, then the knot spline (4 per interval, log2
// space), sigma and offset interpolants (4 per interval), raw sigma and
// offset values
constexpr int kMH = 8;
constexpr int kOffK = kMH, kOffS = kMH + 4 * kMaxK, kOffO = kMH + 8 * kMaxK;
constexpr int kOffSV = kMH + 12 * kMaxK, kOffOV = kMH + 13 * kMaxK;
__device__ __forceinline__ double* model_ptr(const Work2& wk, int w) {
  return wk.model + static_cast<size_t>(w) * kModelStride;
}

// largest index k with sigfac*(iflux*k)^2 >= -cut (the noise factor of the
// component is above exp(-cut)); n/2 when sigma is not positive
__device__ int kmax_axis(double sigma, double iflux, double cut, int kcap) {
  if (!(sigma > 0)) return kcap;
  const double sigfac = -0.5 * sigma * sigma;
  const double est = sqrt(2.0 * cut) / (sigma * iflux);
  long k = (est > static_cast<double>(kcap)) ? kcap : static_cast<long>(est);
  auto keep = [&](long kk) {
    const double w = mul_rn(iflux, static_cast<double>(kk));
    return mul_rn(mul_rn(sigfac, w), w) >= -cut;
  };
  while (k < kcap && keep(k + 1)) ++k;
  while (k > 0 && !keep(k)) --k;
  return static_cast<int>(k);
}

// GSL natural cubic spline coefficients (cspline_init, coeff_calc) of
// (x, y) into cf[4*i..]: y_i, b_i, c_i, d_i; no contraction, thread 0 only
__device__ void cspline_coefs(int n, const double* x, const double* y, double* cf,
                              double* scratch /* 6*kMaxK */) {
  double* c = scratch;
  double* diag = scratch + kMaxK;
  double* off = scratch + 2 * kMaxK;
  double* g = scratch + 3 * kMaxK;
  double* alpha = scratch + 4 * kMaxK;
  double* gamma = scratch + 5 * kMaxK;
  const int sys = n - 2;
  for (int i = 0; i < n; ++i) c[i] = 0.0;
  for (int i = 0; i < sys; ++i) {
    const double h_i = sub_rn(x[i + 1], x[i]);
    const double h_ip1 = sub_rn(x[i + 2], x[i + 1]);
    const double yd_i = sub_rn(y[i + 1], y[i]);
    const double yd_ip1 = sub_rn(y[i + 2], y[i + 1]);
    const double g_i = (h_i != 0.0) ? 1.0 / h_i : 0.0;
    const double g_ip1 = (h_ip1 != 0.0) ? 1.0 / h_ip1 : 0.0;
    off[i] = h_ip1;
    diag[i] = mul_rn(2.0, add_rn(h_ip1, h_i));
    g[i] = mul_rn(3.0, sub_rn(mul_rn(yd_ip1, g_ip1), mul_rn(yd_i, g_i)));
  }
  if (sys == 1) {
    c[1] = g[0] / diag[0];
  } else if (sys > 1) {
    double* z = diag;
    alpha[0] = diag[0];
    gamma[0] = off[0] / alpha[0];
    for (int i = 1; i < sys - 1; ++i) {
      alpha[i] = sub_rn(diag[i], mul_rn(off[i - 1], gamma[i - 1]));
      gamma[i] = off[i] / alpha[i];
    }
    alpha[sys - 1] = sub_rn(diag[sys - 1], mul_rn(off[sys - 2], gamma[sys - 2]));
    z[0] = g[0];
    for (int i = 1; i < sys; ++i) z[i] = sub_rn(g[i], mul_rn(gamma[i - 1], z[i - 1]));
    for (int i = 0; i < sys; ++i) z[i] = z[i] / alpha[i];
    c[sys] = z[sys - 1];
    for (int i = sys - 2; i >= 0; --i) c[i + 1] = sub_rn(z[i], mul_rn(gamma[i], c[i + 2]));
  }
  for (int i = 0; i < n - 1; ++i) {
    const double dx = sub_rn(x[i + 1], x[i]);
    const double dy = sub_rn(y[i + 1], y[i]);
    cf[4 * i] = y[i];
    cf[4 * i + 1] = sub_rn(dy / dx, mul_rn(dx, add_rn(c[i + 1], mul_rn(2.0, c[i]))) / 3.0);
    cf[4 * i + 2] = c[i];
    cf[4 * i + 3] = sub_rn(c[i + 1], c[i]) / mul_rn(3.0, dx);
  }
}

// gsl_interp_bsearch over x[0..n-1]
__device__ __forceinline__ int bsearch_k(const double* x, int n, double v) {
  int lo = 0, hi = n - 1;
  while (hi > lo + 1) {
    const int m = (lo + hi) >> 1;
    if (x[m] > v)
      hi = m;
    else
      lo = m;
  }
  return lo;
}

__device__ __forceinline__ double spline_eval(const double* x, const double* cf, int n,
                                              double v) {
  const int k = bsearch_k(x, n, v);
  const double dx = sub_rn(v, x[k]);
  const double* c = cf + 4 * k;
  return add_rn(c[0], mul_rn(dx, add_rn(c[1], mul_rn(dx, add_rn(c[2], mul_rn(dx, c[3]))))));
}

// getSigmaInner / getOffsetInner (src/numberCountsDoubleLogNormal.cc:1172-1193)
__device__ double colour_eval(const double* x, const double* vals, const double* cf,
                              int n, double f1, double floorv, bool floored) {
  if (n == 1) return vals[0];
  if (f1 <= x[0]) return vals[0];
  if (f1 >= x[n - 1]) return vals[n - 1];
  double val;
  if (n == 2) {  // gsl_interp_linear
    const double dx = sub_rn(x[1], x[0]);
    val = (dx > 0.0) ? add_rn(vals[0], mul_rn(sub_rn(f1, x[0]) / dx, sub_rn(vals[1], vals[0])))
                     : 0.0;
  } else {
    val = spline_eval(x, cf, n, f1);
  }
  if (floored && val < floorv) val = floorv;
  return val;
}

}  // namespace

// ===========================================================================
// prep2d: model set-up, one thread per walker
// ===========================================================================
__global__ __launch_bounds__(64) void prep2d_kernel(const Set2Dev s, const Work2 wk,
                                                    const float* __restrict__ theta,
                                                    const uint32_t stride,
                                                    const int32_t* __restrict__ prev_status,
                                                    const int accumulate) {
  __shared__ double scratch[6 * kMaxK];
  __shared__ double vals[kMaxK];
  if (threadIdx.x != 0) return;
  const int w = blockIdx.x;
  double* m = model_ptr(wk, w);
  const float* th = theta + static_cast<size_t>(w) * stride;
  const int nk = s.nk, ns = s.ns, no = s.no;
  int status = accumulate ? prev_status[w] : POFD_OK;
  const double sm1 = th[nk + ns + no], sm2 = th[nk + ns + no + 1];
  // setParams and the validity checks (src/numberCountsDoubleLogNormal.cc:
  // 1010-1119): log2 knot values, sigma and offset values as doubles
  bool valid = true;
  for (int i = 0; i < nk; ++i) {
    vals[i] = mul_rn(s.logfac, static_cast<double>(th[i]));
    if (isnan(vals[i])) valid = false;
  }
  if (valid) cspline_coefs(nk, s.logknots, vals, m + kOffK, scratch);
  for (int i = 0; i < ns; ++i) {
    const double v = th[nk + i];
    if (isnan(v) || isinf(v)) valid = false;
    vals[i] = v;
    m[kOffSV + i] = v;
  }
  if (valid && ns > 2) cspline_coefs(ns, s.sigmaknots, vals, m + kOffS, scratch);
  for (int i = 0; i < no; ++i) {
    const double v = th[nk + ns + i];
    if (isnan(v)) valid = false;
    vals[i] = v;
    m[kOffOV + i] = v;
  }
  if (valid && no > 2) cspline_coefs(no, s.offsetknots, vals, m + kOffO, scratch);
  if (status == POFD_OK) {
    if (isnan(sm1) || isnan(sm2))
      status = POFD_E_ARG;
    else if (mul_rn(s.maxsig1, sm1) < 0.0 || mul_rn(s.maxsig2, sm2) < 0.0)
      status = POFD_E_BADLIKE;  // calcLikeDoubleSingle::bad_like, :571-574
    else if (!valid || !(s.min_sigma >= 0.0))
      status = POFD_E_INVALID_MODEL;
  }
  // spectral bounds of the widest dataset
  int K1 = 0, K2 = 0;
  for (int f = 0; f < s.nfields; ++f) {
    K1 = max(K1, kmax_axis(sm1 * s.fields[f].sigma_base1, s.iflux1, s.spectral_cut, s.n / 2));
    K2 = max(K2, kmax_axis(sm2 * s.fields[f].sigma_base2, s.iflux2, s.spectral_cut, s.n / 2));
  }
  m[0] = status;
  m[1] = sm1;
  m[2] = sm2;
  m[3] = K1;
  m[4] = K2;
  m[5] = valid ? 1.0 : 0.0;
}

// ===========================================================================
// bonus2d: getNS, getFluxPerArea and getFluxSqPerArea of both bands
// (numberCountsDoubleLogNormal::splineInt, src/numberCountsDoubleLogNormal.cc:
// 1549-1673, integrand evalPowfNDoubleLogNormal :2424-2519):
// int S1^(a+b) exp(b mu(S1) + b^2/2 sigma(S1)^2) n1(S1) dS1 as Gauss-Legendre
// sums in log2 S1 between consecutive knots of the band-1, sigma and offset
// models (analytic there).  One 64-lane workgroup per walker.
// ===========================================================================
__global__ __launch_bounds__(64) void bonus2d_kernel(const Set2Dev s, const Work2 wk) {
  __shared__ double red[1];
  const int w = blockIdx.x;
  const double* m = model_ptr(wk, w);
  double* bo = wk.bonus + static_cast<size_t>(w) * 8;
  if (m[5] == 0.0) {  // invalid model: splineInt returns NaN
    if (threadIdx.x < 5) bo[threadIdx.x] = __longlong_as_double(0x7ff8000000000000ULL);
    return;
  }
  const int nk = s.nk, ns = s.ns, no = s.no;
  const double* kcf = m + kOffK;
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  const int npts = (s.nbp - 1) * 32;
  for (int t = threadIdx.x; t < npts; t += 64) {
    const int k = t >> 5, g = t & 31;
    const double v0 = s.bpts[k], v1 = s.bpts[k + 1];
    if (!(v1 > v0)) continue;
    const double h = 0.5 * (v1 - v0), c = 0.5 * (v1 + v0);
    const double v = c + h * s.glx[g];
    const double s1 = exp2(v);
    const double lc = spline_eval(s.logknots, kcf, nk, v);
    double sg = colour_eval(s.sigmaknots, m + kOffSV, m + kOffS, ns, s1, s.min_sigma, true);
    if (sg < s.min_sigma) sg = s.min_sigma;
    const double mu = colour_eval(s.offsetknots, m + kOffOV, m + kOffO, no, s1, 0.0, false);
    const double base = s.glw[g] * h * exp2(lc + v);  // S1 n1(S1) per unit log2 S1
    const double e1 = exp(mu + 0.5 * sg * sg);         // beta = 1
    const double e2 = exp(2.0 * mu + 2.0 * sg * sg);   // beta = 2
    acc[0] += base;
    acc[1] += base * s1;
    acc[2] += base * s1 * e1;
    acc[3] += base * s1 * s1;
    acc[4] += base * s1 * s1 * e2;
  }
  const double ln2 = 0.69314718055994530942;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const double tot = block_sum(acc[q], red);
    if (threadIdx.x == 0) bo[q] = ln2 * tot;
  }
}

// ===========================================================================
// R on (f1[i], f2[j])
// ===========================================================================
// The pieces of R that depend on the row flux f1 but not on f2, per row
// of the grid and beam element (RWork, :1868-1950): weight (0 where the
// element adds nothing), log-flux centre and Gaussian width factor, into
// wk.rpieces for the kernels that make R.  One thread per (row, element), so
// that their logs, exp2s and colour splines run in parallel.
__global__ __launch_bounds__(kT) void rpieces2d_kernel(const Set2Dev s, const Work2 wk,
                                                       const RGrid g) {
  __shared__ double lk[kMaxK], lkcf[4 * kMaxK];
  __shared__ double sk[kMaxK], scf[4 * kMaxK], svl[kMaxK];
  __shared__ double ok[kMaxK], ocf[4 * kMaxK], ovl[kMaxK];
  const int w = blockIdx.y;
  const double* m = model_ptr(wk, w);
  if (m[0] != POFD_OK) return;  // uniform
  const int nk = s.nk, ns = s.ns, no = s.no;
  for (int t = threadIdx.x; t < kMaxK; t += kT) {
    lk[t] = s.logknots[t];
    sk[t] = s.sigmaknots[t];
    ok[t] = s.offsetknots[t];
    svl[t] = m[kOffSV + t];
    ovl[t] = m[kOffOV + t];
  }
  for (int t = threadIdx.x; t < 4 * kMaxK; t += kT) {
    lkcf[t] = m[kOffK + t];
    scf[t] = m[kOffS + t];
    ocf[t] = m[kOffO + t];
  }
  __syncthreads();
  const int maxc = wk.rpieces_w / 3;
  const int t = blockIdx.x * kT + threadIdx.x;
  const int i = t / maxc, e = t - i * maxc;
  if (i >= g.n1) return;
  double f1val = g.f1[i];
  if ((f1val == 0) || (f1val < 0 && !s.hasneg1)) return;  // a row of zeros
  int sgn1 = 0;
  if (!(f1val > 0)) {
    sgn1 = 2;
    f1val = fabs(f1val);
  }
  const int np = s.comp[sgn1].n, nn = s.comp[sgn1 + 1].n;
  if (e >= np + nn) return;
  const double minknot = s.knots[0], maxknot = s.knots[nk - 1];
  const double ilog2toe = 1.4426950408889634074;  // 1/ln 2
  const double logf1 = log(f1val);
  const int k = (e < np) ? 0 : 1;
  const BeamComp& bc = s.comp[sgn1 + k];
  const int jj = (k == 0) ? e : e - np;
  double* c = wk.rpieces + static_cast<size_t>(w) * wk.rpieces_stride +
              static_cast<size_t>(i) * wk.rpieces_w + 3 * e;
  double c0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (f1val < bc.maxf1) {
#pragma clang fp contract(off)
    const double ieta1 = bc.ieta1[jj];
    const double f1prod = f1val * ieta1;
    if (f1prod >= minknot && f1prod < maxknot) {
      const double cts = exp2(spline_eval(lk, lkcf, nk, log2(f1prod)));
      if (cts > 0) {
        const double isigma = 1.0 / colour_eval(sk, svl, scf, ns, f1prod, s.min_sigma, true);
        c0 = (bc.w ? bc.w[jj] * ieta1 * isigma * cts * s.prefac
                   : cts * ieta1 * isigma * s.prefac);
        c1 = logf1 + colour_eval(ok, ovl, ocf, no, f1prod, 0.0, false) - bc.logratio[jj];
        c2 = -0.5 * isigma * isigma * ilog2toe;
        // an infinite weight (a colour width of zero) has no value where its
        // Gaussian is zero: NaN at every point, as a term that the fill may
        // not skip
        if (!isfinite(c0)) c1 = __longlong_as_double(0x7ff8000000000000ULL);
      }
    }
  }
  c[0] = c0;
  c[1] = c1;
  c[2] = 32.0 * c2;  // the exponent in the units of exp2_32
}

// 2^(t/32) by Tang's table-driven method (ACM TOMS 15:144, 1989): t = 32 n +
// j + u, 2^n tab[j] 2^(u/32).  Zero from t = -34560 (2^-1080) down; NaN stays.
// About one ulp, in 12 instructions of the 20 of exp2.
__device__ __forceinline__ double exp2_32(double t, const double* tab) {
  t = (t < -35000.0) ? -35000.0 : t;
  const double n = rint(t);
  const int ni = __double2int_rn(t);
  return ldexp(tab[ni & 31] * pofd::exp2_near(t - n), ni >> 5);
}
__device__ __forceinline__ void load_exp2(double* tab) {
  if (threadIdx.x < 32) tab[threadIdx.x] = exp2(static_cast<double>(threadIdx.x) * 0.03125);
}

// R at f1val and the kEdgePts points f2[j0 + q step], j < n2, of a grid from
// the row's pieces, the beam elements' Gaussian colour terms summed in element
// order; the pieces are read once for all points.
constexpr int kEdgePts = 4;
__device__ __forceinline__ void r_values(const Set2Dev& s, const RGrid& g, const double f1val,
                                         const double* __restrict__ prow, const int j0,
                                         const int step, const double* tab, double* r) {
#pragma unroll
  for (int q = 0; q < kEdgePts; ++q) r[q] = 0.0;
  if ((f1val == 0) || (f1val < 0 && !s.hasneg1)) return;
  const int sgn1 = (f1val > 0) ? 0 : 2;
  double lf[kEdgePts];
#pragma unroll 1
  for (int sg = 0; sg < 2; ++sg) {
    const int cn = s.comp[sgn1 + sg].n;
    if (cn == 0) continue;
    // a point of the other sign, or of no flux: an exponent of -infinity
#pragma unroll
    for (int q = 0; q < kEdgePts; ++q) {
      const int j = j0 + q * step;
      lf[q] = (j < g.n2 && g.f2inv[j] != 0 && g.f2sgn[j] == sg) ? g.f2log[j] : 1e160;
    }
    const double* base = prow + (sg ? 3 * s.comp[sgn1].n : 0);
    for (int k = 0; k < cn; ++k) {
#pragma clang fp contract(off)
      const double c0 = base[3 * k], c1 = base[3 * k + 1], c2 = base[3 * k + 2];
      if (c0 == 0) continue;
#pragma unroll
      for (int q = 0; q < kEdgePts; ++q) {
        const double tfac = lf[q] - c1;
        r[q] += c0 * exp2_32(tfac * tfac * c2, tab);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kEdgePts; ++q) {
    const int j = j0 + q * step;
    r[q] = (j < g.n2) ? (r[q] * g.f2inv[j]) * g.scale : 0.0;
  }
}

// ===========================================================================
// edge integrals (initR with setEdge, src/PDFactoryDouble.cc:386-544)
// ===========================================================================
// Per row of a grid the trapezoid over its columns (the linear edge in band
// 2): a wavefront per row, R summed as it is made.  The edge integrals take
// 217 us for 32 walkers at 2048 and 256 edge points, bound by the
// exponentials; three grids to memory and one thread per sum took 306 + 237
// (and 570 one point at a time, waiting for each element's pieces).
__global__ __launch_bounds__(kT) void edge2d_rows_kernel(const Set2Dev s, const Work2 wk,
                                                         const RGrid g,
                                                         double* __restrict__ out) {
  __shared__ double tab[32];
  const int w = blockIdx.y;
  if (model_ptr(wk, w)[0] != POFD_OK) return;  // uniform
  load_exp2(tab);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane(
      static_cast<int>(blockIdx.x * (kT / 64) + (threadIdx.x >> 6)));
  if (i >= g.n1) return;
  const double f1val = g.f1[i];
  const double* prow = wk.rpieces + static_cast<size_t>(w) * wk.rpieces_stride +
                       static_cast<size_t>(i) * wk.rpieces_w;
  double sc = 0.0;
  for (int j0 = lane; j0 - lane < g.n2; j0 += 64 * kEdgePts) {
    double r[kEdgePts];
    r_values(s, g, f1val, prow, j0, 64, tab, r);
#pragma unroll
    for (int q = 0; q < kEdgePts; ++q) {
      const int j = j0 + 64 * q;
      sc += ((j == 0 || j == g.n2 - 1) ? 0.5 : 1.0) * r[q];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sc += __shfl_xor(sc, o);
  if (lane == 0) out[static_cast<size_t>(w) * wk.edge_stride + i] = sc;
}

// The log-x trapezoid over the nedge rows of R(edge1, RFlux2[j]), kEdgePts
// columns a thread: the rows of part blockIdx.y, for edge2d_sum_kernel
__global__ __launch_bounds__(kT) void edge2d_cols_kernel(const Set2Dev s, const Work2 wk,
                                                         const RGrid g) {
  __shared__ double tab[32];
  const int w = blockIdx.z;
  if (model_ptr(wk, w)[0] != POFD_OK) return;  // uniform
  load_exp2(tab);
  __syncthreads();
  const int j0 = blockIdx.x * kT * kEdgePts + threadIdx.x;
  const int ne = g.n1, part = blockIdx.y, parts = gridDim.y;
  const int i0 = part * ne / parts, i1 = (part + 1) * ne / parts;
  double acc[kEdgePts] = {0.0, 0.0, 0.0, 0.0};
  for (int i = i0; i < i1; ++i) {
    const double* prow = wk.rpieces + static_cast<size_t>(w) * wk.rpieces_stride +
                         static_cast<size_t>(i) * wk.rpieces_w;
    const double wi = ((i == 0 || i == ne - 1) ? 0.5 : 1.0) * s.edge1[i];
    double r[kEdgePts];
    r_values(s, g, g.f1[i], prow, j0, kT, tab, r);
#pragma unroll
    for (int q = 0; q < kEdgePts; ++q) acc[q] += wi * r[q];
  }
#pragma unroll
  for (int q = 0; q < kEdgePts; ++q) {
    const int j = j0 + q * kT;
    if (j < g.n2)
      wk.ex[static_cast<size_t>(w) * wk.ex_stride + static_cast<size_t>(part) * g.n2 + j] = acc[q];
  }
}

// Rx[j] from its parts, and R[0,0] (times dflux1 dflux2) from the row sums of
// the nedge x nedge grid to rx[0]; rowfft2d_kernel puts rx and ry in place of
// row 0 and column 0
__global__ __launch_bounds__(kT) void edge2d_sum_kernel(const Set2Dev s, const Work2 wk,
                                                        const int parts) {
  __shared__ double red[kT / 64];
  const int w = blockIdx.y;
  if (model_ptr(wk, w)[0] != POFD_OK) return;  // uniform
  double* rx = wk.rx + static_cast<size_t>(w) * wk.edge_stride;
  const int j = blockIdx.x * kT + threadIdx.x;
  if (j > 0 && j < s.n) {
    const double* ex = wk.ex + static_cast<size_t>(w) * wk.ex_stride + j;
    double acc = 0.0;
    for (int p = 0; p < parts; ++p) acc += ex[static_cast<size_t>(p) * s.n];
    rx[j] = acc * s.iRxnorm;
  }
  if (blockIdx.x == 0) {
    const double* r00rows = wk.r00rows + static_cast<size_t>(w) * wk.edge_stride;
    const int ne = s.nedge;
    double sc = 0.0;
    for (int i = threadIdx.x; i < ne; i += kT)
      sc += ((i == 0 || i == ne - 1) ? 0.5 : 1.0) * s.edge1[i] * r00rows[i];
    sc = block_sum(sc, red);
    if (threadIdx.x == 0) rx[0] = (sc * s.iR00norm) * (s.dflux1 * s.dflux2);
  }
}

// ===========================================================================
// LDS transforms
// ===========================================================================
constexpr int kTR = 1024;  // threads per workgroup of the transforms
// Rows and columns a workgroup transforms together: as many as fill 128 KB
// with both buffers, no more than eight.  Four rows of 2048 give the 64
// contiguous bytes in which the transposed spectra are written and read.
inline int rows_together(const int n) { return std::min(8, 8192 / n); }
constexpr int kMaxPairs = 4;  // pairs of a row's points per thread: n rg / 2 kTR
inline int cols_together(const int n) { return std::min(8, 4096 / n); }

// Element i of a transform of length L is at slot(i): the exclusive-or of
// bits 4 and 5 into bits 0 to 3 keeps a stage's writes (strides of 4 to 32
// elements between 16 lanes) and reads on distinct banks; short transforms
// (swz 0) are in order.  turn_slot does the same for the twiddles, which are
// read at strides of L / 4 Ns.
__device__ __forceinline__ int swizzle_of(const int L) { return L >= 256 ? 15 : 0; }
__device__ __forceinline__ int slot(const int i, const int swz) {
  const int t = (i >> 4) & 3;
  return i ^ ((t ^ (t << 2)) & swz);
}
__device__ __forceinline__ int turn_slot(const int t) { return t ^ ((t >> 4) & 15) ^ (t >> 8); }

// Forward transform of length L (a power of two from 32 on) from a, by T
// threads of which this is t; every thread of the workgroup calls it, with
// the same L.  Radix 4 after a radix-2 stage when log2 L is odd.
// tw[turn_slot(t)] = e^{-2 pi i t/L}, t < L/4.  Returns the buffer that holds
// the result.  (The inverse: the same with real and imaginary parts
// exchanged before and after.)
__device__ __forceinline__ double2* fft_lds(double2* a, double2* b, const int L,
                                            const double2* tw, const int t, const int T) {
  const int swz = swizzle_of(L);
  double2* src = a;
  double2* dst = b;
  int Ns = 1;
  if (__builtin_ctz(static_cast<unsigned>(L)) & 1) {
    const int h = L >> 1;
    for (int j = t; j < h; j += T) {
      const double2 v0 = src[slot(j, swz)], v1 = src[slot(j + h, swz)];
      dst[slot(2 * j, swz)] = cadd(v0, v1);
      dst[slot(2 * j + 1, swz)] = csub(v0, v1);
    }
    __syncthreads();
    double2* u = src;
    src = dst;
    dst = u;
    Ns = 2;
  }
  const int q = L >> 2;
  auto quarter = [](const double2 v, const bool on) {
    return on ? make_double2(v.y, -v.x) : v;
  };
  for (; Ns < L; Ns *= 4) {
    const int ts = L / (4 * Ns);
    for (int j = t; j < q; j += T) {
      const int jm = j & (Ns - 1);
      const double2* sj = src + slot(j, swz);  // q is a multiple of 64, or swz 0
      double2 v0 = sj[0], v1 = sj[q], v2 = sj[2 * q], v3 = sj[3 * q];
      if (Ns > 1) {
        const int t1 = jm * ts, t2 = 2 * t1, t3 = 3 * t1;  // t1 < q
        v1 = cmul(v1, tw[turn_slot(t1)]);
        v2 = quarter(cmul(v2, tw[turn_slot(t2 & (q - 1))]), t2 & q);
        v3 = quarter(cmul(v3, tw[turn_slot(t3 & (q - 1))]), t3 & q);
        if (t3 & (2 * q)) v3 = make_double2(-v3.x, -v3.y);
      }
      const double2 a0 = cadd(v0, v2), a1 = csub(v0, v2);
      const double2 a2 = cadd(v1, v3), a3 = csub(v1, v3);
      const int d = (j - jm) * 4 + jm;
      dst[slot(d, swz)] = cadd(a0, a2);
      dst[slot(d + Ns, swz)] = make_double2(a1.x + a3.y, a1.y - a3.x);
      dst[slot(d + 2 * Ns, swz)] = csub(a0, a2);
      dst[slot(d + 3 * Ns, swz)] = make_double2(a1.x - a3.y, a1.y + a3.x);
    }
    __syncthreads();
    double2* u = src;
    src = dst;
    dst = u;
  }
  return src;
}
__device__ __forceinline__ void load_turns(double2* tw, const double2* __restrict__ table,
                                           const int L) {
  for (int t = threadIdx.x; t < L / 4; t += kTR) tw[turn_slot(t)] = table[t];
}

// ===========================================================================
// rowfft2d: R row by row, its trapezoid moments along each axis (partials per
// workgroup) and the r2c transform of every row; outputs k2 = 0..K2 to
// YT[k2][i].  R goes to memory nowhere.  rg rows together, T = kTR / rg
// threads each (whole wavefronts, so that a row's pieces are uniform reads,
// made once for a thread's eight points).  Bound by the exponentials of R:
// 1590 us for 32 walkers at 2048 (1648 with the library's exp2), where R to memory, its moments, the row
// transforms from it and their transposition took 1274 + 265 + 588 + 195
// (2489 with the pieces read again for each point).
// ===========================================================================
__global__ __launch_bounds__(kTR) void rowfft2d_kernel(const Set2Dev s, const Work2 wk,
                                                       const RGrid g, const int rg) {
  extern __shared__ double2 lds[];
  __shared__ double red[kTR / 64], ex2[32];
  const int w = blockIdx.y;
  const double* m = model_ptr(wk, w);
  if (m[0] != POFD_OK) return;
  const int K2 = static_cast<int>(m[4]);
  const int n = s.n, h = n / 2, tid = threadIdx.x;
  const int T = kTR / rg, grp = tid / T, t = tid & (T - 1);
  const int swz = swizzle_of(h);
  double2* tw = lds;
  double2* rows = lds + h / 4;
  const int rs = n + 2;  // the rows' elements k on distinct banks
  load_turns(tw, s.tw_half, h);
  load_exp2(ex2);
  __syncthreads();
  const double* pieces = wk.rpieces + static_cast<size_t>(w) * wk.rpieces_stride;
  const double* rx = wk.rx + static_cast<size_t>(w) * wk.edge_stride;
  const double* ry = wk.ry + static_cast<size_t>(w) * wk.edge_stride;
  const double fluxfac = s.dflux1 * s.dflux2;
  double2* YT = wk.YT + static_cast<size_t>(w) * wk.YT_stride;
  double m1 = 0, m2 = 0, v1 = 0, v2 = 0;
  for (int i0 = blockIdx.x * rg; i0 < n; i0 += gridDim.x * rg) {
    const int i = __builtin_amdgcn_readfirstlane(i0 + grp);
    double2* a = rows + grp * rs;
    const double f1val = g.f1[i];
    const bool none = (f1val == 0) || (f1val < 0 && !s.hasneg1);  // a row of zeros
    const int sgn1 = (f1val > 0) ? 0 : 2;
    const double* prow = pieces + static_cast<size_t>(i) * wk.rpieces_w;
    const double edge0 = (s.edge_integ && i > 0) ? (ry[i] * s.iRynorm) * fluxfac : 0.0;
    const double wi = (i == 0 || i == n - 1) ? 0.5 : 1.0;
    const double cf1 = s.rflux1[i];
    // this thread's points: pairs t + q T of the row; the elements' pieces are
    // read once for all of them
    double x[2 * kMaxPairs], lf[2 * kMaxPairs];
#pragma unroll
    for (int q = 0; q < 2 * kMaxPairs; ++q) x[q] = 0.0;
    if (!none) {
#pragma unroll 1
      for (int sg = 0; sg < 2; ++sg) {
        const int cn = s.comp[sgn1 + sg].n;
        if (cn == 0) continue;
        // a point of the other sign, or of no flux: an exponent of -infinity
#pragma unroll
        for (int q = 0; q < 2 * kMaxPairs; ++q) {
          const int e = t + (q >> 1) * T, j = 2 * e + (q & 1);
          lf[q] = (e < h && g.f2inv[j] != 0 && g.f2sgn[j] == sg) ? g.f2log[j] : 1e160;
        }
        const double* base = prow + (sg ? 3 * s.comp[sgn1].n : 0);
        for (int k = 0; k < cn; ++k) {
          const double c0 = base[3 * k], c1 = base[3 * k + 1], c2 = base[3 * k + 2];
          if (c0 == 0) continue;
#pragma unroll
          for (int q = 0; q < kMaxPairs; ++q) {
#pragma clang fp contract(off)
            if (q * T >= h) break;  // uniform
            const double ta = lf[2 * q] - c1, tb = lf[2 * q + 1] - c1;
            const double ea = ta * ta * c2, eb = tb * tb * c2;
            // below the smallest number for the whole wavefront: adds nothing
            if (__any(!(ea <= -34560.0 && eb <= -34560.0))) {
              x[2 * q] += c0 * exp2_32(ea, ex2);
              x[2 * q + 1] += c0 * exp2_32(eb, ex2);
            }
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kMaxPairs; ++q) {
      const int e = t + q * T;
      if (e >= h) break;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int j = 2 * e + u;
        double r = (x[2 * q + u] * g.f2inv[j]) * g.scale;
        if (s.edge_integ && i == 0) r = (j == 0) ? rx[0] : rx[j] * fluxfac;
        if (s.edge_integ && i > 0 && j == 0) r = edge0;
        x[2 * q + u] = r;
        const double wj = (j == 0 || j == n - 1) ? 0.5 : 1.0;
        const double cR = wi * r;
        const double p1 = wj * cf1 * cR;
        m1 += p1;
        v1 += cf1 * p1;
        const double cf2 = s.rflux2[j];
        const double p2 = wj * cf2 * cR;
        m2 += p2;
        v2 += cf2 * p2;
      }
      a[slot(e, swz)] = make_double2(x[2 * q], x[2 * q + 1]);
    }
    __syncthreads();
    const double2* z = fft_lds(a, a + h, h, tw, t, T) - grp * rs;  // row 0's
    for (int o = tid; o < rg * (K2 + 1); o += kTR) {
      const int k = o / rg, row = o - k * rg;
      const double2* zr = z + row * rs;
      const double2 zk = zr[slot((k == h) ? 0 : k, swz)];
      const double2 zh = zr[slot((k == 0) ? 0 : h - k, swz)];
      const double2 zm = make_double2(zh.x, -zh.y);
      const double2 A = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y + zm.y));
      const double2 B = make_double2(0.5 * (zk.y - zm.y), -0.5 * (zk.x - zm.x));
      const double2 wv = (k == h) ? make_double2(-1.0, 0.0) : s.tw_n[k];
      YT[static_cast<size_t>(k) * n + i0 + row] = cadd(A, cmul(B, wv));
    }
    __syncthreads();
  }
  double* part = wk.rstat_part + (static_cast<size_t>(w) * gridDim.x + blockIdx.x) * 4;
  const double s1 = block_sum(m1, red), s2 = block_sum(m2, red);
  const double q1 = block_sum(v1, red), q2 = block_sum(v2, red);
  if (tid == 0) {
    part[0] = s1;
    part[1] = s2;
    part[2] = q1;
    part[3] = q2;
  }
}

// ===========================================================================
// colpass2d: for every kept column k2 the spectrum exp(X - r0) with the
// shifts, times dataset f's noise factor, and the inverse transform into
// Q[k2][i] (in place of YT's column).  kForward: from YT by the forward
// transform, the spectrum kept in PR when more datasets follow; else from PR.
// cg columns together.  Bound by LDS traffic and barriers of the stages:
// 651 us for 32 walkers at 2048, 534 + 526 as two kernels with the spectrum
// through memory between them.
// ===========================================================================
template <bool kForward>
__global__ __launch_bounds__(kTR) void colpass2d_kernel(const Set2Dev s, const Work2 wk,
                                                        const int f, const int cg) {
  extern __shared__ double2 lds[];
  const int w = blockIdx.y;
  const double* m = model_ptr(wk, w);
  if (m[0] != POFD_OK) return;
  const int K1 = static_cast<int>(m[3]), K2 = static_cast<int>(m[4]);
  const int n = s.n, ncplx = n / 2 + 1, tid = threadIdx.x;
  const int T = kTR / cg, grp = tid / T, t = tid & (T - 1);
  const int swz = swizzle_of(n);
  double2* tw = lds;
  double2* a = lds + n / 4 + static_cast<size_t>(grp) * 2 * n;
  double2* b = a + n;
  load_turns(tw, s.tw_n, n);
  const double* st = wk.stats + static_cast<size_t>(w) * kStats;
  const double r0 = st[ST2_R0];
  const bool ds1 = st[ST2_DOSHIFT1] != 0.0, ds2 = st[ST2_DOSHIFT2] != 0.0;
  const double sf1 = st[ST2_SHIFT1] * s.iflux1, sf2 = st[ST2_SHIFT2] * s.iflux2;
  const double sigma1 = m[1] * s.fields[f].sigma_base1;
  const double sigma2 = m[2] * s.fields[f].sigma_base2;
  const bool noisy = (sigma1 > 0 || sigma2 > 0);
  const double sigfac1 = -0.5 * sigma1 * sigma1 * s.iflux1 * s.iflux1;
  const double sigfac2 = -0.5 * sigma2 * sigma2 * s.iflux2 * s.iflux2;
  for (int c0 = blockIdx.x * cg; c0 <= K2; c0 += gridDim.x * cg) {  // uniform
    const int k2 = c0 + grp;
    const bool on = k2 <= K2;
    double2* col = wk.YT + static_cast<size_t>(w) * wk.YT_stride + static_cast<size_t>(k2) * n;
    double2* pr = wk.PR + static_cast<size_t>(w) * wk.PR_stride + static_cast<size_t>(k2) * n;
    const double2* X = nullptr;
    double2* z = a;
    if (kForward) {
      if (on)
        for (int e = t; e < n; e += T) a[slot(e, swz)] = col[e];
      __syncthreads();
      X = fft_lds(a, b, n, tw, t, T);
      z = (X == a) ? b : a;
    }
    if (on) {
      for (int k1 = t; k1 < n; k1 += T) {
        const bool kept = (k1 <= K1) || (k1 >= n - K1);
        double2 v = make_double2(0.0, 0.0);
        if (kept) {
#pragma clang fp contract(off)
          if (kForward) {
            const double2 xv = X[slot(k1, swz)];
            const double rval = xv.x - r0;
            double ival = xv.y;
            double sp1 = 0.0;
            if (ds1)
              sp1 = (k1 < ncplx) ? sf1 * static_cast<double>(k1)
                                 : -sf1 * static_cast<double>(n - k1);
            if (ds1 && ds2)
              ival = ival - sp1 - sf2 * static_cast<double>(k2);
            else if (ds1)
              ival = ival - sp1;
            else if (ds2)
              ival = ival - sf2 * static_cast<double>(k2);
            const double ef = exp(rval);
            double sn, cs;
            sincos(ival, &sn, &cs);
            v = make_double2(ef * cs, ef * sn);
            if (k1 == 0 && k2 == 0) v = make_double2(1.0, 0.0);
            if (s.nfields > 1) pr[k1] = v;
          } else {
            v = pr[k1];
          }
          if (noisy) {
            const double didx1 =
                (k1 < ncplx) ? static_cast<double>(k1) : static_cast<double>(n - k1);
            const double didx2 = static_cast<double>(k2);
            const double ef = exp(sigfac1 * didx1 * didx1 + sigfac2 * didx2 * didx2);
            v = make_double2(ef * v.x, ef * v.y);
          }
          if (k1 == 0 && k2 == 0) v = make_double2(1.0, 0.0);
        }
        z[slot(k1, swz)] = make_double2(v.y, v.x);
      }
    }
    __syncthreads();
    const double2* q = fft_lds(z, (z == a) ? b : a, n, tw, t, T);
    if (on)
      for (int i = t; i < n; i += T) {
        const double2 v = q[slot(i, swz)];
        col[i] = make_double2(v.y, v.x);
      }
    __syncthreads();
  }
}

// ===========================================================================
// rowifft2d: c2r of every row from Q[0..n/2][i] (zero beyond K2), clamp,
// store P, the row trapezoid marginal and this workgroup's share of the
// column one.  rg rows together, as rowfft2d.  Bound by LDS traffic and
// barriers of the stages: 673 us for 32 walkers at 2048, 195 + 642 as a
// transposition and the rows.
// ===========================================================================
__global__ __launch_bounds__(kTR) void rowifft2d_kernel(const Set2Dev s, const Work2 wk,
                                                        const int f, const int rg) {
  extern __shared__ double2 lds[];
  __shared__ double red[kTR / 64];
  const int w = blockIdx.y;
  const double* m = model_ptr(wk, w);
  if (m[0] != POFD_OK) return;
  const int K2 = static_cast<int>(m[4]);
  const int n = s.n, h = n / 2, tid = threadIdx.x;
  const int T = kTR / rg, grp = tid / T, t = tid & (T - 1);
  const int swz = swizzle_of(h);
  double2* tw = lds;
  double2* rows = lds + h / 4;
  const int rs = n + 2;
  load_turns(tw, s.tw_half, h);
  const size_t wf = static_cast<size_t>(w) * s.nfields + f;
  const double2* Q = wk.YT + static_cast<size_t>(w) * wk.YT_stride;
  double cacc[2 * kMaxPairs];
#pragma unroll
  for (int q = 0; q < 2 * kMaxPairs; ++q) cacc[q] = 0.0;
  for (int i0 = blockIdx.x * rg; i0 < n; i0 += gridDim.x * rg) {
    for (int o = tid; o < rg * (h / 2 + 1); o += kTR) {
      const int k = o / rg, row = o - k * rg, mk = h - k;
      const double2* X = Q + i0 + row;
      double2 xa = (k <= K2) ? X[static_cast<size_t>(k) * n] : make_double2(0.0, 0.0);
      double2 xb = (mk <= K2) ? X[static_cast<size_t>(mk) * n] : make_double2(0.0, 0.0);
      if (k == 0) {  // FFTW's c2r ignores Im of the k2 = 0 and n/2 entries
        xa.y = 0.0;
        xb.y = 0.0;
      }
      const double2 E = make_double2(xa.x + xb.x, xa.y - xb.y);
      const double2 D = make_double2(xa.x - xb.x, xa.y + xb.y);
      const double2 wv = s.tw_n[k];  // e^{-2 pi i k/n}
      const double2 O = cmul(D, make_double2(wv.x, -wv.y));
      double2* a = rows + row * rs;  // (real and imaginary parts exchanged)
      a[slot(k, swz)] = make_double2(E.y + O.x, E.x - O.y);
      if (k > 0 && k < mk) {  // h - k: conj E, -conj D, and the turn -wv
        const double2 O2 = cmul(make_double2(D.x, -D.y), wv);
        a[slot(mk, swz)] = make_double2(-E.y + O2.x, E.x - O2.y);
      }
    }
    __syncthreads();
    const int i = i0 + grp;
    double2* a = rows + grp * rs;
    const double2* z = fft_lds(a, a + h, h, tw, t, T);
    double2* P = reinterpret_cast<double2*>(wk.P + wf * wk.P_stride + static_cast<size_t>(i) * n);
    const double wi = (i == 0 || i == n - 1) ? 0.5 : 1.0;
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < kMaxPairs; ++q) {
      const int m2 = t + q * T;
      if (m2 < h) {
        const double2 v = z[slot(m2, swz)];
        // unwrapAndNormalizePD positivity
        const double x0 = (v.y < 0) ? 0.0 : v.y, x1 = (v.x < 0) ? 0.0 : v.x;
        P[m2] = make_double2(x0, x1);
        const double w0 = (m2 == 0) ? 0.5 : 1.0;
        const double w1 = (m2 == h - 1) ? 0.5 : 1.0;
        part += w0 * x0 + w1 * x1;
        cacc[2 * q] += wi * x0;
        cacc[2 * q + 1] += wi * x1;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
    if ((tid & 63) == 0) red[tid >> 6] = part;
    __syncthreads();
    if (t == 0) {
      double v = red[tid >> 6];
      for (int u = 1; u < T / 64; ++u) v += red[(tid >> 6) + u];
      wk.rsum1[wf * wk.edge_stride + i] = v;
    }
    // (red is written again behind the next transform's barriers)
  }
  // the column sums of the rg rows' threads, in row order
  __syncthreads();
  double2* cs = rows;
#pragma unroll
  for (int q = 0; q < kMaxPairs; ++q) {
    const int m2 = t + q * T;
    if (m2 < h) cs[grp * h + m2] = make_double2(cacc[2 * q], cacc[2 * q + 1]);
  }
  __syncthreads();
  double2* cp = reinterpret_cast<double2*>(wk.colpart + static_cast<size_t>(w) * wk.colpart_stride +
                                           static_cast<size_t>(blockIdx.x) * n);
  for (int e = tid; e < h; e += kTR) {
    double2 v = cs[e];
    for (int u = 1; u < rg; ++u) v = cadd(v, cs[u * h + e]);
    cp[e] = v;
  }
}

// column trapezoid marginal (unwrapAndNormalizePD, src/PDFactoryDouble.cc:
// 1001-1011) from the per-workgroup partial sums of rowifft2d, thread per
// column
__global__ void colsum2d_kernel(const Set2Dev s, const Work2 wk, const int f) {
  const int w = blockIdx.y;
  if (model_ptr(wk, w)[0] != POFD_OK) return;
  const int n = s.n;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const size_t wf = static_cast<size_t>(w) * s.nfields + f;
  const double* cp = wk.colpart + static_cast<size_t>(w) * wk.colpart_stride + j;
  double acc = 0.0;
  for (int b = 0; b < kRowBlocks2; ++b) acc += cp[static_cast<size_t>(b) * n];
  wk.rsum2[wf * wk.edge_stride + j] = acc;
}

// ===========================================================================
// split2d: findSplitPoint (src/PDFactoryDouble.cc:784-975) on the marginal of
// one axis; one workgroup per (axis, walker)
// ===========================================================================
__global__ __launch_bounds__(kT) void split2d_kernel(const Set2Dev s, const Work2 wk,
                                                     const int f) {
  __shared__ double red[kT / 64];
  __shared__ int ired[kT / 64];
  __shared__ int ires[3];
  __shared__ double dres[1];
  const int axis = blockIdx.x, w = blockIdx.y;
  const double* m = model_ptr(wk, w);
  if (m[0] != POFD_OK) return;  // uniform
  const int tid = threadIdx.x;
  const size_t wf = static_cast<size_t>(w) * s.nfields + f;
  double* dbg = wk.dbg + wf * kDbg2;
  const double* st = wk.stats + static_cast<size_t>(w) * kStats;
  const double sigma = m[1 + axis] * (axis ? s.fields[f].sigma_base2 : s.fields[f].sigma_base1);
  const double var = st[ST2_VAR1 + axis];
  const double sgpos = sqrt(var + sigma * sigma);
  const double sgneg = (9 * sigma * sigma > var) ? sigma : sgpos;  // getPD, :1413-1420
  const double* data = (axis ? wk.rsum2 : wk.rsum1) + wf * wk.edge_stride;
  const double dflux = axis ? s.dflux2 : s.dflux1;
  const int cs = s.n;
  const double n1 = 2.25, f1 = 5e-14, f2 = 1.5e-5, f3 = 5;
  int status = POFD_OK;
  if (sgpos <= 0 || sgneg <= 0) status = POFD_E_SPLIT;
  const double fluxrange = cs * dflux;
  const double n1sigpos = n1 * sgpos, n1signeg = n1 * sgneg;
  if (fluxrange < (n1sigpos + n1signeg)) status = POFD_E_SPLIT;
  auto clampi = [](double v) { return static_cast<int>(v > 2e9 ? 2e9 : (v < -2e9 ? -2e9 : v)); };
  const int topidx = cs - clampi(n1signeg / dflux) - 1;
  const int botidx = clampi(n1sigpos / dflux);
  if (topidx >= cs || botidx < 0 || botidx > topidx) status = POFD_E_SPLIT;
  int split = -1;
  if (status == POFD_OK) {  // uniform across the workgroup
    double pk = -1.0;
    for (int i = tid; i < cs; i += kT) pk = fmax(pk, data[i]);
    const double peak = block_max(pk, red);
    // first minimum over [botidx, topidx]
    double mv = 0.0;
    int mi = -1;
    for (int i = botidx + tid; i <= topidx; i += kT) {
      const double v = data[i];
      if (mi < 0 || v < mv) {
        mv = v;
        mi = i;
      }
    }
    block_argmin(mv, mi, red, ired);
    if (tid == 0) {
      int stt = (peak <= 0.0 || mv > f2 * peak) ? POFD_E_SPLIT : POFD_OK;
      int decided = 0, sp = -1;
      double minval = mv, jitter = 0.0;
      const int minidx = mi;
      if (stt == POFD_OK) {
        const int pre_jitter_n = 17;
        if (minidx > pre_jitter_n) {
          bool mono = true;
          const int initidx = minidx - pre_jitter_n;
          double prev = data[initidx];
          jitter = prev;
          for (int i = initidx + 1; i < minidx; ++i) {
            const double cv = data[i];
            if (cv >= prev) mono = false;
            jitter += cv;
            prev = cv;
          }
          if (mono) {
            sp = minidx;
            decided = 1;
          } else {
            jitter += minval;
            jitter = 1.1 * jitter / static_cast<double>(pre_jitter_n + 1);
          }
        } else {
          jitter = f1 * peak;
          if (minval > jitter) {
            sp = minidx;
            decided = 1;
          }
        }
      }
      if (stt == POFD_OK && !decided) {
        if (minval <= 0.0) {
          const int nminup = 3;
          int bi, ti;
          if (minidx < botidx)
            bi = botidx;
          else
            bi = (minidx >= nminup) ? (minidx - nminup) : minidx;
          ti = (minidx > topidx - nminup) ? topidx - nminup : minidx + nminup;
          ti = (ti >= cs) ? (cs - 1) : ti;
          for (int i = bi; i < ti; ++i)
            if (data[i] > minval) minval = data[i];
        }
        if (minval > 0) jitter = (f3 * minval) < jitter ? (f3 * minval) : jitter;
        if (botidx >= topidx || data[topidx] < jitter) stt = POFD_E_SPLIT;
      }
      ires[0] = stt;
      ires[1] = decided;
      ires[2] = sp;
      dres[0] = jitter;
    }
    __syncthreads();
    status = ires[0];
    split = ires[2];
    if (status == POFD_OK && !ires[1]) {
      // the largest i in [botidx, topidx - 1] with data[i] < jitter
      const double jitter = dres[0];
      int cand = -1;
      for (int i = botidx + tid; i <= topidx - 1; i += kT)
        if (data[i] < jitter) cand = i;
      const int found = block_max_int(cand, ired);
      if (found < 0)
        status = POFD_E_SPLIT;
      else
        split = found + 1;
    }
  }
  if (tid == 0) {
    dbg[D2_ST1 + axis] = status;
    dbg[D2_SPLIT1 + axis] = split;
    dbg[D2_SG1POS + axis] = sgpos;
    dbg[D2_SIGMA1 + axis] = sigma;
  }
}

// norm2d: the split status, then integral, means and minflux of the rotated
// array (PDDouble::getIntegral / getMeans), one workgroup per walker.  The
// trapezoid sums of its rows and columns are the marginals of the unrotated
// array, with the ends' weights moved: A = rsum1 + (P[i][0] + P[i][n-1]) / 2
// - (P[i][s2] + P[i][s2-1]) / 2, and so for the columns; all terms are
// non-negative parts of the sum.  Latency of 8 n gathered values and the 2 n
// of the marginals; summing
// the array itself again read 1.07 GB (268 us at 32 walkers, n = 2048).
constexpr int kTN = 1024;
__global__ __launch_bounds__(kTN) void norm2d_kernel(const Set2Dev s, const Work2 wk,
                                                     const int f) {
  __shared__ double red[kTN / 64];
  const int w = blockIdx.x;
  if (model_ptr(wk, w)[0] != POFD_OK) return;
  const size_t wf = static_cast<size_t>(w) * s.nfields + f;
  double* dbg = wk.dbg + wf * kDbg2;
  const int st1 = static_cast<int>(dbg[D2_ST1]), st2 = static_cast<int>(dbg[D2_ST2]);
  const int sst = (st1 != POFD_OK) ? st1 : st2;  // band 1 is searched first
  if (sst != POFD_OK) {
    if (threadIdx.x == 0) dbg[D2_STATUS] = sst;
    return;
  }
  const int n = s.n;
  const int s1 = static_cast<int>(dbg[D2_SPLIT1]), s2 = static_cast<int>(dbg[D2_SPLIT2]);
  const int e1 = (s1 + n - 1) & (n - 1), e2 = (s2 + n - 1) & (n - 1);
  const double* P = wk.P + wf * wk.P_stride;
  const double* r1 = wk.rsum1 + wf * wk.edge_stride;
  const double* r2 = wk.rsum2 + wf * wk.edge_stride;
  const double *p0 = P, *pn = P + static_cast<size_t>(n - 1) * n;
  const double *ps = P + static_cast<size_t>(s1) * n, *pe = P + static_cast<size_t>(e1) * n;
  double tp = 0.0, m1p = 0.0, m2p = 0.0;
  for (int ip = threadIdx.x; ip < n; ip += kTN) {
    const double wi = (ip == 0 || ip == n - 1) ? 0.5 : 1.0;
    const int i = (ip + s1) & (n - 1), j = (ip + s2) & (n - 1);
    const double* row = P + static_cast<size_t>(i) * n;
    const double A = r1[i] + 0.5 * (row[0] + row[n - 1]) - 0.5 * (row[s2] + row[e2]);
    const double C = r2[j] + 0.5 * (p0[j] + pn[j]) - 0.5 * (ps[j] + pe[j]);
    tp += wi * A;
    m1p += wi * static_cast<double>(ip) * A;
    m2p += wi * static_cast<double>(ip) * C;
  }
  const double tot = block_sum(tp, red);
  const double mean1 = block_sum(m1p, red);
  const double mean2 = block_sum(m2p, red);
  if (threadIdx.x == 0) {
    const double integral = tot * s.dflux1 * s.dflux2;
    const double itot = 1.0 / integral;
    // getMeans on the normalised array (PDDouble.cc:355-452, donorm false)
    const double m1 = mean1 * itot * (s.dflux1 * s.dflux1 * s.dflux2);
    const double m2 = mean2 * itot * (s.dflux1 * s.dflux2 * s.dflux2);
    int status = POFD_OK;
    if (isinf(m1) || isnan(m1) || isinf(m2) || isnan(m2)) status = POFD_E_MEAN;
    dbg[D2_STATUS] = status;
    dbg[D2_INTEGRAL] = integral;
    dbg[D2_ITOT] = itot;
    dbg[D2_MINFLUX1] = -m1;
    dbg[D2_MINFLUX2] = -m2;
  }
}

// like2d: bilinear interpolation of log2 of the normalised, rotated P(D)
// over bins (binned) or pixel pairs; partial sums per block
__global__ __launch_bounds__(kT) void like2d_kernel(const Set2Dev s, const Work2 wk,
                                                    const int f) {
  __shared__ double red[kT / 64];
  const int w = blockIdx.y;
  const size_t wf = static_cast<size_t>(w) * s.nfields + f;
  double* part = wk.lpart + wf * kLikeBlocks + blockIdx.x;
  const double* dbg = wk.dbg + wf * kDbg2;
  if (model_ptr(wk, w)[0] != POFD_OK || dbg[D2_STATUS] != POFD_OK) {
    if (threadIdx.x == 0) *part = 0.0;
    return;
  }
  const Field2Dev& fd = s.fields[f];
  const int n = s.n;
  const int s1 = static_cast<int>(dbg[D2_SPLIT1]), s2 = static_cast<int>(dbg[D2_SPLIT2]);
  const double itot = dbg[D2_ITOT];
  const double minflux1 = dbg[D2_MINFLUX1], minflux2 = dbg[D2_MINFLUX2];
  const double dflux1 = s.dflux1, dflux2 = s.dflux2;
  const double* P = wk.P + wf * wk.P_stride;
  auto L = [&](int i, int j) {  // log2 of the rotated, normalised P(D)
    int ii = i + s1;
    if (ii >= n) ii -= n;
    int jj = j + s2;
    if (jj >= n) jj -= n;
    return log2_or_small(P[static_cast<size_t>(ii) * n + jj] * itot);
  };
  double acc = 0.0;
  {
#pragma clang fp contract(off)
    const double maxflux1 = minflux1 + static_cast<double>(n - 1) * dflux1;
    const double maxflux2 = minflux2 + static_cast<double>(n - 1) * dflux2;
    const double idflux1 = 1.0 / dflux1, idflux2 = 1.0 / dflux2;
    const uint64_t nitems = fd.binned ? static_cast<uint64_t>(fd.nb1) * fd.nb2 : fd.npix;
    const uint64_t per = (nitems + kLikeBlocks - 1) / kLikeBlocks;
    const uint64_t i0 = per * blockIdx.x;
    const uint64_t i1 = (i0 + per < nitems) ? i0 + per : nitems;
    for (uint64_t it = i0 + threadIdx.x; it < i1; it += kT) {
      double c1, c2, wgt;
      if (fd.binned) {
        const uint32_t nin = fd.bins[it];
        if (nin == 0) continue;
        const uint32_t b1 = static_cast<uint32_t>(it / fd.nb2), b2 = static_cast<uint32_t>(it % fd.nb2);
        c1 = fd.bincent01 + static_cast<double>(b1) * fd.bindelta1;
        c2 = fd.bincent02 + static_cast<double>(b2) * fd.bindelta2;
        wgt = static_cast<double>(nin);
      } else {
        c1 = fd.d1[it];
        c2 = fd.d2[it];
        wgt = 1.0;
      }
      const double delt1 = (c1 - minflux1) * idflux1;
      const double delt2 = (c2 - minflux2) * idflux2;
      const int idx1 = static_cast<int>(delt1), idx2 = static_cast<int>(delt2);
      double iv;
      // binned uses </> at the edges, unbinned <=/>= (PDDouble.cc:1029-1048,
      // 1140-1158)
      const bool lo1 = fd.binned ? (c1 < minflux1) : (c1 <= minflux1);
      const bool hi1 = fd.binned ? (c1 > maxflux1) : (c1 >= maxflux1);
      const bool lo2 = fd.binned ? (c2 < minflux2) : (c2 <= minflux2);
      const bool hi2 = fd.binned ? (c2 > maxflux2) : (c2 >= maxflux2);
      if (lo1) {
        iv = lo2 ? L(0, 0) : (hi2 ? L(0, n - 1) : L(0, idx2));
      } else if (hi1) {
        iv = lo2 ? L(n - 1, 0) : (hi2 ? L(n - 1, n - 1) : L(n - 1, idx2));
      } else if (lo2) {
        iv = L(idx1, 0);
      } else if (hi2) {
        iv = L(idx1, n - 1);
      } else {
        const double t = delt1 - static_cast<double>(idx1);
        const double u = delt2 - static_cast<double>(idx2);
        const double omu = 1.0 - u, omt = 1.0 - t;
        iv = omt * (omu * L(idx1, idx2) + u * L(idx1, idx2 + 1)) +
             t * (omu * L(idx1 + 1, idx2) + u * L(idx1 + 1, idx2 + 1));
      }
      acc += wgt * iv;
    }
  }
  const double sb = block_sum(acc, red);
  if (threadIdx.x == 0) *part = sb;
}

// combine2d: per walker, datasets in order
__global__ void combine2d_kernel(const Set2Dev s, const Work2 wk, const int accumulate,
                                 double* __restrict__ loglike, int32_t* __restrict__ status) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= wk.nwalk) return;
  const double* m = model_ptr(wk, w);
  const int st = static_cast<int>(m[0]);
  const double prev = accumulate ? loglike[w] : 0.0;
  if (st == POFD_E_BADLIKE) {
    status[w] = st;
    loglike[w] = prev + 1e25;
    return;
  }
  if (st != POFD_OK) {
    status[w] = st;
    loglike[w] = __longlong_as_double(0x7ff8000000000000ULL);
    return;
  }
  double total = 0.0;
  for (int f = 0; f < s.nfields; ++f) {
    const size_t wf = static_cast<size_t>(w) * s.nfields + f;
    double* dbg = wk.dbg + wf * kDbg2;
    const int fs = static_cast<int>(dbg[D2_STATUS]);
    if (fs != POFD_OK) {
      status[w] = fs;
      loglike[w] = __longlong_as_double(0x7ff8000000000000ULL);
      return;
    }
    const double* lp = wk.lpart + wf * kLikeBlocks;
    double s2 = 0.0;
    for (int b = 0; b < kLikeBlocks; ++b) s2 += lp[b];
    const double curr = 0.69314718055994530942 * s2;  // log2toe
    dbg[D2_LL] = curr;
    total += (curr - s.fields[f].like_offset) / s.fields[f].like_norm;
  }
  status[w] = POFD_OK;
  loglike[w] = prev + total;
}

// combine the moments' partials, decide the shifts, and r0 = Re X[0][0]: the
// k2 = 0 column transform at k1 = 0 is the sum of the k2 = 0 row outputs;
// one workgroup per walker
__global__ __launch_bounds__(kT) void rstats2d_kernel(const Set2Dev s, const Work2 wk,
                                                      const int nparts) {
  __shared__ double red[kT / 64];
  const int w = blockIdx.x;
  if (model_ptr(wk, w)[0] != POFD_OK) return;
  const double2* col = wk.YT + static_cast<size_t>(w) * wk.YT_stride;  // k2 = 0
  double a = 0.0;
  for (int i = threadIdx.x; i < s.n; i += kT) a += col[i].x;
  const double r0 = block_sum(a, red);
  const double* part = wk.rstat_part + static_cast<size_t>(w) * nparts * 4;
  double mom[4] = {0.0, 0.0, 0.0, 0.0};
  for (int b = threadIdx.x; b < nparts; b += kT)
    for (int q = 0; q < 4; ++q) mom[q] += part[4 * b + q];
  for (int q = 0; q < 4; ++q) mom[q] = block_sum(mom[q], red);
  if (threadIdx.x != 0) return;
  double* st = wk.stats + static_cast<size_t>(w) * kStats;
  st[ST2_R0] = r0;
  st[ST2_MN1] = mom[0];
  st[ST2_MN2] = mom[1];
  st[ST2_VAR1] = mom[2];
  st[ST2_VAR2] = mom[3];
  const double sg1 = sqrt(mom[2]), sg2 = sqrt(mom[3]);
  const bool d1 = (sg1 > s.dflux1) && (fabs(mom[0]) > s.dflux1);
  const bool d2 = (sg2 > s.dflux2) && (fabs(mom[1]) > s.dflux2);
  st[ST2_DOSHIFT1] = d1 ? 1.0 : 0.0;
  st[ST2_DOSHIFT2] = d2 ? 1.0 : 0.0;
  st[ST2_SHIFT1] = d1 ? -mom[0] : 0.0;
  st[ST2_SHIFT2] = d2 ? -mom[1] : 0.0;
}

}  // namespace pofd2

namespace pofd2 {

// dynamic LDS of the transforms: a quarter turn of twiddles and both buffers
// of each row or column
inline size_t row_lds(const int n) {
  return (static_cast<size_t>(n / 8) + rows_together(n) * (n + 2)) * sizeof(double2);
}
inline size_t col_lds(const int n) {
  return (static_cast<size_t>(n / 4) + cols_together(n) * 2 * n) * sizeof(double2);
}

// Allows the transforms the LDS of the largest grid on the current device.
// The attribute belongs to the kernel, not to a context: one value for all,
// so that no thread lowers it between another's call and launch.
int init_kernels2d() {
  size_t row = 0, col = 0;
  for (int n = kMinN; n <= kMaxN; n *= 2) {
    row = std::max(row, row_lds(n));
    col = std::max(col, col_lds(n));
  }
  auto allow = [](const void* k, const size_t bytes) {
    return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(bytes)) == hipSuccess;
  };
  const bool ok = allow(reinterpret_cast<const void*>(rowfft2d_kernel), row) &&
                  allow(reinterpret_cast<const void*>(rowifft2d_kernel), row) &&
                  allow(reinterpret_cast<const void*>(colpass2d_kernel<true>), col) &&
                  allow(reinterpret_cast<const void*>(colpass2d_kernel<false>), col);
  return ok ? POFD_OK : POFD_E_INTERNAL;
}

int launch_loglike2d(const Set2Dev& s, const Work2& wk, const RGrid& gmain,
                     const RGrid& g00, const RGrid& gx, const RGrid& gy,
                     const float* d_theta, uint32_t stride, double* d_ll,
                     int32_t* d_st, int accumulate, void* stream, hipEvent_t* ev) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int W = wk.nwalk, n = s.n, ne = s.nedge;
  auto mark = [&](int i) {
    if (ev) (void)hipEventRecord(ev[i], st);
  };
  // a grid's per-row beam pieces
  auto pieces = [&](const RGrid& g) {
    const int pb = static_cast<int>((static_cast<size_t>(g.n1) * (wk.rpieces_w / 3) + kT - 1) / kT);
    hipLaunchKernelGGL(rpieces2d_kernel, dim3(pb, W), dim3(kT), 0, st, s, wk, g);
  };
  auto edge_rows = [&](const RGrid& g, double* out) {
    hipLaunchKernelGGL(edge2d_rows_kernel, dim3((g.n1 + kT / 64 - 1) / (kT / 64), W), dim3(kT), 0,
                       st, s, wk, g, out);
  };
  mark(POFD_STAGE_PREP);
  hipLaunchKernelGGL(prep2d_kernel, dim3(W), dim3(64), 0, st, s, wk, d_theta, stride, d_st,
                     accumulate);
  if (s.bonus) hipLaunchKernelGGL(bonus2d_kernel, dim3(W), dim3(64), 0, st, s, wk);
  mark(POFD_STAGE_FORWARD);
  // (the edge grids' rows are edge1, then rflux1 as in the main grid: two
  // sets of pieces serve the four)
  if (s.edge_integ) {
    const int eparts = std::min(kEdgeParts, ne);
    pieces(g00);
    edge_rows(g00, wk.r00rows);
    hipLaunchKernelGGL(edge2d_cols_kernel,
                       dim3((n + kT * kEdgePts - 1) / (kT * kEdgePts), eparts, W), dim3(kT), 0, st, s,
                       wk, gx);
    hipLaunchKernelGGL(edge2d_sum_kernel, dim3((n + kT - 1) / kT, W), dim3(kT), 0, st, s, wk,
                       eparts);
  }
  pieces(gmain);
  if (s.edge_integ) edge_rows(gy, wk.ry);
  const int nparts = 64;
  const int rg = rows_together(n), cg = cols_together(n);
  const size_t lds_row = row_lds(n), lds_col = col_lds(n);
  hipLaunchKernelGGL(rowfft2d_kernel, dim3(nparts, W), dim3(kTR), lds_row, st, s, wk, gmain, rg);
  hipLaunchKernelGGL(rstats2d_kernel, dim3(W), dim3(kT), 0, st, s, wk, nparts);
  mark(POFD_STAGE_INVERSE);
  for (int f = 0; f < s.nfields; ++f) {
    if (f == 0)
      hipLaunchKernelGGL((colpass2d_kernel<true>), dim3(64, W), dim3(kTR), lds_col, st, s, wk, f,
                         cg);
    else
      hipLaunchKernelGGL((colpass2d_kernel<false>), dim3(64, W), dim3(kTR), lds_col, st, s, wk, f,
                         cg);
    hipLaunchKernelGGL(rowifft2d_kernel, dim3(kRowBlocks2, W), dim3(kTR), lds_row, st, s, wk, f,
                       rg);
    hipLaunchKernelGGL(colsum2d_kernel, dim3((n + 255) / 256, W), dim3(256), 0, st, s, wk, f);
  }
  mark(POFD_STAGE_FINALIZE);
  for (int f = 0; f < s.nfields; ++f) {
    hipLaunchKernelGGL(split2d_kernel, dim3(2, W), dim3(kT), 0, st, s, wk, f);
    hipLaunchKernelGGL(norm2d_kernel, dim3(W), dim3(kTN), 0, st, s, wk, f);
  }
  mark(POFD_STAGE_PIXELS);
  for (int f = 0; f < s.nfields; ++f)
    hipLaunchKernelGGL(like2d_kernel, dim3(kLikeBlocks, W), dim3(kT), 0, st, s, wk, f);
  mark(POFD_STAGE_COMBINE);
  hipLaunchKernelGGL(combine2d_kernel, dim3((W + 63) / 64), dim3(64), 0, st, s, wk, accumulate,
                     d_ll, d_st);
  mark(POFD_NSTAGES);
  return hipGetLastError() == hipSuccess ? POFD_OK : POFD_E_INTERNAL;
}

// calcLikeDouble::getLogLike's prior terms (src/calcLikeDouble.cc:
// 1230-1280): Gaussian priors on the two sigma multipliers (mean 1), on the
// mean flux per area of each band (the CFIRB) and on the mean flux^2 per
// area of each band (the Poisson noise), and the difference regularisation
// of the band-1 knot slopes (numberCountsDoubleLogNormal::
// differenceRegularize, src/numberCountsDoubleLogNormal.cc:2154-2173)
__global__ void prior2d_kernel(const Set2Dev s, const Work2 w, const Prior2Dev pr,
                               const float* __restrict__ theta, const uint32_t stride,
                               const uint32_t nwalk, double* __restrict__ loglike,
                               const int32_t* __restrict__ status) {
  const uint32_t walker = blockIdx.x * blockDim.x + threadIdx.x;
  if (walker >= nwalk) return;
  const int st = status[walker];
  if (st != POFD_OK && st != POFD_E_BADLIKE) return;
  const double h = 0.918938517570495605469;  // log(2 pi) / 2
  const float* t = theta + static_cast<size_t>(walker) * stride;
  const double* bo = w.bonus + static_cast<size_t>(walker) * 8;
  const int nmp = s.nk + s.ns + s.no;
  double add = 0.0;
  for (int b = 0; b < 2; ++b) {
    if (pr.flags & (kP2Sigma1 << b)) {
      const double v = (static_cast<double>(t[nmp + b]) - 1.0) / pr.sigma_width[b];
      add -= h + log(pr.sigma_width[b]) + 0.5 * v * v;
    }
  }
  for (int b = 0; b < 2; ++b) {
    if (pr.flags & (kP2Cfirb1 << b)) {
      const double v = (pr.cfirb_mean[b] - bo[1 + b]) / pr.cfirb_sigma[b];
      add -= h + log(pr.cfirb_sigma[b]) + 0.5 * v * v;
    }
  }
  for (int b = 0; b < 2; ++b) {
    if (pr.flags & (kP2Poisson1 << b)) {
      const double v = (pr.poisson_mean[b] - bo[3 + b]) / pr.poisson_sigma[b];
      add -= h + log(pr.poisson_sigma[b]) + 0.5 * v * v;
    }
  }
  if (pr.reg_alpha > 0.0 && s.nk > 1) {
    const int n = s.nk;
    double mean = 0.0;
    for (int i = 1; i < n; ++i)
      mean += (s.logfac * static_cast<double>(t[i]) - s.logfac * static_cast<double>(t[i - 1])) /
              (s.logknots[i] - s.logknots[i - 1]);
    mean /= static_cast<double>(n - 1);
    double pen = 0.0;
    for (int i = 1; i < n; ++i) {
      const double d =
          (s.logfac * static_cast<double>(t[i]) - s.logfac * static_cast<double>(t[i - 1])) /
              (s.logknots[i] - s.logknots[i - 1]) -
          mean;
      pen -= d * d;
    }
    add += pr.reg_alpha * pen;
  }
  loglike[walker] += add;
}

int launch_prior2d(const Set2Dev& s0, const Work2& w0, const Prior2Dev& pr, const float* d_theta,
                   uint32_t stride, uint32_t nwalk, double* d_ll, const int32_t* d_st,
                   void* stream) {
  hipLaunchKernelGGL(prior2d_kernel, dim3((nwalk + 63) / 64), dim3(64), 0,
                     static_cast<hipStream_t>(stream), s0, w0, pr, d_theta, stride, nwalk, d_ll,
                     d_st);
  return hipGetLastError() == hipSuccess ? POFD_OK : POFD_E_INTERNAL;
}

}  // namespace pofd2
