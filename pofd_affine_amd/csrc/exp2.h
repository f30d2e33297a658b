// The exponential that the one- and two-band fills share.
#pragma once
#include <hip/hip_runtime.h>

namespace pofd {

// 2^(u/32) = exp(u ln 2 / 32) for |u| <= 1/2 as its Taylor polynomial of
// degree 6 (truncation below 4e-18 relative)
__device__ __forceinline__ double exp2_near(const double u) {
  double p = 0x1p-30 * 1.5403530393381609954e-4;      // (ln 2)^6 / 720
  p = fma(p, u, 0x1p-25 * 1.3333558146428443423e-3);  // (ln 2)^5 / 120
  p = fma(p, u, 0x1p-20 * 9.6181291076284771620e-3);  // (ln 2)^4 / 24
  p = fma(p, u, 0x1p-15 * 5.5504108664821579953e-2);  // (ln 2)^3 / 6
  p = fma(p, u, 0x1p-10 * 2.4022650695910071233e-1);  // (ln 2)^2 / 2
  p = fma(p, u, 0x1p-5 * 6.9314718055994530942e-1);   // ln 2
  return fma(p, u, 1.0);
}

}  // namespace pofd
