// The logarithm of the split correction's pair loop.
//
// log x for x > 0 by a table of 128 reciprocals (Tang's method): x = 2^e m, m in
// [0.707, 1.414), c near the midpoint of m's interval (1/256 of [0.707, 1), 1/128
// of [1, 1.414)), log x = e log 2 - log(1/c) + log1p(m / c - 1), the last a
// polynomial of degree 7 (|m / c - 1| <= 1/256, next to x = 1 1/128: truncated at
// 1e-20 and 2e-18).  Around x = 1 e is 0 and c 1: nothing cancels and the error is
// relative, 2.5 units of the last place of log x at most (the library's 0.6), in
// 16 instructions.  2D, 4096 boxes: k = 40, 36 points, kernel 251 us with the library's
// log, 138 so; k = 2, 64 points 285.  Subnormal x gives some finite value, which the
// pair loop multiplies by x (by a component of the difference under a derivative).
#pragma once

#include <cmath>
#include <cstring>

#ifdef __HIPCC__
#define VL1_LOG_FN __host__ __device__ __forceinline__
#else
#define VL1_LOG_FN inline
#endif

namespace vl1 {

constexpr int kSplitLogs = 128;
constexpr int kSplitLogFirst = 0x3fe6a000;  // high word of the first interval's start
constexpr int kSplitLogOne = 75;            // the interval that begins at 1

struct SplitLog {
  double inv, log_c;  // 1 / c rounded, -log of that
};

VL1_LOG_FN void split_log_table(SplitLog* t, int i) {
  const int k = i - kSplitLogOne;
  const double inv = k == 0 || k == -1 ? 1.0 : 1.0 / (1.0 + (k + 0.5) / (k < 0 ? 256.0 : 128.0));
  t[i] = SplitLog{inv, 0.0 - log(inv)};
}

VL1_LOG_FN double split_log(double x, const SplitLog* t) {
#ifdef __HIP_DEVICE_COMPILE__
  const int hi = __double2hiint(x), off = hi - kSplitLogFirst;
  const double m = __hiloint2double(hi - (off & ~0xfffff), __double2loint(x));
#else
  long long bits;
  std::memcpy(&bits, &x, sizeof(bits));
  const int hi = (int)(bits >> 32), off = hi - kSplitLogFirst;
  bits -= (long long)(off & ~0xfffff) * (1ll << 32);
  double m;
  std::memcpy(&m, &bits, sizeof(m));
#endif
  const SplitLog q = t[(off >> 13) & (kSplitLogs - 1)];
  const double r = fma(m, q.inv, -1.0), r2 = r * r;
  double p = fma(r, 1.0 / 7.0, -1.0 / 6.0);
  p = fma(p, r, 1.0 / 5.0);
  p = fma(p, r, -1.0 / 4.0);
  p = fma(p, r, 1.0 / 3.0);
  p = fma(p, r, -1.0 / 2.0);
  const double log2 = 0.693147180559945309417;
  return fma((double)(off >> 20), log2, q.log_c) + fma(p, r2, r);
}

}  // namespace vl1
