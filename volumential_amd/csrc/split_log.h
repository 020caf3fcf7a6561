// The logarithm of the split correction's pair loop.
//
// log x for x > 0 by a table of 128 reciprocals (Tang's method): x = 2^e m, m in
// [1/2, 1), c near the midpoint of m's 1/256 interval, log x = e log 2 -
// log(1/c) + log1p(m / c - 1), the last a polynomial of degree 7 (|m / c - 1| <=
// 1/256, next to x = 1 1/128: truncated at 1e-20 and 2e-18).  The intervals below
// 1/sqrt(2) hold log 2m, so that e = 0 around x = 1, and the two next to x = 1
// have c = 1: nothing cancels and the error is relative, 2.5 units of the last
// place of log x at most (the library's 0.6), in 17 instructions.  2D, k = 40, 4096
// boxes of 36 points: kernel 251 us with the library's log, 140 so; k = 2, 64
// points 293 (282 with a table whose error is relative to max(1, |log x|)).
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
constexpr int kSplitLogTwice = 53;  // intervals below 1/sqrt(2): 2m, 2^(e-1)

struct SplitLog {
  double inv, log_c;  // 1 / c rounded, -log of that (or of its half)
};

VL1_LOG_FN void split_log_table(SplitLog* t, int i) {
  const bool twice = i < kSplitLogTwice;
  const double inv = i == 0 ? 2.0 : (i == kSplitLogs - 1 ? 1.0 : 1.0 / (0.5 + (i + 0.5) / (2.0 * kSplitLogs)));
  t[i] = SplitLog{inv, 0.0 - log(twice ? 0.5 * inv : inv)};
}

VL1_LOG_FN double split_log(double x, const SplitLog* t) {
#ifdef __HIP_DEVICE_COMPILE__
  const double m = __builtin_amdgcn_frexp_mant(x);
  const int e = __builtin_amdgcn_frexp_exp(x);
  const int hi = __double2hiint(m);
#else
  int e;
  const double m = std::frexp(x, &e);
  long long bits;
  std::memcpy(&bits, &m, sizeof(bits));
  const int hi = (int)(bits >> 32);
#endif
  const int i = (hi >> 13) & (kSplitLogs - 1);
  const SplitLog q = t[i];
  const double r = fma(m, q.inv, -1.0), r2 = r * r;
  double p = fma(r, 1.0 / 7.0, -1.0 / 6.0);
  p = fma(p, r, 1.0 / 5.0);
  p = fma(p, r, -1.0 / 4.0);
  p = fma(p, r, 1.0 / 3.0);
  p = fma(p, r, -1.0 / 2.0);
  const double log2 = 0.693147180559945309417;
  return fma((double)(e - (i < kSplitLogTwice)), log2, q.log_c) + fma(p, r2, r);
}

}  // namespace vl1
