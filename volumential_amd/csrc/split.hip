// Helmholtz split correction of list 1 (base quadrature).
//
// With the split, list 1 of a Helmholtz (or Yukawa, k = i lambda) potential
// is the Laplace-table evaluation plus an online point-to-point sum of the
// smooth remainder R = G_k - G_0 over every list-1 (target box, source box)
// pair (volumential/expansion_wrangler_fpnd.py:3491-3836):
//   corr[t] = sum_{s in list-1 boxes of t} R(|x_t - y_s|) * strength[s],
// strength = density x quadrature weight.  R is the reference's series
// (_HelmholtzSplitSeriesRemainderKernel, 212-312; split_series.h), by Horner.
// At r = 0 it gives the self-pair limit of 5293-5317, so self pairs need no
// special case.  N is the caller's series length (4337-4389).  For an axis
// target (source) derivative wrapper of the output kernel (3884-3957) the
// pair value is +(-)(x_a - y_a) R'(r) / r, and self pairs give 0 (the
// reference's limit for a wrapped chain, 5293-5300).
//
// GPU mapping: one workgroup per target box.  The sources of its boxes, up to
// 64 boxes' at a time, are staged in LDS in chunks regardless of box limits
// (coordinates and the complex strengths of RC densities); a lane owns one
// target point and a share of the sources; R is evaluated once per (target,
// source) pair and applied to all RC densities; partial sums are reduced
// through LDS.
// Bound: FP64 VALU, about 2 N + 60 instructions per pair for a real wave
// number.  The series coefficients are kernel arguments, so that a term is one
// instruction with a scalar operand; from LDS each wave took 32 bytes per lane
// and term, and the LDS return path (128 bytes per clock and CU) was the bound:
// 2D, 4096 boxes of 36 points, k = 40, one density 509 us, 138 us so
// (251 us with the library's log).
// A lane takes four sources at a time for the same coefficient.  Where the
// imaginary parts are a quarter of the real log series (real k, order 1), that
// chain serves both.
#include <algorithm>
#include <cmath>
#include <complex>
#include <string>
#include <type_traits>
#include <vector>

#include "internal.h"
#include "split_log.h"
#include "split_series.h"

namespace vl1 {

constexpr int kSplitBlock = 256;

// Pair value: the remainder series, its axis derivative, or the closed
// forms of G_k - G_0 (legacy subtraction).
constexpr int kPairSeries = 0, kPairDeriv = 1, kPairLegacy = 2, kPairLegacyDeriv = 3;

struct SplitParams {
  int dim, n_rhs, nt, n_terms, chunk;
  double k_re, k_im;   // wave number (legacy subtraction)
  int deriv_axis;      // derivative wrapper (DERIV kernels): axis and sign
  double deriv_sign;   // +1 target derivative, -1 source derivative
  const int32_t* target_boxes;
  const int32_t* nbr_starts;
  const int32_t* nbr_lists;
  const int32_t* box_starts;
  const int32_t* box_counts;
  const double* points;  // [dim][n_points]
  int64_t n_points;
  const int32_t* src_starts;  // sources: the targets, or a separate set
  const int32_t* src_counts;
  const double* src_points;   // [dim][n_src]
  int64_t n_src;
  const double* strengths;  // [n_rhs][lds] interleaved complex
  int64_t lds;
  double* result;  // [n_rhs][ldr] interleaved complex
  int64_t ldr;
};

// split_coefficients / split_derivative_coefficients: 2 + 4 values a term at most
struct SplitCoef {
  double v[2 + 4 * kSplitMaxTerms];
};

constexpr int kSplitBoxes = 64;  // source boxes staged together
constexpr int kSplitPairs = 4;   // sources per lane and pass over the series

// The series of remainder_value / remainder_radial_derivative at U points, with
// each coefficient read once.  QUARTER (2D): s_n real and Im b_n = s_n / 4.
template <int DIM, bool DERIV, bool QUARTER, int U>
__device__ __forceinline__ void split_series(const double (&r2)[U], const SplitCoef& cf,
                                             const SplitLog* logs, int N, double (&vr)[U],
                                             double (&vi)[U]) {
  if constexpr (DIM == 2) {
    constexpr int base = DERIV ? 0 : 2;
    double ar[U], ai[U], br[U], bi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) ar[u] = ai[u] = br[u] = bi[u] = 0.0;
    for (int n = N; n >= 1; --n) {
      const double* c = cf.v + base + 4 * (n - 1);
      const double c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ar[u] = fma(ar[u], r2[u], c0);
        br[u] = fma(br[u], r2[u], c2);
        if constexpr (!QUARTER) {
          ai[u] = fma(ai[u], r2[u], c1);
          bi[u] = fma(bi[u], r2[u], c3);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double lg = r2[u] > 0.0 ? -0.25 / M_PI * split_log(r2[u], logs) : 0.0;  // -log(r) / (2 pi)
      if constexpr (QUARTER) bi[u] = 0.25 * ar[u];
      const double w = DERIV ? 1.0 : r2[u];
      vr[u] = w * br[u] + lg * (w * ar[u]);
      vi[u] = QUARTER ? w * bi[u] : w * bi[u] + lg * (w * ai[u]);
      if constexpr (!DERIV) {
        vr[u] += cf.v[0];
        vi[u] += cf.v[1];
      }
    }
  } else {
    double r[U], pr[U], pi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      r[u] = sqrt(r2[u]);
      pr[u] = pi[u] = 0.0;
    }
    for (int n = DERIV ? N - 1 : N; n >= 1; --n) {
      const double c0 = cf.v[2 * (n - 1)], c1 = cf.v[2 * (n - 1) + 1];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        pr[u] = fma(pr[u], r[u], c0);
        pi[u] = fma(pi[u], r[u], c1);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double w = DERIV ? 1.0 / r[u] : 1.0;
      vr[u] = w * pr[u];
      vi[u] = w * pi[u];
    }
  }
}

template <int DIM, int RC, int MODE, bool QUARTER>
__global__ void __launch_bounds__(kSplitBlock)
    split_correction_kernel(const SplitParams p, const SplitCoef cf) {
  constexpr bool DERIV = MODE == kPairDeriv || MODE == kPairLegacyDeriv;
  constexpr bool LEGACY = MODE == kPairLegacy || MODE == kPairLegacyDeriv;
  constexpr int U = LEGACY ? 1 : kSplitPairs;
  extern __shared__ __align__(16) double smem[];
  __shared__ int sOff[kSplitBoxes + 1], sBeg[kSplitBoxes];
  __shared__ __align__(16) SplitLog sLog[kSplitLogs];
  const int N = p.n_terms;
  const int P = kSplitBlock / p.nt;
  const int chunk = p.chunk;         // source points staged per pass
  double* sF = smem;                 // strengths [chunk][RC][2]
  double* sX = sF + (size_t)chunk * RC * 2;  // source coordinates [DIM][chunk]
  double* red = smem;                // part sums [256][RC][2], after the staging is done
  const int tid = threadIdx.x;
  const int lane_t = tid % p.nt;
  const int part = tid / p.nt;
  if (DIM == 2 && tid < kSplitLogs) split_log_table(sLog, tid);  // (a barrier follows)

  const int tbox = blockIdx.x;
  const int tb = p.target_boxes[tbox];
  const int tbeg = p.box_starts[tb];
  const int ntb = p.box_counts[tb];
  const int l0 = p.nbr_starts[tbox], l1 = p.nbr_starts[tbox + 1];

  for (int r0 = 0; r0 < p.n_rhs; r0 += RC) {
    const int rc = min(RC, p.n_rhs - r0);
    for (int t0 = 0; t0 < ntb; t0 += p.nt) {
      const int ti = t0 + lane_t;
      const bool tact = ti < ntb;
      double xt[DIM];
#pragma unroll
      for (int a = 0; a < DIM; ++a) xt[a] = tact ? p.points[(int64_t)a * p.n_points + tbeg + ti] : 0.0;
      double acc[RC], aci[RC];
#pragma unroll
      for (int r = 0; r < RC; ++r) acc[r] = aci[r] = 0.0;
      for (int lb = l0; lb < l1; lb += kSplitBoxes) {
        const int nb = min(kSplitBoxes, l1 - lb);
        __syncthreads();  // the previous boxes are done with
        if (tid < kSplitBoxes) {  // one wave: the boxes' places in the run of sources
          const int sb = tid < nb ? p.nbr_lists[lb + tid] : -1;
          const int ns = sb < 0 ? 0 : p.src_counts[sb];
          int sum = ns;
          for (int o = 1; o < kSplitBoxes; o <<= 1) {
            const int v = __shfl_up(sum, o);
            if (tid >= o) sum += v;
          }
          sOff[tid + 1] = sum;
          if (tid == 0) sOff[0] = 0;
          sBeg[tid] = (sb < 0 ? 0 : p.src_starts[sb]) - (sum - ns);
        }
        __syncthreads();
        const int total = sOff[nb];
        for (int c0 = 0; c0 < total; c0 += chunk) {
          const int nc = min(chunk, total - c0);
          if (c0 > 0) __syncthreads();  // previous chunk done with LDS
          for (int j = tid; j < nc; j += kSplitBlock) {
            int b = 0;  // the last box that begins at or before source c0 + j
#pragma unroll
            for (int o = kSplitBoxes / 2; o > 0; o >>= 1)
              if (b + o < nb && sOff[b + o] <= c0 + j) b += o;
            const int64_t src = (int64_t)sBeg[b] + c0 + j;
#pragma unroll
            for (int a = 0; a < DIM; ++a) sX[a * chunk + j] = p.src_points[(int64_t)a * p.n_src + src];
#pragma unroll
            for (int r = 0; r < RC; ++r) {
              double fr = 0.0, fi = 0.0;
              if (r < rc) {
                const double* f = p.strengths + (int64_t)(r0 + r) * p.lds + 2 * src;
                fr = f[0];
                fi = f[1];
              }
              sF[((size_t)j * RC + r) * 2] = fr;
              sF[((size_t)j * RC + r) * 2 + 1] = fi;
            }
          }
          __syncthreads();
          if (tact && part < P) {  // threads past P * nt (nt not dividing 256) idle
            for (int j0 = part; j0 < nc; j0 += U * P) {
              double r2[U], da[U], vr[U], vi[U];
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int j = min(j0 + u * P, nc - 1);  // past the chunk: not added below
                r2[u] = da[u] = 0.0;
#pragma unroll
                for (int a = 0; a < DIM; ++a) {
                  const double d = xt[a] - sX[a * chunk + j];
                  r2[u] = fma(d, d, r2[u]);
                  if (DERIV && a == p.deriv_axis) da[u] = d;
                }
              }
              if constexpr (LEGACY) {
                // closed forms off the diagonal; a self pair takes the series at
                // r = 0, the limit the reference adds back (0 under a derivative)
                vr[0] = vi[0] = 0.0;
                if constexpr (MODE == kPairLegacyDeriv) {
                  if (r2[0] > 0.0) legacy_radial_derivative<DIM>(r2[0], p.k_re, p.k_im, vr[0], vi[0]);
                } else if (r2[0] > 0.0) {
                  legacy_difference<DIM>(r2[0], p.k_re, p.k_im, vr[0], vi[0]);
                } else {
                  split_series<DIM, false, false>(r2, cf, sLog, N, vr, vi);
                }
              } else {
                split_series<DIM, DERIV, QUARTER>(r2, cf, sLog, N, vr, vi);
              }
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int j = j0 + u * P;
                if (DERIV) {
                  // +-(x_a - y_a) R'(r) / r; the self pair (r = 0) gives 0
                  const double f = p.deriv_sign * da[u];
                  vr[u] = r2[u] > 0.0 ? vr[u] * f : 0.0;
                  vi[u] = r2[u] > 0.0 ? vi[u] * f : 0.0;
                }
                if (u > 0 && j >= nc) continue;
                const double* f = sF + (size_t)j * RC * 2;
#pragma unroll
                for (int r = 0; r < RC; ++r) {
                  const double fr = f[2 * r], fi = f[2 * r + 1];
                  acc[r] = fma(vr[u], fr, fma(-vi[u], fi, acc[r]));
                  aci[r] = fma(vr[u], fi, fma(vi[u], fr, aci[r]));
                }
              }
            }
          }
        }
      }
      if (P > 1) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          red[((part * p.nt + lane_t) * RC + r) * 2] = acc[r];
          red[((part * p.nt + lane_t) * RC + r) * 2 + 1] = aci[r];
        }
        __syncthreads();
        if (part == 0)
          for (int q = 1; q < P; ++q)
#pragma unroll
            for (int r = 0; r < RC; ++r) {
              acc[r] += red[((q * p.nt + lane_t) * RC + r) * 2];
              aci[r] += red[((q * p.nt + lane_t) * RC + r) * 2 + 1];
            }
      }
      if (part == 0 && tact)
        for (int r = 0; r < rc; ++r) {
          p.result[(int64_t)(r0 + r) * p.ldr + 2 * (int64_t)(tbeg + ti)] = acc[r];
          p.result[(int64_t)(r0 + r) * p.ldr + 2 * (int64_t)(tbeg + ti) + 1] = aci[r];
        }
      __syncthreads();  // reduction buffer reused by the next target chunk
    }
  }
}

template <int DIM, int RC, int MODE, bool QUARTER>
static hipError_t launch_split(const SplitParams& prm, const SplitCoef& cf, int grid, size_t smem,
                               hipStream_t s) {
  auto fn = split_correction_kernel<DIM, RC, MODE, QUARTER>;
  hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(kSplitBlock), smem, s, prm, cf);
  return hipGetLastError();
}

}  // namespace vl1

using namespace vl1;

extern "C" int vl1_split_correction(const vl1_split_args* a, void* stream) {
  clear_error();
  if (!a) return fail(VL1_E_ARG, "vl1_split_correction: null argument");
  if (a->dim != 2 && a->dim != 3) return fail(VL1_E_ARG, "vl1_split_correction: dim must be 2 or 3");
  if (a->split_order < 1 || 2 * (a->split_order - 1) > kSplitMaxTerms)
    return fail(VL1_E_ARG, "vl1_split_correction: split_order must be 1..49");
  if (a->series_nmax < 1 || a->series_nmax > kSplitMaxTerms)
    return fail(VL1_E_ARG, "vl1_split_correction: series_nmax must be 1..96");
  if (a->n_tgt_boxes < 0 || a->n_rhs < 1 || a->n_points < 1 || a->max_box_points < 1)
    return fail(VL1_E_ARG, "vl1_split_correction: bad sizes");
  if (a->n_tgt_boxes == 0) return VL1_OK;
  if (!a->target_boxes || !a->nbr_starts || !a->nbr_lists || !a->box_starts || !a->box_counts ||
      !a->points || !a->strengths || !a->result)
    return fail(VL1_E_ARG, "vl1_split_correction: null device array");
  const bool sep = a->src_points != nullptr;
  if (sep && (!a->src_box_starts || !a->src_box_counts || a->n_src_points < 1 ||
              a->max_src_box_points < 1))
    return fail(VL1_E_ARG, "vl1_split_correction: incomplete separate source set");
  const int64_t n_src = sep ? a->n_src_points : a->n_points;
  if (a->n_rhs > 1 && (a->ld_strengths < 2 * n_src || a->ld_result < 2 * a->n_points))
    return fail(VL1_E_ARG, "vl1_split_correction: bad leading dimension");
  if (a->deriv_kind < VL1_SPLIT_DERIV_NONE || a->deriv_kind > VL1_SPLIT_DERIV_SOURCE)
    return fail(VL1_E_ARG, "vl1_split_correction: bad deriv_kind");
  const bool deriv = a->deriv_kind != VL1_SPLIT_DERIV_NONE;
  if (deriv && (a->deriv_axis < 0 || a->deriv_axis >= a->dim))
    return fail(VL1_E_ARG, "vl1_split_correction: deriv_axis out of range");

  if (a->legacy_subtraction != 0 && a->legacy_subtraction != 1)
    return fail(VL1_E_ARG, "vl1_split_correction: legacy_subtraction must be 0 or 1");
  const bool legacy = a->legacy_subtraction == 1;
  if (legacy && (a->coefficients || a->split_order != 1))
    return fail(VL1_E_UNSUPPORTED,
                "vl1_split_correction: the legacy subtraction takes split order 1 and no "
                "coefficients");
  if (legacy && a->k_im < 0.0)
    return fail(VL1_E_ARG, "vl1_split_correction: the legacy subtraction needs Im k >= 0");
  hipStream_t s = (hipStream_t)stream;
  const std::complex<double> k(a->k_re, a->k_im);
  std::vector<double> coef;
  if (a->coefficients) {
    // value layout, or with a derivative wrapper the R'(r)/r layout
    const int nc = deriv ? (a->dim == 2 ? 4 * a->series_nmax : 2 * (a->series_nmax - 1))
                         : (a->dim == 2 ? 2 + 4 * a->series_nmax : 2 * a->series_nmax);
    coef.assign(a->coefficients, a->coefficients + nc);
    for (double c : coef)
      if (!std::isfinite(c)) return fail(VL1_E_ARG, "vl1_split_correction: coefficients must be finite");
  } else {
    coef = deriv ? split_derivative_coefficients(a->dim, k, a->series_nmax, a->split_order)
                 : split_coefficients(a->dim, k, a->series_nmax, a->split_order);
  }
  SplitCoef cf{};  // zeros past the coefficients (3D derivative with one term: R' = 0)
  std::copy(coef.begin(), coef.end(), cf.v);
  bool quarter = a->dim == 2;
  for (size_t i = deriv ? 0 : 2; i + 3 < coef.size() && quarter; i += 4)
    quarter = coef[i + 1] == 0.0 && coef[i + 3] == 0.25 * coef[i];

  SplitParams prm{};
  prm.dim = a->dim;
  prm.n_rhs = a->n_rhs;
  prm.n_terms = a->series_nmax;
  prm.k_re = a->k_re;
  prm.k_im = a->k_im;
  prm.deriv_axis = deriv ? a->deriv_axis : -1;
  prm.deriv_sign = a->deriv_kind == VL1_SPLIT_DERIV_SOURCE ? -1.0 : 1.0;
  prm.target_boxes = a->target_boxes;
  prm.nbr_starts = a->nbr_starts;
  prm.nbr_lists = a->nbr_lists;
  prm.box_starts = a->box_starts;
  prm.box_counts = a->box_counts;
  prm.points = a->points;
  prm.n_points = a->n_points;
  prm.src_starts = sep ? a->src_box_starts : a->box_starts;
  prm.src_counts = sep ? a->src_box_counts : a->box_counts;
  prm.src_points = sep ? a->src_points : a->points;
  prm.n_src = n_src;
  prm.strengths = a->strengths;
  prm.lds = a->n_rhs > 1 ? a->ld_strengths : 2 * n_src;
  prm.result = a->result;
  prm.ldr = a->n_rhs > 1 ? a->ld_result : 2 * a->n_points;
  // a lane per target (the box's targets, at most a block), P = 256 / nt
  // source parts: 36 targets use 7 parts = 252 of the 256 threads
  const int nt = std::min(a->max_box_points, kSplitBlock);
  prm.nt = nt;
  const int P = kSplitBlock / nt;
  // the remainder is evaluated once per (target, source) pair and RC-chunk;
  // RC <= 8 keeps the LDS small enough for several workgroups per CU
  const int RC = a->n_rhs == 1 ? 1 : (a->n_rhs <= 4 ? 4 : 8);
  // source points staged per pass
  const int chunk = RC == 1 ? 512 : 256;
  prm.chunk = chunk;
  const size_t stage = (size_t)a->dim * chunk + (size_t)chunk * RC * 2;
  const size_t reduce = P > 1 ? (size_t)kSplitBlock * RC * 2 : 0;  // aliases the staging
  const size_t smem = sizeof(double) * std::max(stage, reduce);
  const int grid = a->n_tgt_boxes;
  const int mode = deriv ? (legacy ? kPairLegacyDeriv : kPairDeriv)
                         : (legacy ? kPairLegacy : kPairSeries);
  auto pick = [&](auto dimc, auto modec) {
    constexpr int D = decltype(dimc)::value, M = decltype(modec)::value;
    if constexpr (D == 2 && (M == kPairSeries || M == kPairDeriv)) {
      if (quarter)
        return RC == 1   ? launch_split<D, 1, M, true>(prm, cf, grid, smem, s)
               : RC == 4 ? launch_split<D, 4, M, true>(prm, cf, grid, smem, s)
                         : launch_split<D, 8, M, true>(prm, cf, grid, smem, s);
    }
    return RC == 1   ? launch_split<D, 1, M, false>(prm, cf, grid, smem, s)
           : RC == 4 ? launch_split<D, 4, M, false>(prm, cf, grid, smem, s)
                     : launch_split<D, 8, M, false>(prm, cf, grid, smem, s);
  };
  using D2 = std::integral_constant<int, 2>;
  using D3 = std::integral_constant<int, 3>;
  using MS = std::integral_constant<int, kPairSeries>;
  using MD = std::integral_constant<int, kPairDeriv>;
  using ML = std::integral_constant<int, kPairLegacy>;
  using MLD = std::integral_constant<int, kPairLegacyDeriv>;
  auto by_mode = [&](auto dimc) {
    switch (mode) {
      case kPairDeriv: return pick(dimc, MD{});
      case kPairLegacy: return pick(dimc, ML{});
      case kPairLegacyDeriv: return pick(dimc, MLD{});
      default: return pick(dimc, MS{});
    }
  };
  hipError_t e = a->dim == 2 ? by_mode(D2{}) : by_mode(D3{});
  // as documented: the result is there on return
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return fail(VL1_E_HIP, std::string("vl1_split_correction: ") + hipGetErrorString(e));
  return VL1_OK;
}
