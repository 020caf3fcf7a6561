// FP64 Duffy quadrature of 3D near-field table entries by sum factorization.
//
// The entries of one target point x share every node y and kernel value; with
// the rule's tensor structure they share far more.  A node of sign block b and
// axis order (a0, a1, a2) is
//   y_{a0} = v + sl rho,  y_{a1} = v + sl rho eta1,  y_{a2} = v + sl rho eta1 eta2
// (sl = sign x len), so with l_m the Lagrange basis
//   T[m] = sum_rho l_{m a0}(y_{a0}) sum_eta1 w l_{m a1}(y_{a1}) G_{rho eta1}[m a2],
//   G[m] = sum_eta2 w2 K(x - y) l_m(y_{a2}):
// only G is summed node by node, q multiply-adds each, for all q^3 modes; the
// node sum of duffy.hip does 3 per node and entry (65 entries per target point
// at q = 6).  Products are formed per axis without division, so a node on an
// interpolation node needs no rule of its own: the basis is 1 and 0 there to
// rounding.
//
// A workgroup takes one (target point, sign block): rows (axis order, rho) in
// chunks of up to 256 pairs (row, eta1), one thread each, for G; then H[row][m1]
// [m2] = sum_eta1 through LDS; then every entry adds its rows.  Empty blocks (some
// len = 0) write zeros, and a second kernel adds the eight blocks in order.
// Bound: FP64 VALU, about 45 instructions per node and target.  3D Laplace q =
// 6, rule 20 / 20, 140496 entries of 2160 target points: 18.3 ms with the node
// sum, 1.04 ms so.
#include <algorithm>
#include <cmath>
#include <string>

#include "duffy_kernels.h"
#include "internal.h"

namespace vl1 {

constexpr int kDtThreads = 256;
constexpr int kDtAcc = 4;  // entries per thread

struct DuffyTensorParams {
  int q, axis, n_rho, n_tail, rows, pitch;  // rows of a chunk; pairs' pitch in LDS
  double k, H;
  int64_t n_targets, n_entries;
  const double* xt;         // [3][n_targets]
  const int64_t* start;     // [n_targets + 1]
  const int32_t* mode;      // [n_entries]
  const double* rho;        // [n_rho], w_rho
  const double* w_rho;
  const double* eta;        // [n_tail], w_eta
  const double* w_eta;
  const double* xi;         // [q]
  double* part;             // [8][n_entries] (x2 complex)
};

// axis a_i of axis order `perm` (0..5): 012 021 102 120 201 210
__device__ inline int dt_axis(int perm, int i) {
  // axes 2 bits each, orders 6 bits each
  constexpr uint64_t t = (0x24ull) | (0x18ull << 6) | (0x21ull << 12) | (0x09ull << 18) |
                         (0x12ull << 24) | (0x06ull << 30);
  return (int)(t >> (6 * perm + 2 * i)) & 3;
}

template <int KIND, int Q>
__global__ void __launch_bounds__(kDtThreads) duffy_tensor_kernel(const DuffyTensorParams p) {
  constexpr int VW = kind_is_complex(KIND) ? 2 : 1, MQ = Q > 0 ? Q : 16;
  const int q = Q > 0 ? Q : p.q;
  // read-only and uniform: scalar loads (as vector loads, two per node, 1.25 ms)
  typedef const __attribute__((address_space(4))) double* scalar_ptr;
  const scalar_ptr xi = (scalar_ptr)(uintptr_t)p.xi;
  const scalar_ptr eta = (scalar_ptr)(uintptr_t)p.eta, w_eta = (scalar_ptr)(uintptr_t)p.w_eta;
  extern __shared__ double dt_smem[];
  double* sL1 = dt_smem;                          // [q][pitch] l(y_a1) x weights
  double* sG = sL1 + (size_t)q * p.pitch;         // [VW][q][pitch]
  double* sL0 = sG + (size_t)VW * q * p.pitch;    // [rows][q]
  double* sH = sL0 + (size_t)p.rows * q;          // [VW][rows][q][q]
  const int tid = threadIdx.x;
  const int64_t tgt = blockIdx.x;
  const int b = blockIdx.y;
  const int64_t first = p.start[tgt], last = p.start[tgt + 1];
  const int64_t e0 = first + (int64_t)blockIdx.z * kDtThreads * kDtAcc;
  // (uniform; entries of ranges outside the arrays, and those past max_entries
  // or of no target point, keep duffy_tensor_fill_kernel's NaN)
  if (last <= e0 || first < 0 || last > p.n_entries) return;
  const int ne = (int)min<int64_t>(last - e0, kDtThreads * kDtAcc);
  double* out = p.part + ((int64_t)b * p.n_entries + e0) * VW;

  double x[3], v[3], sl[3], lenprod = 1.0;
  bool live = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    x[a] = p.xt[a * p.n_targets + tgt];
    v[a] = fmin(fmax(x[a], 0.0), p.H);
    const bool plus = (b >> (2 - a)) & 1;
    const double len = plus ? p.H - v[a] : v[a];
    sl[a] = plus ? len : -len;
    lenprod *= len;
    live = live && len > 0.0;
  }
  if (!live) {  // empty sub-box: every node inactive
    for (int i = tid; i < ne * VW; i += kDtThreads) out[i] = 0.0;
    return;
  }
  double cm[MQ];  // 1 / prod_{j != m} (xi_m - xi_j)
#pragma unroll
  for (int i = 0; i < MQ; ++i) {
    if (Q == 0 && i >= q) break;
    double den = 1.0;
#pragma unroll
    for (int j = 0; j < MQ; ++j)
      if ((Q > 0 || j < q) && j != i) den *= xi[i] - xi[j];
    cm[i] = 1.0 / den;
  }
  // s l_m(y) / c_m for all m, by prefix products (s included) and suffix products
  auto basis = [&](double y, double s, auto&& use) {
    double d[MQ], pre[MQ], acc = s;
#pragma unroll
    for (int j = 0; j < MQ; ++j) {
      if (Q == 0 && j >= q) break;
      d[j] = y - xi[j];
      pre[j] = acc;
      acc *= d[j];
    }
    double suf = 1.0;
#pragma unroll
    for (int j = MQ - 1; j >= 0; --j) {
      if (Q == 0 && j >= q) continue;
      use(j, pre[j], suf);
      suf *= d[j];
    }
  };

  int m0[kDtAcc], m1[kDtAcc], m2[kDtAcc];
  unsigned refused = 0;  // entries with a mode outside the box
  double acc[kDtAcc][VW];
#pragma unroll
  for (int c = 0; c < kDtAcc; ++c) {
    const int i = tid + c * kDtThreads;
    int m = i < ne ? p.mode[e0 + i] : 0;
    if ((unsigned)m >= (unsigned)(q * q * q)) {
      m = 0;
      refused |= 1u << c;
    }
    m2[c] = m % q;
    m1[c] = m / q % q;
    m0[c] = m / (q * q);
#pragma unroll
    for (int w = 0; w < VW; ++w) acc[c][w] = 0.0;
  }

  const int n_rows = 6 * p.n_rho;
  const int pr = tid / p.n_tail, t1 = tid % p.n_tail;  // this thread's pair of a chunk
  for (int r0 = 0; r0 < n_rows; r0 += p.rows) {
    const int nr = min(p.rows, n_rows - r0);
    if (pr < nr) {
      const int row = r0 + pr, perm = row / p.n_rho, ir = row % p.n_rho;
      const int a0 = dt_axis(perm, 0), a1 = dt_axis(perm, 1), a2 = dt_axis(perm, 2);
      auto sel = [](const double (&z)[3], int a) { return a == 0 ? z[0] : (a == 1 ? z[1] : z[2]); };
      const double rho = p.rho[ir], eta1 = p.eta[t1], u1 = rho * eta1;
      const double y0 = fma(sel(sl, a0), rho, sel(v, a0)), y1 = fma(sel(sl, a1), u1, sel(v, a1));
      const double d0 = sel(x, a0) - y0, d1 = sel(x, a1) - y1;
      const double s2 = sel(sl, a2) * u1, v2 = sel(v, a2), x2 = sel(x, a2);
      const double r01 = fma(d0, d0, d1 * d1);
      double g[VW][MQ];
#pragma unroll
      for (int w = 0; w < VW; ++w)
#pragma unroll
        for (int j = 0; j < MQ; ++j) g[w][j] = 0.0;
      for (int t = 0; t < p.n_tail; ++t) {
        const double y2 = fma(s2, eta[t], v2), d2 = x2 - y2, r2 = fma(d2, d2, r01);
        double da = 0.0;
        if (kind_is_deriv(KIND)) da = a0 == p.axis ? d0 : (a1 == p.axis ? d1 : d2);
        double kr = 0.0, ki = 0.0;
        kernel_value<3, KIND>(r2, da, p.k, kr, ki);
        const double w2 = w_eta[t];
        kr = r2 > 0.0 ? kr * w2 : 0.0;
        if (VW == 1) {
          basis(y2, kr, [&](int j, double pre, double suf) { g[0][j] = fma(pre, suf, g[0][j]); });
        } else {
          ki = r2 > 0.0 ? ki * w2 : 0.0;
          basis(y2, 1.0, [&](int j, double pre, double suf) {
            const double l = pre * suf;
            g[0][j] = fma(kr, l, g[0][j]);
            g[VW - 1][j] = fma(ki, l, g[VW - 1][j]);
          });
        }
      }
      // the weights outside the innermost sum go with the second axis
      basis(y1, rho * rho * eta1 * p.w_eta[t1] * p.w_rho[ir] * lenprod,
            [&](int j, double pre, double suf) { sL1[j * p.pitch + tid] = cm[j] * (pre * suf); });
#pragma unroll
      for (int j = 0; j < MQ; ++j) {
        if (Q == 0 && j >= q) break;
#pragma unroll
        for (int w = 0; w < VW; ++w) sG[(w * q + j) * p.pitch + tid] = cm[j] * g[w][j];
      }
      if (t1 == 0)
        basis(y0, 1.0, [&](int j, double pre, double suf) { sL0[pr * q + j] = cm[j] * (pre * suf); });
    }
    __syncthreads();
    // H[row][m1][m2], kMG of the m2 per thread
    constexpr int MG = MQ <= 5 ? MQ : (MQ == 6 ? 3 : 4);
    const int ng = (q + MG - 1) / MG;
    for (int i = tid; i < nr * q * ng; i += kDtThreads) {
      const int gq = i % ng * MG, m = i / ng % q, row = i / (ng * q);
      const double* l1 = sL1 + m * p.pitch + row * p.n_tail;
#pragma unroll
      for (int w = 0; w < VW; ++w) {
        const double* gg = sG + (size_t)(w * q) * p.pitch + row * p.n_tail;
        double h[MG];
#pragma unroll
        for (int c = 0; c < MG; ++c) h[c] = 0.0;
        for (int t = 0; t < p.n_tail; ++t) {
          const double l = l1[t];
#pragma unroll
          for (int c = 0; c < MG; ++c) h[c] = fma(l, gg[min(gq + c, q - 1) * p.pitch + t], h[c]);
        }
#pragma unroll
        for (int c = 0; c < MG; ++c)
          if (gq + c < q) sH[((size_t)(w * p.rows + row) * q + m) * q + gq + c] = h[c];
      }
    }
    __syncthreads();
    for (int row = 0; row < nr; ++row) {
      const int perm = (r0 + row) / p.n_rho;
      const int a0 = dt_axis(perm, 0), a1 = dt_axis(perm, 1), a2 = dt_axis(perm, 2);
#pragma unroll
      for (int c = 0; c < kDtAcc; ++c) {
        if (c * kDtThreads >= ne) break;  // uniform
        auto sel = [&](int a) { return a == 0 ? m0[c] : (a == 1 ? m1[c] : m2[c]); };
        const double l0 = sL0[row * q + sel(a0)];
#pragma unroll
        for (int w = 0; w < VW; ++w)
          acc[c][w] = fma(l0, sH[((size_t)(w * p.rows + row) * q + sel(a1)) * q + sel(a2)], acc[c][w]);
      }
    }
    __syncthreads();  // the next chunk overwrites sL0, sL1 and sG
  }
#pragma unroll
  for (int c = 0; c < kDtAcc; ++c) {
    const int i = tid + c * kDtThreads;
    if (i < ne)
#pragma unroll
      for (int w = 0; w < VW; ++w)
        out[i * VW + w] = (refused >> c) & 1 ? __builtin_nan("") : acc[c][w];
  }
}

__global__ void __launch_bounds__(256) duffy_tensor_fill_kernel(int64_t n, double* __restrict__ part) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) part[i] = __builtin_nan("");
}

__global__ void __launch_bounds__(256)
    duffy_tensor_sum_kernel(int64_t n, const double* __restrict__ part, double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
#pragma unroll
  for (int b = 0; b < 8; ++b) s += part[b * n + i];
  out[i] = s;
}

template <int KIND, int Q>
static hipError_t launch_tensor_q(DuffyTensorParams p, int64_t max_entries, double* out,
                                  hipStream_t s) {
  constexpr int vw = kind_is_complex(KIND) ? 2 : 1;
  // rows of a chunk: 256 pairs, within LDS
  p.rows = std::max(1, kDtThreads / p.n_tail);
  p.rows = std::min(p.rows, 6 * p.n_rho);
  p.pitch = kDtThreads + 1;
  auto bytes = [&]() {
    return sizeof(double) * ((size_t)(1 + vw) * p.q * p.pitch + (size_t)p.rows * p.q +
                             (size_t)vw * p.rows * p.q * p.q);
  };
  while (bytes() > 150 * 1024 && p.rows > 1) --p.rows;
  const size_t lds = bytes();
  auto fn = duffy_tensor_kernel<KIND, Q>;
  hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     160 * 1024);
  if (e != hipSuccess) return e;
  const int64_t per = kDtThreads * kDtAcc, n = p.n_entries * vw;
  const dim3 flat((unsigned)((n + 255) / 256));
  hipLaunchKernelGGL(duffy_tensor_fill_kernel, flat, dim3(256), 0, s, n, p.part);  // first sign block
  hipLaunchKernelGGL(fn, dim3((unsigned)p.n_targets, 8, (unsigned)((max_entries + per - 1) / per)),
                     dim3(kDtThreads), lds, s, p);
  hipLaunchKernelGGL(duffy_tensor_sum_kernel, flat, dim3(256), 0, s, n, p.part, out);
  return hipGetLastError();
}

template <int KIND>
static hipError_t launch_tensor(const DuffyTensorParams& p, int64_t max_entries, double* out,
                                hipStream_t s) {
  switch (p.q) {
    case 2: return launch_tensor_q<KIND, 2>(p, max_entries, out, s);
    case 3: return launch_tensor_q<KIND, 3>(p, max_entries, out, s);
    case 4: return launch_tensor_q<KIND, 4>(p, max_entries, out, s);
    case 5: return launch_tensor_q<KIND, 5>(p, max_entries, out, s);
    case 6: return launch_tensor_q<KIND, 6>(p, max_entries, out, s);
    case 8: return launch_tensor_q<KIND, 8>(p, max_entries, out, s);
    default: return launch_tensor_q<KIND, 0>(p, max_entries, out, s);
  }
}

}  // namespace vl1

using namespace vl1;

extern "C" int vl1_duffy_build_tensor(const vl1_duffy_tensor_args* a, void* stream) {
  clear_error();
  if (!a) return fail(VL1_E_ARG, "vl1_duffy_build_tensor: null argument");
  if (a->dim != 3) return fail(VL1_E_UNSUPPORTED, "vl1_duffy_build_tensor: dim must be 3");
  if (a->quad_order < 1 || a->quad_order > 16)
    return fail(VL1_E_ARG, "vl1_duffy_build_tensor: quad_order");
  if (a->n_targets < 0 || a->n_entries < 0 || a->max_entries < 0 || a->n_radial < 1 || a->n_tail < 1)
    return fail(VL1_E_ARG, "vl1_duffy_build_tensor: bad counts");
  if (a->n_tail > kDtThreads)
    return fail(VL1_E_UNSUPPORTED, "vl1_duffy_build_tensor: more than 256 tail nodes");
  if (a->n_targets > INT32_MAX || a->n_entries > (int64_t)INT32_MAX || a->n_radial > (1 << 24))
    return fail(VL1_E_UNSUPPORTED, "vl1_duffy_build_tensor: too many entries");
  if (!(a->source_box_extent > 0))
    return fail(VL1_E_ARG, "vl1_duffy_build_tensor: extent must be > 0");
  if (a->n_targets == 0 || a->n_entries == 0) return VL1_OK;
  if (!a->target_points || !a->entry_start || !a->modes || !a->radial_x || !a->radial_w ||
      !a->tail_x || !a->tail_w || !a->interp_nodes || !a->work || !a->result)
    return fail(VL1_E_ARG, "vl1_duffy_build_tensor: null device array");
  const bool deriv = kind_is_deriv(a->kernel_kind);
  if (deriv && (a->deriv_axis < 0 || a->deriv_axis >= a->dim))
    return fail(VL1_E_ARG, "vl1_duffy_build_tensor: derivative axis out of range");
  const bool radial = a->kernel_kind == VL1_KERNEL_POWER || a->kernel_kind == VL1_KERNEL_POWER_LOG ||
                      kind_is_power_deriv(a->kernel_kind);
  const bool needs_pos = a->kernel_kind != VL1_KERNEL_POWER;
  if (radial && (a->power < 0 || a->power > 32 || (needs_pos && a->power == 0)))
    return fail(VL1_E_ARG,
                "vl1_duffy_build_tensor: power must be 0..32 (1..32 with the log or a derivative)");
  DuffyTensorParams p{a->quad_order, deriv ? a->deriv_axis : -1, a->n_radial, a->n_tail, 0, 0,
                      radial ? (double)a->power : a->helmholtz_k, a->source_box_extent,
                      a->n_targets, a->n_entries, a->target_points, a->entry_start, a->modes,
                      a->radial_x, a->radial_w, a->tail_x, a->tail_w, a->interp_nodes, a->work};
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = hipErrorInvalidValue;
  switch (a->kernel_kind) {
#define VL1_DT_KIND(K) \
  case K: e = launch_tensor<K>(p, a->max_entries, a->result, s); break;
    VL1_DT_KIND(VL1_KERNEL_CONSTANT)
    VL1_DT_KIND(VL1_KERNEL_LAPLACE)
    VL1_DT_KIND(VL1_KERNEL_HELMHOLTZ)
    VL1_DT_KIND(VL1_KERNEL_LAPLACE_TARGET_DERIV)
    VL1_DT_KIND(VL1_KERNEL_LAPLACE_SOURCE_DERIV)
    VL1_DT_KIND(VL1_KERNEL_HELMHOLTZ_TARGET_DERIV)
    VL1_DT_KIND(VL1_KERNEL_HELMHOLTZ_SOURCE_DERIV)
    VL1_DT_KIND(VL1_KERNEL_POWER)
    VL1_DT_KIND(VL1_KERNEL_POWER_LOG)
    VL1_DT_KIND(VL1_KERNEL_POWER_TARGET_DERIV)
    VL1_DT_KIND(VL1_KERNEL_POWER_SOURCE_DERIV)
    VL1_DT_KIND(VL1_KERNEL_POWER_LOG_TARGET_DERIV)
    VL1_DT_KIND(VL1_KERNEL_POWER_LOG_SOURCE_DERIV)
#undef VL1_DT_KIND
    default: return fail(VL1_E_UNSUPPORTED, "vl1_duffy_build_tensor: kernel kind");
  }
  if (e != hipSuccess)
    return fail(VL1_E_HIP, std::string("duffy tensor launch: ") + hipGetErrorString(e));
  return VL1_OK;
}
