// Plain FP64 list-1 evaluation with the reference's general CSR semantics.
//
// Semantics follow the loopy `near_field` kernel of
// volumential/list1.py:1057-1148: for every target box of `target_boxes`
// (CSR order) and every target particle `tid` of the box,
//   result[tbeg + tid] = sum_{sbox in list1} sum_{sid}
//       coef[sbeg + sid] * (T[lev, row(case, s, t)] * scaling + displacement)
// with case = case_indices[int(sum_d ((c_t - c_s)/h_s*4 + shift + bias) base^k + 0.5)]
// (list1.py:439-459, 1083-1091), s/t the box-local mode ids of the particles,
// and the scaling/level policy of list1.py:361-437.
//
// GPU mapping: one workgroup per target box, taken in CSR order.  For every
// source box the densities of up to RC right-hand sides are staged in LDS;
// each lane owns one target node and walks the source modes.  The table
// values come from the payload's expanded per-(level, case) blocks
// D[s][t] (built once, on the first plain evaluation, while they stay
// under 8 GiB): one coalesced line per source mode.  Beyond that size the
// canonical orbit block is staged in LDS when it fits and gathered through
// the per-case row map.  For boxes with fewer than 256 nodes the lanes are
// split into P parts over the source modes and reduced through LDS at the
// end ("wavefront reduction over list-1 sources").
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <string>

#include <type_traits>

#include "internal.h"

namespace vl1 {

struct NFParams {
  // custom scaling and displacement factor per source level [VL1_MAX_LEVELS]
  // (device); first in the struct: further down, the ROCm 7.2 compiler
  // fails on the VALU kernel's load of them ("illegal instruction")
  const double* lsc;
  const double* ldisp;
  const double* centers;
  int nboxes;
  const uint8_t* levels;
  const int32_t* src_counts;
  const int32_t* src_starts;
  const int32_t* tgt_counts;
  const int32_t* tgt_starts;
  const int32_t* nbr_starts;
  const int32_t* nbr_lists;
  const int32_t* target_boxes;
  const int32_t* src_ids;
  const int32_t* tgt_ids;
  const int64_t* case_indices;
  int n_codes;
  const uint16_t* ranks;
  const int32_t* offs;
  const double* table;
  int64_t n_entries;
  int n_tables;
  const double* nmlz;
  const void* rowmap;
  const double* dense;  // expanded table (DENSE kernels), [n_tables][n_cases][n][n] (x VW)
  int n_cases;
  int dim, n;
  int scaling_mode, scaling_power, log_disp;
  double root_extent, table_root_extent;
  int table_starting_level;
  double enc_shift, enc_bias;
  int enc_base;
  int n_rhs;
  int64_t ldf, ldy;
  const double* f;
  double* y;
  int32_t* err;
  int tbuf;   // doubles of LDS for the staged orbit block
  int nt;     // lanes per target set (power of two)
};

constexpr int kNFBlock = 256;

// CPLX: complex table, densities and result (interleaved re, im doubles;
// leading dimensions in doubles); products are complex, the scaling real.
// DENSE: table values read from the expanded per-(level, case) blocks,
// [s][t] with t fastest, so the lanes of a wave (consecutive target nodes)
// read one coalesced line per source mode instead of a row-map load plus an
// LDS gather; no orbit block is staged.
template <typename IdxT, int RC, bool CPLX, bool DENSE>
__global__ void __launch_bounds__(kNFBlock) near_field_f64_kernel(const NFParams p) {
  extern __shared__ double smem[];
  constexpr int VW = CPLX ? 2 : 1;  // doubles per value
  const int n = p.n;
  const int P = kNFBlock / p.nt;
  double* sT = smem;
  double* sF = sT + p.tbuf;
  double* sD = sF + (size_t)n * RC * VW;
  double* red = sD + n;
  int* sMode = (int*)(red + (P > 1 ? kNFBlock * RC * VW : 0));

  const int tid = threadIdx.x;
  const int lane_t = tid % p.nt;
  const int part = tid / p.nt;

  const int tbox = blockIdx.x;
  const int tb = p.target_boxes[tbox];
  const int tbeg = p.tgt_starts[tb];
  const int ntb = min(p.tgt_counts[tb], n);
  const int l0 = p.nbr_starts[tbox];
  const int l1 = p.nbr_starts[tbox + 1];
  double ct[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < p.dim; ++d) ct[d] = p.centers[(int64_t)d * p.nboxes + tb];

  for (int r0 = 0; r0 < p.n_rhs; r0 += RC) {
    const int rc = min(RC, p.n_rhs - r0);
    for (int t0 = 0; t0 < ntb; t0 += p.nt) {
      const int ti = t0 + lane_t;
      const int tm_raw = ti < ntb ? p.tgt_ids[tbeg + ti] : -1;
      const bool tact = (unsigned)tm_raw < (unsigned)n;
      const int tmode = tact ? tm_raw : 0;
      double acc[RC], aci[RC];  // aci: imaginary parts (complex data only)
#pragma unroll
      for (int r = 0; r < RC; ++r) acc[r] = aci[r] = 0.0;

      for (int li = l0; li < l1; ++li) {
        const int sb = p.nbr_lists[li];
        const int lvl = p.levels[sb];
        const double sext = p.root_extent * (1.0 / (double)(1 << lvl));
        double code = 0.0;
        for (int d = 0; d < p.dim; ++d) {
          const double cs = p.centers[(int64_t)d * p.nboxes + sb];
          code = code * (double)p.enc_base + ((ct[d] - cs) / sext * 4.0 + p.enc_shift + p.enc_bias);
        }
        const int64_t vid = (int64_t)(code + 0.5);
        const int cid = (vid >= 0 && vid < p.n_codes) ? (int)p.case_indices[vid] : -1;
        __syncthreads();  // previous source box done with LDS
        if (cid < 0) {    // uniform over the workgroup
          if (tid == 0 && p.err) atomicOr(p.err, 1);
          continue;
        }
        int tlev = 0;
        double scal = 1.0, dscale = 0.0;
        if (p.scaling_mode == VL1_SCALING_CANONICAL) {
          double num = 1.0, den = 1.0;
          for (int k = 0; k < p.scaling_power; ++k) {
            num *= sext;
            den *= p.table_root_extent;
          }
          scal = num / den;
          if (p.log_disp) dscale = -0.5 / M_PI * scal * log(sext / p.table_root_extent);
        } else if (p.scaling_mode == VL1_SCALING_CUSTOM) {
          scal = p.lsc[min(lvl, VL1_MAX_LEVELS - 1)];
          dscale = p.ldisp[min(lvl, VL1_MAX_LEVELS - 1)];
        } else if (p.scaling_mode == VL1_SCALING_PER_LEVEL) {
          const int rel = lvl - p.table_starting_level;
          tlev = lvl < p.table_starting_level ? 0 : (rel < p.n_tables ? rel : p.n_tables - 1);
        }
        int off = 0, cnt = 0;  // the case's canonical orbit (row-map kernels only)
        if constexpr (!DENSE) {
          const int rank = p.ranks[cid];
          off = p.offs[rank];
          cnt = p.offs[rank + 1] - off;
        }
        const double* gT = p.table + ((int64_t)tlev * p.n_entries + off) * VW;
        const bool staged = !DENSE && cnt * VW <= p.tbuf;
        const double* gD =
            DENSE ? p.dense + (((int64_t)tlev * p.n_cases + cid) * n * n + tmode) * VW : nullptr;
        const int sbeg = p.src_starts[sb];
        const int ns = min(p.src_counts[sb], n);
        if (staged)
          for (int i = tid; i < cnt * VW; i += kNFBlock) sT[i] = gT[i];
        for (int i = tid; i < ns * RC * VW; i += kNFBlock) {
          const int c = i % VW, rs = i / VW;
          const int r = rs / ns, sid = rs % ns;
          sF[(sid * RC + r) * VW + c] =
              r < rc ? p.f[(int64_t)(r0 + r) * p.ldf + (int64_t)(sbeg + sid) * VW + c] : 0.0;
        }
        for (int i = tid; i < ns; i += kNFBlock) {
          sMode[i] = p.src_ids[sbeg + i];
          sD[i] = p.log_disp ? dscale * p.nmlz[(int64_t)tlev * n + i] : 0.0;
        }
        __syncthreads();
        if (tact) {
          const IdxT* rm = static_cast<const IdxT*>(p.rowmap) + (int64_t)cid * n * n + tmode;
          for (int sid = part; sid < ns; sid += P) {
            const int s = sMode[sid];
            if ((unsigned)s >= (unsigned)n) continue;  // malformed mode id: no contribution
            double tr, ti;  // table value (imaginary part for complex data)
            double esc = scal;  // scaling times the entry sign of signed kernels
            if constexpr (DENSE) {
              tr = gD[(int64_t)s * n * VW];
              ti = CPLX ? gD[(int64_t)s * n * VW + 1] : 0.0;
              // dense kind: no entry (NaN) -> no contribution, displacement
              // included (list1.py:1111-1116)
              if (tr != tr) continue;
            } else {
              int rel = (int)rm[(int64_t)s * n];
              if constexpr (std::is_signed<IdxT>::value) {
                double sg;
                rel = decode_signed_row(rel, sg);
                esc *= sg;
              }
              tr = staged ? sT[rel * VW] : gT[rel * VW];
              ti = CPLX ? (staged ? sT[rel * VW + 1] : gT[rel * VW + 1]) : 0.0;
            }
            const double* fs = sF + sid * RC * VW;
            if constexpr (!CPLX) {
              const double v = tr * esc + sD[sid];
#pragma unroll
              for (int r = 0; r < RC; ++r) acc[r] = fma(fs[r], v, acc[r]);
            } else {
              const double vr = tr * esc;
              const double vi = ti * esc;
#pragma unroll
              for (int r = 0; r < RC; ++r) {
                const double fr = fs[2 * r], fi = fs[2 * r + 1];
                acc[r] = fma(fr, vr, fma(-fi, vi, acc[r]));
                aci[r] = fma(fr, vi, fma(fi, vr, aci[r]));
              }
            }
          }
        }
      }

      if (P > 1) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          red[((part * p.nt + lane_t) * RC + r) * VW] = acc[r];
          if (CPLX) red[((part * p.nt + lane_t) * RC + r) * VW + 1] = aci[r];
        }
        __syncthreads();
        if (part == 0) {
          for (int j = 1; j < P; ++j)
#pragma unroll
            for (int r = 0; r < RC; ++r) {
              acc[r] += red[((j * p.nt + lane_t) * RC + r) * VW];
              if (CPLX) aci[r] += red[((j * p.nt + lane_t) * RC + r) * VW + 1];
            }
        }
      }
      if (part == 0 && tact) {
        for (int r = 0; r < rc; ++r) {
          p.y[(int64_t)(r0 + r) * p.ldy + (int64_t)(tbeg + ti) * VW] = acc[r];
          if (CPLX) p.y[(int64_t)(r0 + r) * p.ldy + (int64_t)(tbeg + ti) * VW + 1] = aci[r];
        }
      }
      __syncthreads();
    }
  }
}

// ------------------------------------------------------------------------
// FP64-MFMA form of the same evaluation (real tables, boxes of at most 256
// nodes): per target box and group of 16 NC densities, every list-1 pair is a
// product Y[tid][r] += sum_sid A[tid][sid] X[sid][r] with
//   A[tid][sid] = D[lev][case][mode(sid)][mode(tid)]  (expanded blocks),
//   X[sid][r]   = scaling * f[r][sbeg + sid],
// rows indexed by the target particles and K by the source particles of
// the pair, so ragged boxes, permuted, repeated or invalid mode ids keep the
// semantics of the scalar kernel above: an invalid id (or a missing entry,
// NaN in the expanded blocks) gives A = 0.  v_mfma_f64_16x16x4f64 tiles:
// wave w owns row tiles w, w + 8 (16 rows each) and all NC 16-column tiles
// (1, 2 or 4, by the densities: see launch_nf_mfma).  K advances in chunks of KC source
// particles; a chunk's densities go through a two-slot LDS ring and its table
// fragments through registers, both loaded one chunk ahead, and a pair's source
// modes two pairs ahead.  Pair descriptors (a chain of four dependent loads
// each) are made 64 at a time, one per thread.  The 2D log displacement is the
// same for every target of a pair: sum_sid nmlz[sid] f[sid], accumulated in
// LDS while the densities are staged and added when the pair ends (only
// used where no entry is missing: the scalar kernel drops the displacement
// of a missing entry, list1.py:1111-1116).
// Bound: the FP64 matrix pipe.  3D q = 4, 4096 boxes, 16 densities (1.3e10
// flop): 1752 us with 64 columns whatever the densities and each descriptor
// made by all threads when its pair began; 404 us so (32 TFLOP/s: the pipe is
// busy 45% of the time, the rest goes to the loads' issue and the sums' chain).
constexpr int kNFPairs = 64;  // pair descriptors made at a time
constexpr int kNFMaxK = 256;  // source particles per box in the MFMA form

typedef __attribute__((ext_vector_type(4))) double nf_doublex4;

struct NFPair {
  int sbeg, ns;
  int64_t dbase;  // first value of the pair's expanded block
  double scal, dscale;
  int tlev;
  bool ok;
};

__device__ inline NFPair nf_pair(const NFParams& p, int li, const double (&ct)[3]) {
  NFPair d;
  const int sb = p.nbr_lists[li];
  const int lvl = p.levels[sb];
  const double sext = p.root_extent * (1.0 / (double)(1 << lvl));
  double code = 0.0;
  for (int k = 0; k < p.dim; ++k) {
    const double cs = p.centers[(int64_t)k * p.nboxes + sb];
    code = code * (double)p.enc_base + ((ct[k] - cs) / sext * 4.0 + p.enc_shift + p.enc_bias);
  }
  const int64_t vid = (int64_t)(code + 0.5);
  const int cid = (vid >= 0 && vid < p.n_codes) ? (int)p.case_indices[vid] : -1;
  d.ok = cid >= 0;
  d.tlev = 0;
  d.scal = 1.0;
  d.dscale = 0.0;
  if (p.scaling_mode == VL1_SCALING_CANONICAL) {
    double num = 1.0, den = 1.0;
    for (int k = 0; k < p.scaling_power; ++k) {
      num *= sext;
      den *= p.table_root_extent;
    }
    d.scal = num / den;
    if (p.log_disp) d.dscale = -0.5 / M_PI * d.scal * log(sext / p.table_root_extent);
  } else if (p.scaling_mode == VL1_SCALING_CUSTOM) {
    d.scal = p.lsc[min(lvl, VL1_MAX_LEVELS - 1)];
    d.dscale = p.ldisp[min(lvl, VL1_MAX_LEVELS - 1)];
  } else if (p.scaling_mode == VL1_SCALING_PER_LEVEL) {
    const int rel = lvl - p.table_starting_level;
    d.tlev = lvl < p.table_starting_level ? 0 : (rel < p.n_tables ? rel : p.n_tables - 1);
  }
  d.dbase = d.ok ? ((int64_t)d.tlev * p.n_cases + cid) * p.n * p.n : 0;
  d.sbeg = p.src_starts[sb];
  d.ns = min(p.src_counts[sb], p.n);
  if (!d.ok) d.ns = 0;
  return d;
}

template <int W, int NRT, int NC, int KC>
__global__ void __launch_bounds__(64 * W, NC * NRT == 1 ? 4 : 1)
near_field_mfma_kernel(const NFParams p, int KP, int n_tgt_boxes, int finite) {
  constexpr int T = 64 * W, COLS = 16 * NC, KU = KC / 4;
  constexpr int VPT = KC * COLS / T;  // densities of a chunk per thread
  constexpr int PITCH = KC + 2;       // doubles per column of a staged chunk
  __shared__ __align__(16) double sX[2][COLS * PITCH];
  __shared__ NFPair sPair[2][kNFPairs];
  constexpr int KMAX = (16 * W * NRT + 31) / 32 * 32;  // KP at most
  __shared__ __align__(16) int sRow[3][KMAX];  // table row of a source particle, in bytes
  __shared__ bool sOk[3][KMAX];                // whether it has one
  __shared__ double sDisp[3][COLS];

  const int n = p.n;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int l16 = lane % 16, lg = lane / 16;
  // neighbouring boxes on one XCD (workgroup i runs on XCD i % 8): their
  // sources meet in its L2
  const int per = (n_tgt_boxes + 7) / 8;
  const int tbox = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (tbox >= n_tgt_boxes) return;  // uniform over the workgroup
  const int r0 = blockIdx.y * COLS;
  const int rc = min(COLS, p.n_rhs - r0);
  const int tb = p.target_boxes[tbox];
  const int tbeg = p.tgt_starts[tb];
  const int ntb = min(p.tgt_counts[tb], n);
  const int l0 = p.nbr_starts[tbox];
  const int npairs = p.nbr_starts[tbox + 1] - l0;
  const int nkc = KP / KC;  // KP: a multiple of KC
  double ct[3] = {0.0, 0.0, 0.0};
  for (int k = 0; k < p.dim; ++k) ct[k] = p.centers[(int64_t)k * p.nboxes + tb];

  // whether this wave's second row tile holds any of the box's targets
  const bool rows_rt1 = NRT > 1 && 16 * (wave + W) < ntb;
  // this lane's A rows (target particles) and their modes (-1: no row)
  int tmA[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
    const int row = 16 * (wave + W * rt) + l16;
    const int m = row < ntb ? p.tgt_ids[tbeg + row] : -1;
    tmA[rt] = (unsigned)m < (unsigned)n ? m : -1;
  }

  // descriptors of pairs [64 blk, 64 blk + 64)
  auto make_pairs = [&](int blk) {
    const int k = blk * kNFPairs + tid;
    if (tid < kNFPairs && k < npairs) {
      const NFPair d = nf_pair(p, l0 + k, ct);
      if (!d.ok && p.err) atomicOr(p.err, 1);
      sPair[blk & 1][tid] = d;
    }
  };
  auto pair = [&](int k) -> const NFPair& { return sPair[(k / kNFPairs) & 1][k % kNFPairs]; };
  // pair k's source modes (-1 past the box or invalid: a zero density and any
  // row); its displacement sums start at zero
  auto mode_of = [&](int k) {
    if (k >= npairs || tid >= KP) return -1;
    const NFPair& d = pair(k);
    const int m = tid < d.ns ? p.src_ids[d.sbeg + tid] : -1;
    return (unsigned)m < (unsigned)n ? m : -1;
  };
  auto put_mode = [&](int k, int m) {
    if (tid < KP) {
      sRow[k % 3][tid] = 8 * n * max(m, 0);
      sOk[k % 3][tid] = m >= 0;
    }
    if (tid < COLS) sDisp[k % 3][tid] = 0.0;
  };
  // densities of chunk kc of a pair: thread value v is column xcol + v T / KC,
  // source particle KC kc + xk (consecutive threads read consecutive particles
  // of one density); loads past the box or the densities read a valid one
  static_assert(T % KC == 0, "a thread keeps one particle of the chunk");
  const int xk = tid % KC, xcol = tid / KC;
  int64_t xoff[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) xoff[v] = (int64_t)min(xcol + v * (T / KC), rc - 1) * p.ldf;
  auto load_x = [&](const NFPair& d, int kc, double (&x)[VPT]) {
    const int ns = __builtin_amdgcn_readfirstlane(d.ns);
    const double* f = p.f + (int64_t)r0 * p.ldf + __builtin_amdgcn_readfirstlane(d.sbeg);
    if (ns > 0) {
      const int sid = min(KC * kc + xk, ns - 1);
#pragma unroll
      for (int v = 0; v < VPT; ++v) x[v] = f[xoff[v] + sid];
    }
  };
  auto store_x = [&](const NFPair& d, int kc, int k, int ring, const double (&x)[VPT]) {
    const int slot = k % 3, sid = KC * kc + xk;
    const bool live = sOk[slot][sid];
    const double scal = d.scal;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      const int col = xcol + v * (T / KC);
      sX[ring][col * PITCH + xk] = live ? scal * x[v] : 0.0;
      if (p.log_disp && live && x[v] != 0.0)
        atomicAdd(&sDisp[slot][col], p.nmlz[(int64_t)d.tlev * n + sid] * x[v]);
    }
  };
  // table fragments of chunk kc: lane (l16, lg) of k group u holds
  // A[row 16 rt16 + l16][sid KC kc + KU lg + u] (a lane's particles adjacent, so
  // that their rows and densities come in 16-byte LDS reads).  A row without a
  // target reads another's entries: its sums go nowhere.
  int rowA[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) rowA[rt] = 8 * max(tmA[rt], 0);
  double ac[NRT][KU];
  auto base_of = [&](const NFPair& d) {
    const int lo = __builtin_amdgcn_readfirstlane((int)(unsigned)d.dbase);
    const int hi = __builtin_amdgcn_readfirstlane((int)(d.dbase >> 32));
    return reinterpret_cast<const char*>(p.dense + ((int64_t)hi << 32 | (unsigned)lo));
  };
  typedef __attribute__((ext_vector_type(4))) int int4_t;
  typedef __attribute__((ext_vector_type(2))) double double2_t;
  // the lane's particles 4 g .. 4 g + 3 of chunk kc
  auto rows_of = [&](int kc, int k, int g) {
    return *reinterpret_cast<const int4_t*>(&sRow[k % 3][KC * kc + KU * lg + 4 * g]);
  };
  auto load_a = [&](const char* D, int row, int u) {
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
      ac[rt][u] = *reinterpret_cast<const double*>(D + (unsigned)(row + rowA[rt]));
  };

  nf_doublex4 yacc[NRT][NC];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c) yacc[rt][c] = nf_doublex4{0.0, 0.0, 0.0, 0.0};

  double x[VPT] = {};
  const int total = npairs * nkc;
  if (total > 0) {
    make_pairs(0);
    make_pairs(1);
    __syncthreads();
    put_mode(0, mode_of(0));
    put_mode(1, mode_of(1));
    __syncthreads();
    load_x(pair(0), 0, x);
    const char* D = base_of(pair(0));
#pragma unroll
    for (int u = 0; u < KU; ++u) load_a(D, rows_of(0, 0, u / 4)[u % 4], u);
    store_x(pair(0), 0, 0, 0, x);
  }
  __syncthreads();

  for (int it = 0, k = 0, kc = 0; it < total; ++it) {
    const bool has_next = it + 1 < total;
    const bool pair_end = kc + 1 == nkc;
    // the chunk to load: the next one, or this one again after the last
    const int kn = pair_end && has_next ? k + 1 : k, kcn = !has_next ? kc : (pair_end ? 0 : kc + 1);
    int m2 = -1;
    if (kc == 0) {
      // the block after the one entered, into the slot of the one left
      if (k > 0 && k % kNFPairs == 0) make_pairs(k / kNFPairs + 1);
      m2 = mode_of(k + 2);
    }
    load_x(pair(kn), kcn, x);
    const char* Dn = base_of(pair(kn));
    const double* rX = &sX[it & 1][l16 * PITCH + KU * lg];
    auto mul = [&](auto finite) {
#pragma unroll
      for (int g = 0; g < KU / 4; ++g) {
        const int4_t rows = rows_of(kcn, kn, g);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int u = 4 * g + h;
          double bx[NC];
#pragma unroll
          for (int c = 0; c < NC; ++c)
            bx[c] = (*reinterpret_cast<const double2_t*>(rX + 16 * c * PITCH + (u & ~1)))[u & 1];
          bool ok = true;
          if constexpr (!decltype(finite)::value) ok = sOk[k % 3][KC * kc + KU * lg + u];
#pragma unroll
          for (int rt = 0; rt < NRT; ++rt)
            if (rt == 0 || rows_rt1) {  // a second row tile past the box's targets is skipped
              double a = ac[rt][u];
              if constexpr (!decltype(finite)::value) a = ok && a == a ? a : 0.0;  // NaN: no entry
#pragma unroll
              for (int c = 0; c < NC; ++c)
                yacc[rt][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bx[c], yacc[rt][c], 0, 0, 0);
            }
          load_a(Dn, rows[h], u);  // in place: a chunk ahead
        }
        // (else all groups' LDS reads move up and their registers spill)
        if constexpr (NRT * NC >= 4) __builtin_amdgcn_sched_barrier(0);
      }
    };
    // a finite table needs no look at its entries: the densities are zero
    // where no source is
    if (finite) mul(std::true_type{});
    else mul(std::false_type{});
    if (pair_end && p.log_disp) {
      const double dscale = pair(k).dscale;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const double ds = dscale * sDisp[k % 3][16 * c + l16];
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
          for (int e = 0; e < 4; ++e) yacc[rt][c][e] += ds;
      }
    }
    if (kc == 0) put_mode(k + 2, m2);
    if (has_next) store_x(pair(kn), kcn, kn, (it + 1) & 1, x);
    __syncthreads();
    k = kn;
    kc = kcn;
  }

  // outputs: lane holds rows 16 rt16 + lg + 4 e, column 16 c + l16
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * (wave + W * rt) + lg + 4 * e;
      if (row >= ntb) continue;
      const int m = p.tgt_ids[tbeg + row];
      if ((unsigned)m >= (unsigned)n) continue;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int col = 16 * c + l16;
        if (col < rc) p.y[(int64_t)(r0 + col) * p.ldy + tbeg + row] = yacc[rt][c][e];
      }
    }
  }
}

// Expanded table for the DENSE kernels: D[lev][case][s][t] = sign * T[lev,
// row(case, s, t)], read through the payload's row map.
template <typename IdxT>
__global__ void __launch_bounds__(256)
dense_table_kernel(int n, int n_cases, int n_tables, int vw, const IdxT* __restrict__ rowmap,
                   const uint16_t* __restrict__ ranks, const int32_t* __restrict__ offs,
                   const double* __restrict__ table, int64_t n_entries, double* __restrict__ D,
                   int* __restrict__ not_finite) {
  const int64_t nn = (int64_t)n * n;
  const int64_t total = (int64_t)n_tables * n_cases * nn;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t cst = i % ((int64_t)n_cases * nn);
    const int lev = (int)(i / ((int64_t)n_cases * nn));
    const int c = (int)(cst / nn);
    int rel = (int)rowmap[cst];
    double sg = 1.0;
    if constexpr (std::is_signed<IdxT>::value) rel = decode_signed_row(rel, sg);
    const double* T = table + ((int64_t)lev * n_entries + offs[ranks[c]] + rel) * vw;
    D[i * vw] = sg * T[0];
    if (vw == 2) D[i * vw + 1] = sg * T[1];
    if (!isfinite(T[0])) atomicOr(not_finite, 1);
  }
}

// Build the payload's expanded table once (first plain evaluation).
static hipError_t ensure_dense(const vl1_payload* pl, hipStream_t s) {
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  if (pl->dense.bytes) return hipSuccess;
  const int vw = pl->is_complex ? 2 : 1;
  const int64_t total = (int64_t)pl->n_tables * pl->n_cases * pl->n * pl->n;
  hipError_t e = pl->dense.alloc((size_t)total * vw * sizeof(double));
  if (e != hipSuccess) return e;
  DevBuf flag;  // an entry is not finite
  int not_finite = 0;
  e = upload(flag, &not_finite, sizeof(int), s);
  if (e != hipSuccess) {
    pl->dense.release();
    return e;
  }
  const int grid = (int)std::min<int64_t>((total + 255) / 256, 65536);
  if (pl->rowmap_u16)
    hipLaunchKernelGGL(dense_table_kernel<uint16_t>, dim3(grid), dim3(256), 0, s, pl->n,
                       pl->n_cases, pl->n_tables, vw, pl->rowmap.as<uint16_t>(),
                       pl->ranks.as<uint16_t>(), pl->offs.as<int32_t>(), pl->table.as<double>(),
                       pl->n_entries, pl->dense.as<double>(), flag.as<int>());
  else
    hipLaunchKernelGGL(dense_table_kernel<int32_t>, dim3(grid), dim3(256), 0, s, pl->n,
                       pl->n_cases, pl->n_tables, vw, pl->rowmap.as<int32_t>(),
                       pl->ranks.as<uint16_t>(), pl->offs.as<int32_t>(), pl->table.as<double>(),
                       pl->n_entries, pl->dense.as<double>(), flag.as<int>());
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&not_finite, flag.ptr, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) pl->dense.release();
  else pl->dense_finite = !not_finite;
  return e;
}

// Column tiles per workgroup: the split of the densities with the least work,
// columns past the last density included.  A wider tile reads each table
// fragment less often; 16 densities cost, against wider tiles per 16 columns
// (us, uniform trees): 3D q = 5, 512 boxes 207, 180 (2 tiles), 160 (4); 3D q =
// 4, 4096 boxes 404, 397, 368; 2D q = 4, 4096 boxes 91, 90, 125 (registers of
// its single wave: boxes of up to two waves take one tile).
// Chunks of 64 source particles where they divide the box and the columns are
// few (the registers of four column tiles leave room for 32).
template <int W, int NRT>
static void launch_nf_mfma(const NFParams& prm, int KP, int n_tgt_boxes, int finite,
                           hipStream_t s) {
  const int t16 = (prm.n_rhs + 15) / 16;
  int nc = 1;
  if (W >= 4) {
    const double c2 = W >= 8 ? 1.75 : 1.97, c4 = W >= 8 ? 3.1 : 3.65;
    const double cost1 = t16, cost2 = (t16 + 1) / 2 * c2, cost4 = (t16 + 3) / 4 * c4;
    nc = cost4 <= cost1 && cost4 <= cost2 ? 4 : (cost2 <= cost1 ? 2 : 1);
  }
  const dim3 grid((n_tgt_boxes + 7) / 8 * 8, (t16 + nc - 1) / nc);
  auto go = [&](auto ncc, auto kcc) {
    hipLaunchKernelGGL((near_field_mfma_kernel<W, NRT, decltype(ncc)::value, decltype(kcc)::value>),
                       grid, dim3(64 * W), 0, s, prm, KP, n_tgt_boxes, finite);
  };
  constexpr std::integral_constant<int, 1> n1{};
  constexpr std::integral_constant<int, 32> k32{};
  if constexpr (W < 4) {
    go(n1, k32);
  } else {
    constexpr std::integral_constant<int, 2> n2{};
    constexpr std::integral_constant<int, 64> k64{};
    const bool wide = KP % 64 == 0;
    if (nc == 1) wide ? go(n1, k64) : go(n1, k32);
    else if (nc == 2) wide ? go(n2, k64) : go(n2, k32);
    else go(std::integral_constant<int, 4>{}, k32);
  }
}

template <typename IdxT, int RC, bool CPLX, bool DENSE>
static hipError_t launch_nf(const NFParams& prm, int grid, size_t smem, hipStream_t s) {
  auto fn = near_field_f64_kernel<IdxT, RC, CPLX, DENSE>;
  hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(kNFBlock), smem, s, prm);
  return hipGetLastError();
}

}  // namespace vl1

using namespace vl1;

// Potential kind 2 (list1.py:1097-1143): y[t] += f[t] x exterior_nmlz[lev_t][mode_t] x
// the target box's scaling, after the list-1 sums.  One thread per (RHS,
// target box, box-local target); real tables, no displacement.
__global__ void exterior_term_kernel(const NFParams p, const double* __restrict__ ext,
                                     int64_t ld_f, int64_t ld_y, int n_tgt) {
  const int64_t total = (int64_t)p.n_rhs * n_tgt * p.n;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int t = (int)(i % p.n);
    const int tbox = (int)((i / p.n) % n_tgt);
    const int r = (int)(i / ((int64_t)p.n * n_tgt));
    const int tb = p.target_boxes[tbox];
    if (t >= min(p.tgt_counts[tb], p.n)) continue;
    const int lvl = p.levels[tb];
    const double text = p.root_extent * (1.0 / (double)(1 << lvl));
    double scal = 1.0;
    int tlev = 0;
    if (p.scaling_mode == VL1_SCALING_CANONICAL) {
      double num = 1.0, den = 1.0;
      for (int k = 0; k < p.scaling_power; ++k) {
        num *= text;
        den *= p.table_root_extent;
      }
      scal = num / den;
    } else if (p.scaling_mode == VL1_SCALING_CUSTOM) {
      scal = p.lsc[min(lvl, VL1_MAX_LEVELS - 1)];
    } else if (p.scaling_mode == VL1_SCALING_PER_LEVEL) {
      const int rel = lvl - p.table_starting_level;
      tlev = lvl < p.table_starting_level ? 0 : (rel < p.n_tables ? rel : p.n_tables - 1);
    }
    const int64_t pt = (int64_t)p.tgt_starts[tb] + t;
    const double e = ext[(int64_t)tlev * p.n + p.tgt_ids[pt]] * scal;
    p.y[(int64_t)r * ld_y + pt] += p.f[(int64_t)r * ld_f + pt] * e;
  }
}

static int exterior_pass(const NFParams& prm, const vl1_near_field_args* a, hipStream_t s) {
  if (!a->exterior_nmlz) return VL1_OK;
  const int64_t total = (int64_t)a->n_rhs * a->n_tgt_boxes * prm.n;
  const int grid = (int)std::min<int64_t>((total + 255) / 256, 65536);
  hipLaunchKernelGGL(exterior_term_kernel, dim3(grid), dim3(256), 0, s, prm, a->exterior_nmlz,
                     a->n_rhs > 1 ? a->ld_coefs : 0, a->n_rhs > 1 ? a->ld_result : 0,
                     a->n_tgt_boxes);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(VL1_E_HIP, std::string("exterior term launch: ") + hipGetErrorString(e));
  return VL1_OK;
}

extern "C" int vl1_near_field_f64(const vl1_payload* pl, const vl1_near_field_args* a,
                                  void* stream) {
  clear_error();
  if (!pl || !a) return fail(VL1_E_ARG, "vl1_near_field_f64: null argument");
  if (pl->is_complex && a->log_displacement && a->scaling_mode == VL1_SCALING_CANONICAL)
    return fail(VL1_E_UNSUPPORTED, "vl1_near_field_f64: the 2D log displacement applies to real tables");
  if (a->n_tgt_boxes < 0 || a->n_rhs < 1 || a->aligned_nboxes < 1)
    return fail(VL1_E_ARG, "vl1_near_field_f64: bad sizes");
  if (a->scaling_mode < 0 || a->scaling_mode > 3)
    return fail(VL1_E_ARG, "vl1_near_field_f64: bad scaling mode");
  if (a->scaling_mode == VL1_SCALING_CUSTOM && (!a->level_scaling || !a->level_disp))
    return fail(VL1_E_ARG, "vl1_near_field_f64: custom scaling needs level_scaling and level_disp");
  if (a->scaling_mode == VL1_SCALING_CANONICAL && (a->scaling_power < 0 || a->scaling_power > 3))
    return fail(VL1_E_ARG, "vl1_near_field_f64: bad scaling power");
  if (a->n_tgt_boxes == 0) return VL1_OK;
  if (!a->result || !a->mode_coefs || !a->box_centers || !a->box_levels ||
      !a->box_source_counts_nonchild || !a->box_source_starts ||
      !a->box_target_counts_nonchild || !a->box_target_starts ||
      !a->neighbor_source_boxes_starts || !a->neighbor_source_boxes_lists || !a->target_boxes ||
      !a->source_mode_ids || !a->target_point_ids)
    return fail(VL1_E_ARG, "vl1_near_field_f64: null device array");
  if (a->n_rhs > 1 && (a->ld_coefs < 1 || a->ld_result < 1))
    return fail(VL1_E_ARG, "vl1_near_field_f64: bad leading dimension");
  if (a->exterior_nmlz &&
      (pl->is_complex || (a->log_displacement && (a->scaling_mode == VL1_SCALING_CANONICAL ||
                                                  a->scaling_mode == VL1_SCALING_CUSTOM))))
    return fail(VL1_E_UNSUPPORTED,
                "vl1_near_field_f64: potential kind 2 takes real tables without a displacement");

  NFParams prm{};
  prm.centers = a->box_centers;
  prm.nboxes = a->aligned_nboxes;
  prm.levels = a->box_levels;
  prm.src_counts = a->box_source_counts_nonchild;
  prm.src_starts = a->box_source_starts;
  prm.tgt_counts = a->box_target_counts_nonchild;
  prm.tgt_starts = a->box_target_starts;
  prm.nbr_starts = a->neighbor_source_boxes_starts;
  prm.nbr_lists = a->neighbor_source_boxes_lists;
  prm.target_boxes = a->target_boxes;
  prm.src_ids = a->source_mode_ids;
  prm.tgt_ids = a->target_point_ids;
  prm.case_indices = pl->case_idx.as<int64_t>();
  prm.n_codes = (int)pl->case_indices.size();
  prm.ranks = pl->ranks.as<uint16_t>();
  prm.offs = pl->offs.as<int32_t>();
  prm.table = pl->table.as<double>();
  prm.n_entries = pl->n_entries;
  prm.n_tables = pl->n_tables;
  prm.nmlz = pl->nmlz.as<double>();
  prm.rowmap = pl->rowmap.ptr;
  prm.dim = pl->dim;
  prm.n = pl->n;
  prm.scaling_mode = a->scaling_mode;
  prm.scaling_power = a->scaling_power;
  prm.lsc = a->scaling_mode == VL1_SCALING_CUSTOM ? a->level_scaling : nullptr;
  prm.ldisp = a->scaling_mode == VL1_SCALING_CUSTOM ? a->level_disp : nullptr;
  prm.log_disp = a->log_displacement ? 1 : 0;
  if (a->scaling_mode == VL1_SCALING_CUSTOM) {
    // the displacement term is on unless the caller declares it zero
    prm.log_disp = a->log_displacement ? 1 : 0;
    if (prm.log_disp && pl->is_complex)
      return fail(VL1_E_UNSUPPORTED,
                  "vl1_near_field_f64: a custom displacement applies to real tables");
  }
  prm.root_extent = a->root_extent;
  prm.table_root_extent = a->table_root_extent;
  prm.table_starting_level = a->table_starting_level;
  prm.enc_shift = a->encoding_shift;
  prm.enc_bias = a->case_encoding_bias;
  prm.enc_base = a->encoding_base;
  prm.n_rhs = a->n_rhs;
  prm.ldf = a->ld_coefs;
  prm.ldy = a->ld_result;
  prm.f = a->mode_coefs;
  prm.y = a->result;
  prm.err = a->error_flags;
  if (prm.enc_base != 13) return fail(VL1_E_ARG, "encoding_base must be 13");

  int nt = 1;
  while (nt < pl->n && nt < kNFBlock) nt *= 2;
  prm.nt = nt;
  const int P = kNFBlock / nt;
  // densities per pass (32 measured 4.6x slower than 16 on 3D q=6: register
  // pressure)
  const int RC = a->n_rhs == 1 ? 1 : (a->n_rhs <= 4 ? 4 : 16);
  const size_t lds_cap = 150 * 1024;
  const size_t vw = pl->is_complex ? 2 : 1;
  hipStream_t s = (hipStream_t)stream;
  // expanded table: coalesced reads per source mode, no row-map gathers;
  // used while it stays under 8 GiB (a cache of the payload)
  // (VL1_PLAIN_TABLE=gather in the environment selects the row-map path)
  const char* mode_env = std::getenv("VL1_PLAIN_TABLE");
  const bool force_gather = mode_env && std::string(mode_env) == "gather";
  const bool dense = pl->dense_kind ||  // dense-kind payloads hold only the expanded blocks
                     (!force_gather && (double)pl->n_tables * pl->n_cases * pl->n * pl->n * vw *
                                               sizeof(double) <= 8.0 * (1ull << 30));
  if (dense) {
    hipError_t de = ensure_dense(pl, s);
    if (de != hipSuccess)
      return fail(VL1_E_HIP, std::string("vl1_near_field_f64: dense table: ") + hipGetErrorString(de));
    prm.dense = pl->dense.as<double>();
  }
  prm.n_cases = pl->n_cases;
  // FP64-MFMA form: real tables, boxes of at most 256 nodes, 5 or more
  // densities (16 columns are computed whatever the count: at 8 densities, 3D
  // q = 4, 4096 boxes 1417 us on the scalar kernel, 404 here; 2D q = 6 337 and
  // 230; at 4 the scalar kernel takes 162 there), and no missing entry under
  // the log displacement (VL1_PLAIN_KERNEL=scalar selects the scalar kernel
  // below)
  const char* kern_env = std::getenv("VL1_PLAIN_KERNEL");
  const bool force_scalar = kern_env && std::string(kern_env) == "scalar";
  if (dense && !force_scalar && !pl->is_complex && pl->n <= kNFMaxK && a->n_rhs >= 5 &&
      !(pl->has_missing && prm.log_disp)) {
    const int m16 = (pl->n + 15) / 16;
    const int KP = (pl->n + 31) / 32 * 32;
    hipStream_t st = (hipStream_t)stream;
    if (m16 <= 1) launch_nf_mfma<1, 1>(prm, KP, a->n_tgt_boxes, pl->dense_finite, st);
    else if (m16 <= 2) launch_nf_mfma<2, 1>(prm, KP, a->n_tgt_boxes, pl->dense_finite, st);
    else if (m16 <= 4) launch_nf_mfma<4, 1>(prm, KP, a->n_tgt_boxes, pl->dense_finite, st);
    else if (m16 <= 8) launch_nf_mfma<8, 1>(prm, KP, a->n_tgt_boxes, pl->dense_finite, st);
    else launch_nf_mfma<8, 2>(prm, KP, a->n_tgt_boxes, pl->dense_finite, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
      return fail(VL1_E_HIP, std::string("near_field_mfma launch: ") + hipGetErrorString(e));
    return exterior_pass(prm, a, st);
  }
  const size_t fixed =
      sizeof(double) * ((size_t)pl->n * RC * vw + pl->n + (P > 1 ? kNFBlock * RC * vw : 0)) +
      sizeof(int) * pl->n;
  if (fixed > lds_cap) return fail(VL1_E_UNSUPPORTED, "vl1_near_field_f64: box too large for LDS");
  size_t tbuf = dense ? 0
                      : std::min<size_t>((size_t)pl->max_orbit_count * vw,
                                         (lds_cap - fixed) / sizeof(double));
  prm.tbuf = (int)tbuf;
  const size_t smem = fixed + sizeof(double) * tbuf;
  hipError_t e;
  const bool u16 = pl->rowmap_u16 != 0;
  const int grid = a->n_tgt_boxes;
#define VL1_NF_LAUNCH(RCV, CPX)                                                                  \
  (dense ? launch_nf<uint16_t, RCV, CPX, true>(prm, grid, smem, s)                               \
         : (u16 ? launch_nf<uint16_t, RCV, CPX, false>(prm, grid, smem, s)                       \
                : launch_nf<int32_t, RCV, CPX, false>(prm, grid, smem, s)))
  if (pl->is_complex)
    e = RC == 1 ? VL1_NF_LAUNCH(1, true) : (RC == 4 ? VL1_NF_LAUNCH(4, true) : VL1_NF_LAUNCH(16, true));
  else
    e = RC == 1 ? VL1_NF_LAUNCH(1, false) : (RC == 4 ? VL1_NF_LAUNCH(4, false) : VL1_NF_LAUNCH(16, false));
#undef VL1_NF_LAUNCH
  if (e != hipSuccess)
    return fail(VL1_E_HIP, std::string("near_field_f64 launch: ") + hipGetErrorString(e));
  return exterior_pass(prm, a, s);
}
