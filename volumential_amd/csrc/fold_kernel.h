// Tile kernel of the folded FP64 form (see fold.h); instantiated in fold_2d.hip,
// fold_2dc.hip, fold_3d.hip and fold_3dodd.hip.
#pragma once

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "fold.h"

namespace vl1 {

typedef __attribute__((ext_vector_type(4))) double fold_double4;
typedef __attribute__((ext_vector_type(2))) double fold_double2;

template <int I, int N, typename F>
__device__ __forceinline__ void fold_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    fold_for<I + 1, N>(f);
  }
}

// 4-row groups of all parities, by the counts of a parity with 0..3 odd axes.
constexpr int fold_rows4(int np, int g0, int g1, int g2, int g3) {
  return 4 * (np == 8 ? g0 + 3 * g1 + 3 * g2 + g3 : (np == 4 ? g0 + 2 * g1 + g2 : (np == 2 ? g0 + g1 : g0)));
}
// Whether all columns' outputs go through LDS at once: in a slot of at most the
// 8 units' and 4.5 KB more (two workgroups of 3D q = 6 still share a CU).
constexpr bool fold_whole(int np, int nct, int g0, int g1, int g2, int g3) {
  return nct == 1 ||
         fold_rows4(np, g0, g1, g2, g3) * (16 * nct + 1) <= kFoldUnits * np * nct * 64 + 576;
}

// For a thread with outputs that came out infinite or NaN: each of its outputs
// again, as the products of the densities' infinities and NaN with their entries
// of the blocks, the signed infinity or NaN that the sum over sources has
// (finite products do not matter; a NaN ends the sum).  Outputs without any keep
// what was written.  Slow and meant for few: 24 densities of 4096 boxes, 3D q = 6,
// all NaN 1.6 ms (finite 1.2), all +inf 730.
template <int NP>
__device__ inline void fold_nonfinite(const FoldParams& p, const double* smem, int wg) {
  const int n_rc = (p.R + p.Rc - 1) / p.Rc;
  const int i8 = wg / 8, bt = i8 / n_rc * 8 + wg % 8, rcx = i8 % n_rc;
  const FoldTileInfo& ti = p.tiles[bt];
  const double* log_sums = smem + p.slot_doubles + 32 * NP * 2 + 64 * NP;
  const FoldBlocks& f = *p.blocks;
  const int row = threadIdx.x % p.rows;
  const double* Xc = p.X + (int64_t)rcx * (p.nb + 1) * p.d.kg * p.Rc * 4;
  // (as in fold_run: one row, every cpt-th column)
  const int cpt = 64 * NP / p.rows;
  for (int c = threadIdx.x / p.rows; c < p.B * p.Rc; c += cpt) {
    const int b = c / p.Rc, r = c % p.Rc, R = rcx * p.Rc + r, box = p.tile_boxes[bt * p.B + b];
    if ((int)threadIdx.x >= cpt * p.rows || R >= p.R || box < 0) continue;
    double sum = 0.0;
    bool any = false;
    int64_t step = ti.step - 1;
    for (int i = 0; i < ti.n_chunks && sum == sum; ++i) {
      const uint32_t w = p.chunks[ti.chunk + i];
      if (!fold_chunk_first(w)) continue;
      ++step;
      const int z = fold_chunk_z(w), blk = f.rep_blk[fold_chunk_cls(w)] * f.n_rg;
      for (int j = 0; j < 1 << fold_chunk_m(w) && sum == sum; ++j) {
        const int src = p.step_src[(step * p.B + b) * NP + j];
        if (src == p.nb) continue;
        int J = 0;  // the slot's negative axes
        for (int a = 0, k = 0; a < 3; ++a)
          if ((z >> a) & 1) J |= ((j >> k++) & 1) << a;
        const int t = row / p.nm * p.nm + reflect_node(f.dim, f.q, row % p.nm, J);
        const double* m = f.M + ((int64_t)(blk + t / f.rg_size) * f.MP + t % f.rg_size) * f.KP;
        const double eps = (__popc((unsigned)J & p.d.sp) & 1) ? -1.0 : 1.0;
        for (int e = 0; e < 4 * p.d.kg && sum == sum; ++e) {
          const double x = Xc[(((int64_t)src * p.d.kg + e / 4) * p.Rc + r) * 4 + e % 4];
          if (fabs(x) <= kFoldMax || (uint64_t)__double_as_longlong(x) == kFoldFinite) continue;
          const FoldSlot s = f.slots[e / 4 * 4 + ((e % 4) ^ ((e % 4) >> 1))];
          int node = s.base;
          for (int a = 0; a < 3; ++a)
            if ((s.par >> a) & 1) node += s.d[a];
          sum += eps * m[node / p.nm * p.nm + reflect_node(f.dim, f.q, node % p.nm, J)] * x;
          any = true;
        }
      }
    }
    if (!any) continue;
    if (p.est) p.est[2 * R] = p.est[2 * R + 1] = __builtin_nan("");
    const int64_t mp = p.mode_point[(int64_t)box * p.nm + row % p.nm];
    p.y[R * p.ldy + (p.cplx ? 2 * mp + row / p.nm : mp)] = p.dl ? sum + log_sums[c] : sum;
  }
}

// A workgroup of NP waves computes 16 NCT columns (B target boxes x Rc
// densities) of all rows; wave w owns the rows of one output parity, G groups
// of 4, in the accumulators of v_mfma_f64_16x16x4f64 (G / 4 full 16-row
// tiles) and v_mfma_f64_4x4x4f64 (the G % 4 <= 2 remaining groups, the table
// fragment the same in the instruction's four blocks): both run at the full
// FP64 rate (measured 76 and 77 TFLOP/s), so rows need no padding to 16.  Three
// remaining groups are padded to a tile all the same: a fragment load returns
// 512 bytes to the wave whatever it reads, at 64 bytes per clock and CU, and
// with four loads per unit (q = 6: 7 groups) that path was as busy as the
// FP64 pipe (24 densities, 4096 boxes: 1093 us against 1060 us with two full
// tiles; q = 5 graded, 14246 boxes, one density: 340 against 307 us).
// G0..G3 are the groups of a parity with 0..3 odd axes: a wave runs the loop
// compiled for its own count (equal for even orders: one loop).
//
// A tile's steps (classes) run in chunks of 8 units per wave, a unit being
// one (sum s, K group of 4) with its block: 8 >> m K rounds of all parities
// for a class with m nonzero axes; which units a wave takes comes from a table
// (scalar loads).  Per chunk every thread loads the same number of values (16
// bytes each), forms the 2^m signed sums of its sources in registers and
// writes them, in MFMA operand order (conflict free), to the LDS slot.  Orders
// of few rounds skip the loads that no unit of theirs reads (known when
// compiled: 3D q = 4, 32768 boxes, 64 densities 5309 -> 5038 us, the digit kernel
// at 5 slices 5066; 3D q = 2 1431 -> 1038; 2D q = 4, 65536 boxes 2318 -> 2006).  The
// loads of the next chunk are issued before this chunk's MFMAs; table
// fragments run one or three units ahead and the lists of source boxes four steps
// ahead (an LDS ring).  All of them are issued unconditionally -- a skipped
// unit, or a chunk past the tile's end, reads some valid place -- so that no
// branch separates a load from its wait.
//
// Bound: the FP64 pipe, which MFMA and the VALU's FP64 additions share
// (measured: the two together reach the same 75 TFLOP/s as either alone).
// In one workgroup the MFMAs, the sums and the waits follow each other, so the
// registers (at most 128 for G <= 8) and the one LDS slot are sized for two
// workgroups per CU, each running its MFMAs while the other loads and sums: 3D
// q = 6, 24 densities, 4096 boxes: 1146 us for one workgroup of 64 columns per
// CU with two slots, 1060 us for two of 32 columns (general form: 7816 us; 1015
// us with the products at raised priority and the tile's entry and exit as below).
// The FP64 pipe is then busy about 55% of the time; the load path (fragments
// and values) about 60%.
// Returns 0, NaN if an output of this thread is not finite.
template <int NP, int NCT, int G, int RMAX, bool WHOLE>
__device__ __forceinline__ double fold_run(const FoldParams& p, double* smem, int bt, int rcx,
                                           int pout, int grow) {
  constexpr int T = 64 * NP, COLS = 16 * NCT, UW = kFoldUnits;
  constexpr int LPT = COLS / 4;             // 16-byte loads per thread and chunk
  // ... of which those past the order's RMAX rounds (the rows of the largest
  // parity, groups of 4) hold nothing: a round is one load of 32 columns, half of
  // 16.  From 4 rounds on all are issued: of the chunks only a step with no
  // nonzero axis has such loads, and the kernel built without them was slower (3D
  // q = 4 complex, 4096 boxes, 5 densities 118 -> 130 us; 2D q = 6 equal).
  constexpr int NU = RMAX >= 4 ? LPT : (COLS == 32 ? RMAX : (RMAX + 1) / 2);
  constexpr int NXB = LPT > NP ? LPT : NP;  // registers for them (2^m <= NP)
  constexpr int SLOT = UW * NP * NCT * 64;  // doubles of the LDS slot
  constexpr int NT = G / 4, GC = G % 4, NF = NT > 0 ? NT : 1, NG = GC > 0 ? GC : 1;
  constexpr int CV = NCT - 1;  // load table of this width
  constexpr bool AHEAD = NP < 8 || G <= 4;  // columns read a unit ahead
  constexpr int NB = AHEAD ? 2 : 1;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r0 = rcx * p.Rc;

  // ---- this thread's share of a chunk's loads
  // lane pairs read the 32 bytes of a K group (in the order k = 0 1 3 2, so
  // that the two halves of a pair go to different LDS banks)
  const int kp = lane & 1;
  const int col = (lane >> 1) & (COLS - 1);
  const int kgo = COLS < 32 ? lane >> 5 : 0;  // K group within the wave's pair
  const int cb = col / p.Rc, cr = col % p.Rc;
  const bool live = cb < p.B && r0 + cr < p.R;
  const uint32_t box_bytes = (uint32_t)p.d.kg * p.Rc * 32;
  const uint32_t kg_bytes = (uint32_t)p.Rc * 32;
  const uint32_t off0 = (uint32_t)(cr * 32 + kp * 16) + kgo * kg_bytes;
  const uint32_t none = (uint32_t)p.nb * box_bytes;  // the zero box
  const char* Xc = reinterpret_cast<const char*>(p.X) + (int64_t)rcx * (p.nb + 1) * box_bytes;

  // ---- sources of the steps: ring of four in LDS (byte offsets of the boxes),
  // one per thread and step
  uint32_t* ring = reinterpret_cast<uint32_t*>(smem + p.slot_doubles);
  double* sPart = smem + p.slot_doubles + 32 * NP * 2;  // [T / COLS][COLS] log-term sums
  double* sD = sPart + T;
  int64_t* sBox = reinterpret_cast<int64_t*>(sD + COLS);  // column -> its box's modes, y row offset
  const int n_src = p.B * NP;  // <= T
  const FoldTileInfo ti = p.tiles[bt];
  const int32_t* srow = p.step_src + (int64_t)ti.step * n_src + (tid < n_src ? tid : 0);
  int step = 0, carry = 0;      // the step last entered; the list on its way to the ring
  bool pending = false;
  // the list fetched when this step was entered (step + 3) into the slot of the
  // step before it, which every wave has left
  auto land = [&]() {
    if (pending) {
      if (tid < n_src) ring[((step + 3) & 3) * 32 * NP + tid] = (uint32_t)carry * box_bytes;
      pending = false;
    }
  };

  fold_double2 xb[NXB];
  const uint2* lutl = p.lut_l + (int64_t)CV * 4 * p.maxc * NP + wave;
  auto load_m = [&](uint2 kgs, auto mc) {
    constexpr int M = decltype(mc)::value;
    constexpr int NI = std::min((LPT >> M) > 0 ? (LPT >> M) : 1, NU);
    const uint32_t* q = ring + (step & 3) * 32 * NP + (live ? cb : 0) * NP;
    uint32_t vo[1 << M];
#pragma unroll
    for (int j = 0; j < (1 << M); ++j) vo[j] = (live ? q[j] : none) + off0;
    fold_for<0, NI>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      const uint32_t kg = ((u < 4 ? kgs.x : kgs.y) >> (8 * (u % 4))) & 255;
      const char* base = Xc + (size_t)kg * kg_bytes;
#pragma unroll
      for (int j = 0; j < (1 << M); ++j)
        xb[(u << M) + j] = *reinterpret_cast<const fold_double2*>(base + vo[j]);
    });
  };
  const int lds0 = (kgo * NCT + col / 16) * 64 + 48 * kp + col % 16;
  auto store_m = [&](auto mc) {
    constexpr int M = decltype(mc)::value;
    constexpr int NI = std::min((LPT >> M) > 0 ? (LPT >> M) : 1, NU), NK = (UW * NP) >> M;
    // (opaque, so that the addresses of every m are not all kept in registers)
    int lds = lds0;
    asm volatile("" : "+v"(lds));
    fold_for<0, NI>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      const int q = wave + NP * u, kgl = COLS == 32 ? q : 2 * q;
      if (kgl >= NK) return;  // uniform
      fold_double2 v[1 << M];
#pragma unroll
      for (int j = 0; j < (1 << M); ++j) v[j] = xb[(u << M) + j];
#pragma unroll
      for (int b = 0; b < M; ++b)
#pragma unroll
        for (int j = 0; j < (1 << M); ++j)
          if (!((j >> b) & 1)) {
            const fold_double2 a = v[j], c = v[j | (1 << b)];
            v[j] = a + c;
            v[j | (1 << b)] = a - c;
          }
      double* dst = smem + kgl * (NCT * 64) + lds;
      double* dsy = dst + 16 - 32 * kp;
#pragma unroll
      for (int j = 0; j < (1 << M); ++j) {
        dst[j * NK * NCT * 64] = v[j].x;
        dsy[j * NK * NCT * 64] = v[j].y;
      }
    });
  };
  using M0 = std::integral_constant<int, 0>;
  using M1 = std::integral_constant<int, NP >= 2 ? 1 : 0>;
  using M2 = std::integral_constant<int, NP >= 4 ? 2 : 0>;
  using M3 = std::integral_constant<int, NP >= 8 ? 3 : 0>;
  auto load_x = [&](uint32_t w, uint2 kgs) {
    const int m = fold_chunk_m(w);
    if (NP >= 8 && m == 3) load_m(kgs, M3{});
    else if (NP >= 4 && m == 2) load_m(kgs, M2{});
    else if (NP >= 2 && m == 1) load_m(kgs, M1{});
    else load_m(kgs, M0{});
  };
  auto store_x = [&](uint32_t w) {
    const int m = fold_chunk_m(w);
    if (NP >= 8 && m == 3) store_m(M3{});
    else if (NP >= 4 && m == 2) store_m(M2{});
    else if (NP >= 2 && m == 1) store_m(M1{});
    else store_m(M0{});
  };

  // ---- table fragments: unit stream, set u % NS, loaded NS - 1 units ahead
  // (many fragments: one, for registers; a unit then takes long enough)
  constexpr int NS = NT + GC > 2 ? 2 : 4;
  double aF[NS][NF], aC[NS][NG];
  const double* Aw = p.A + (int64_t)16 * grow;
  const int lc = (lane / 16) * 4 + lane % 4;
  const uint32_t kg_a = (uint32_t)p.d.rows4 * 4;
  auto load_a = [&](uint32_t w, uint32_t unit, auto uc) {
    constexpr int u = decltype(uc)::value;
    const double* a = Aw + (int64_t)fold_chunk_cls(w) * p.cls_stride + ((unit >> 8) & 255) * kg_a;
#pragma unroll
    for (int t = 0; t < NT; ++t) aF[u][t] = a[64 * t + lane];
#pragma unroll
    for (int g = 0; g < GC; ++g) aC[u][g] = a[64 * NT + 16 * g + lc];
  };
  struct Units {
    uint4 a, b;
  };
  auto units_of = [&](uint32_t w) {
    const uint4* q = p.lut_u + ((fold_chunk_z(w) * p.maxc + fold_chunk_c(w)) * NP + pout) * 2;
    return Units{q[0], q[1]};
  };
  auto kgs_of = [&](uint32_t w) { return lutl[(fold_chunk_m(w) * p.maxc + fold_chunk_c(w)) * NP]; };

  fold_double4 accF[NF][NCT];
  double accC[NG][NCT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
#pragma unroll
    for (int t = 0; t < NF; ++t) accF[t][ct] = fold_double4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int g = 0; g < NG; ++g) accC[g][ct] = 0.0;
  }

  // ---- pipeline.  Words past the tile's last chunk belong to the next tile
  // (or the lists' padding): what they prefetch is valid and not used.
  const int nch = ti.n_chunks;
  const uint32_t* words = p.chunks + ti.chunk;
  uint32_t w0 = ti.words[0], w1 = ti.words[1], w2 = ti.words[2];
  Units uC = units_of(w0), uN = units_of(w1);
  {
    int s4[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) s4[k] = srow[(int64_t)k * n_src];
    load_a(w0, uC.a.x, std::integral_constant<int, 0>{});
    if constexpr (NS > 2) {
      load_a(w0, uC.a.y, std::integral_constant<int, 1>{});
      load_a(w0, uC.a.z, std::integral_constant<int, 2>{});
    }
    if (tid < COLS) {  // for the outputs
      const int b = tid / p.Rc, r = tid % p.Rc;
      const int tb = b < p.B && r0 + r < p.R ? p.tile_boxes[bt * p.B + b] : -1;
      sBox[2 * tid] = tb < 0 ? -1 : (int64_t)tb * p.nm;
      sBox[2 * tid + 1] = (int64_t)(r0 + r) * p.ldy;
    }
    if (tid < n_src)
#pragma unroll
      for (int k = 0; k < 4; ++k) ring[k * 32 * NP + tid] = (uint32_t)s4[k] * box_bytes;
    srow += (int64_t)4 * n_src;
    if (p.dl) {  // 2D log term: this thread's part of its column's sources
      const int n = ti.n_steps * NP;
      const int b = (tid % COLS) / p.Rc, r = (tid % COLS) % p.Rc;
      const bool in = b < p.B && r0 + r < p.R;
      const int32_t* q = p.step_src + (int64_t)ti.step * n_src + (in ? b : 0) * NP;
      const double* dlc = p.dl + (int64_t)rcx * (p.nb + 1) * p.Rc + (in ? r : 0);
      double a = 0.0;
      for (int e = tid / COLS; e < n; e += T / COLS)
        a += dlc[(int64_t)(in ? q[(int64_t)(e / NP) * n_src + e % NP] : p.nb) * p.Rc];
      sPart[tid] = a;
    }
  }
  __syncthreads();
  auto enter = [&](uint32_t w) {  // a chunk that begins a step: its sources
    if (fold_chunk_first(w)) {
      ++step;
      carry = *srow;
      srow += n_src;
      pending = true;
    }
  };
  load_x(w0, kgs_of(w0));
  uint2 kg1 = kgs_of(w1);
  for (int i = 0; i < nch; ++i) {
    const uint32_t w3 = words[i + 3];
    const Units uF = units_of(w2);
    __syncthreads();  // every wave has read the slot (and its sources)
    store_x(w0);
    land();
    enter(w1);
    load_x(w1, kg1);
    kg1 = kgs_of(w2);
    __syncthreads();
    // matrix work first: the other workgroup's sums and loads fill its gaps
    __builtin_amdgcn_s_setprio(1);
    double bx[NB][NCT];
    fold_for<0, UW>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      auto word = [](const Units& x, int k) {
        const uint4& q = k < 4 ? x.a : x.b;
        return k % 4 == 0 ? q.x : (k % 4 == 1 ? q.y : (k % 4 == 2 ? q.z : q.w));
      };
      const uint32_t unit = word(uC, u);
      constexpr int un = u + NS - 1;
      load_a(un < UW ? w0 : w1, un < UW ? word(uC, un % UW) : word(uN, un % UW),
             std::integral_constant<int, un % NS>{});
      // the unit's columns; a unit ahead where the registers allow
      auto columns = [&](uint32_t w, int k) {
        const double* b = smem + (w & 255) * (NCT * 64) + lane;
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) bx[k][ct] = b[64 * ct];
      };
      if (u == 0 || !AHEAD) columns(unit, u % NB);
      if (AHEAD && u + 1 < UW) columns(word(uC, (u + 1) % UW), (u + 1) % NB);
      if (unit >> 16) {  // uniform; no load inside
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct)
            accF[t][ct] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(aF[u % NS][t], bx[u % NB][ct], accF[t][ct], 0, 0, 0);
#pragma unroll
        for (int g = 0; g < GC; ++g)
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct)
            accC[g][ct] =
                __builtin_amdgcn_mfma_f64_4x4x4f64(aC[u % NS][g], bx[u % NB][ct], accC[g][ct], 0, 0, 0);
      }
    });
    __builtin_amdgcn_s_setprio(0);
    uC = uN;
    uN = uF;
    w0 = w1;
    w1 = w2;
    w2 = w3;
  }

  // ---- output: back to box nodes through LDS, all columns at once (WHOLE; 16
  // where the rows are too many); a thread keeps one row (rows <= T) and takes
  // every cpt-th column, KB at a time, with their points loaded a batch ahead
  constexpr int OC = WHOLE ? COLS : 16, PITCH = OC + 1, KB = 4;
  const int cpt = T / p.rows, t = tid % p.rows, cc = tid / p.rows;
  const FoldOut o = p.out[t];
  const int tm = t % p.nm, part = t / p.nm;
  int mp[KB];
  auto points = [&](int c0) {  // of columns c0 + k cpt
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int c = c0 + k * cpt;
      const int64_t bm = cc < cpt && c < COLS ? sBox[2 * c] : -1;
      mp[k] = p.mode_point[bm < 0 ? 0 : bm + tm];
      if (bm < 0) mp[k] = -1;
    }
  };
  points(cc);
  if (p.dl && tid < COLS) {
    double a = 0.0;
    for (int k = 0; k < T / COLS; ++k) a += sPart[k * COLS + tid];
    sD[tid] = a;
  }
  const double scale = 1.0 / (double)(1 << o.shift);
  double finite = 0.0;  // NaN if an output is not finite
  fold_for<0, COLS / OC>([&](auto occ) {
    constexpr int oc = decltype(occ)::value;
    __syncthreads();
    double* yh = smem + (4 * grow + lane / 16) * PITCH + lane % 16;
#pragma unroll
    for (int ct = oc * (OC / 16); ct < (oc + 1) * (OC / 16); ++ct) {
      double* yc = yh + 16 * ct - OC * oc;
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) yc[(16 * k + 4 * e) * PITCH] = accF[k][ct][e];
#pragma unroll
      for (int g = 0; g < GC; ++g) yc[(16 * NT + 4 * g) * PITCH] = accC[g][ct];
    }
    __syncthreads();
    if (cc < cpt) {
      for (int c0 = OC * oc + cc; c0 < OC * (oc + 1); c0 += KB * cpt) {
        int mc[KB];
#pragma unroll
        for (int k = 0; k < KB; ++k) mc[k] = mp[k];
        const int cn = c0 + KB * cpt;
        points(cn < OC * (oc + 1) ? cn : OC * (oc + 1) + cc);
#pragma unroll
        for (int k = 0; k < KB; ++k) {
          const int c = c0 + k * cpt;
          if (mc[k] < 0 || c >= OC * (oc + 1)) continue;
          double v = 0.0;
#pragma unroll
          for (int q = 0; q < NP; ++q)
            if (o.row[q] >= 0) {
              const double h = smem[o.row[q] * PITCH + c - OC * oc];
              v += (__popc(q & o.flips) & 1) ? -h : h;
            }
          v *= scale;
          finite = fma(v, 0.0, finite);
          if (p.dl) v += sD[c];
          p.y[sBox[2 * c + 1] + (p.cplx ? 2 * (int64_t)mc[k] + part : (int64_t)mc[k])] = v;
        }
      }
    }
  });
  return finite;
}

template <int NP, int NCT, int G0, int G1, int G2, int G3>
__global__ void __launch_bounds__(64 * NP, G0 <= 8 ? 4 : 2) fold_f64_kernel(const FoldParams p) {
  extern __shared__ __align__(16) double fold_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // workgroup i runs on XCD i % 8: box tile and density group, the groups of a
  // tile one after the other on its XCD
  const int n_rc = (p.R + p.Rc - 1) / p.Rc;
  const int i = (int)(blockIdx.x / 8), bt = i / n_rc * 8 + (int)(blockIdx.x % 8), rcx = i % n_rc;
  if (bt >= p.n_box_tiles) return;  // uniform over the workgroup
  if (threadIdx.x == 0) {           // for the end of the kernel, out of the registers
    reinterpret_cast<uint64_t*>(fold_smem)[0] = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    reinterpret_cast<int*>(fold_smem)[2] = (int)blockIdx.x;
  }
  // waves 0-3 and 4-7 pair large with small parities on a SIMD (odd orders)
  const int pout = NP == 8 ? (0x35674210 >> (4 * wave)) & 7 : wave;
  int grow = 0;  // groups before this parity
  for (int k = 0; k < NP; ++k)
    if (k < pout) grow += (int)((p.d.groups_lo >> (8 * k)) & 255);
  constexpr bool WHOLE = fold_whole(NP, NCT, G0, G1, G2, G3);
  double finite;
  if constexpr (G0 == G1 && G1 == G2 && G2 == G3) {
    finite = fold_run<NP, NCT, G0, G0, WHOLE>(p, fold_smem + 2, bt, rcx, pout, grow);
  } else {
    // the loops hold the same barriers, so waves may run different ones
    const int odd = __popc(pout);
    if (odd == 0) finite = fold_run<NP, NCT, G0, G0, WHOLE>(p, fold_smem + 2, bt, rcx, pout, grow);
    else if (odd == 1) finite = fold_run<NP, NCT, G1, G0, WHOLE>(p, fold_smem + 2, bt, rcx, pout, grow);
    else if (odd == 2) finite = fold_run<NP, NCT, G2, G0, WHOLE>(p, fold_smem + 2, bt, rcx, pout, grow);
    else if constexpr (NP == 8) finite = fold_run<NP, NCT, G3, G0, WHOLE>(p, fold_smem + 2, bt, rcx, pout, grow);
  }
  if (finite != 0.0) {
    // the arguments read again: kept in registers for this they spill others of
    // the loop (4 to 10 % slower)
    const auto* at = reinterpret_cast<const int*>(fold_smem);
    const int lo = __builtin_amdgcn_readfirstlane(at[0]), hi = __builtin_amdgcn_readfirstlane(at[1]);
    const uint64_t args = (uint64_t)(unsigned)hi << 32 | (unsigned)lo;
    typedef const __attribute__((address_space(4))) uint32_t* scalar_ptr;
    struct Words {
      uint32_t w[sizeof(FoldParams) / 4];
    } words;
#pragma unroll
    for (size_t k = 0; k < sizeof(FoldParams) / 4; ++k) words.w[k] = ((scalar_ptr)args)[k];
    fold_nonfinite<NP>(__builtin_bit_cast(FoldParams, words), fold_smem + 2,
                       __builtin_amdgcn_readfirstlane(at[2]));
  }
}

template <int NP, int NCT, int G0, int G1, int G2, int G3>
hipError_t launch_fold(const FoldParams& p, hipStream_t s) {
  static std::atomic<unsigned> done{0};  // devices whose LDS limit has been raised
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const unsigned bit = 1u << (dev & 31);
  auto fn = fold_f64_kernel<NP, NCT, G0, G1, G2, G3>;
  if (!(done.load(std::memory_order_acquire) & bit)) {
    e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    done.fetch_or(bit, std::memory_order_acq_rel);
  }
  FoldParams q = p;
  const int out_cols = fold_whole(NP, NCT, G0, G1, G2, G3) ? 16 * NCT : 16;
  q.slot_doubles = std::max(kFoldUnits * NP * NCT * 64, p.d.rows4 * (out_cols + 1));
  const size_t doubles = 2 + (size_t)q.slot_doubles + 32 * NP * 2 + 64 * NP + 3 * 16 * NCT;
  const int grid = (p.n_box_tiles + 7) / 8 * 8 * ((p.R + p.Rc - 1) / p.Rc);
  hipLaunchKernelGGL(fn, dim3(grid), dim3(64 * NP), doubles * sizeof(double), s, q);
  return hipGetLastError();
}

// Group counts of a parity with 0..3 odd axes as one number.
constexpr int fold_key(int g0, int g1, int g2, int g3) {
  return ((g0 * 32 + g1) * 32 + g2) * 32 + g3;
}

}  // namespace vl1
