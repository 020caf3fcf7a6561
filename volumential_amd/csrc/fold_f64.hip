// Reflection-folded FP64 contraction (see fold.h): density staging into the
// even/odd basis, the folded table blocks, and the tile kernel.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "fold.h"

namespace vl1 {

// ------------------------------------------------------------------- host
namespace {

int groups_of(const FoldDims& d, int p) { return (int)((d.groups_lo >> (8 * p)) & 255); }

int axis_len(int q, bool folded, bool odd) { return !folded ? q : (odd ? q / 2 : (q + 1) / 2); }

// Row groups of a parity with g K groups: a remainder of three groups beyond
// full 16-row tiles is padded to a tile (one 512-byte fragment load instead of
// three, each of which returns 512 bytes to the lanes; see fold_kernel.h).
int row_groups(int g) { return g % 4 == 3 ? g + 1 : g; }

// 4-entry groups of parity p with the first nf axes folded.
int parity_groups(int dim, int q, int vw, int nf, int p) {
  int len = vw;
  for (int a = 0; a < dim; ++a) len *= axis_len(q, a < nf, (p >> a) & 1);
  return (len + 3) / 4;
}

}  // namespace

bool fold_layout(FoldPlan& f, int dim, int q, int cplx, uint32_t sign_mask, bool few_axes) {
  const int vw = cplx ? 2 : 1;
  // fold as many axes as pay: the products of a class whose nonzero axes are
  // all folded (2^m sums, each with the blocks p -> p ^ s) against one fold
  // less; boxes of 2 nodes per axis keep blocks of at least one 4 x 4 tile
  auto cost = [&](int nf) {
    // per folded axis: one same-parity pair of blocks for offset 0, all four
    // for the offset pair; per unfolded axis three offsets: sum over (p, p')
    // of G_p G_p' 2^(axes where they agree)
    double c = 0.0;
    for (int p = 0; p < (1 << nf); ++p)
      for (int r = 0; r < (1 << nf); ++r)
        c += (double)row_groups(parity_groups(dim, q, vw, nf, p)) * parity_groups(dim, q, vw, nf, r) *
             (1 << (nf - __builtin_popcount(p ^ r)));
    for (int a = nf; a < dim; ++a) c *= 3.0;
    return c;
  };
  if (q < 2) return false;
  int nf = 0;
  for (int k = 1; k <= dim; ++k)
    if (cost(k) < cost(nf)) nf = k;
  // 3D q = 3: all axes folded leave parities of 8 to 1 entries, so that most of
  // a chunk's waves and loads serve padding (plan_fold says what it costs)
  if (few_axes) {
    if (dim != 3 || q != 3) return false;
    nf = cplx ? 2 : 0;
  }
  FoldDims d;
  d.nf = nf;
  d.np = 1 << nf;
  d.sp = sign_mask & (uint32_t)(d.np - 1);
  int order[8];
  for (int p = 0; p < d.np; ++p) order[p] = p;
  auto G = [&](int p) { return parity_groups(dim, q, vw, nf, p); };
  std::stable_sort(order, order + d.np, [&](int a, int b) { return G(a) > G(b); });
  d.rounds = G(order[0]);
  if (d.rounds > kFoldMaxGroups) return false;
  for (int i = 0; i < d.np; ++i) {
    d.ppos |= (uint32_t)i << (4 * order[i]);
    d.groups_lo |= (uint64_t)row_groups(G(i)) << (8 * i);
    d.rows4 += 4 * row_groups(G(i));
  }
  for (int r = 0; r < d.rounds; ++r) {
    int c = 0;
    while (c < d.np && G(order[c]) > r) ++c;
    d.cnt |= (uint64_t)c << (4 * r);
    d.kgs[r / 8] |= (uint64_t)d.kg << (8 * (r % 8));
    d.kg += c;
  }
  if (d.kg > 255 || !fold_has_kernel(d)) return false;
  f.d = d;
  int n = 1;
  for (int a = 0; a < dim; ++a) n *= q;
  f.nm = n;
  f.cplx = cplx;
  f.rows = vw * n;
  int stride[3] = {0, 0, 0};
  for (int a = dim - 1, s = 1; a >= 0; --a, s *= q) stride[a] = s;
  // entries of each parity, lexicographic in the folded indices, imaginary
  // parts after the real ones
  f.slots.assign((size_t)d.kg * 4, FoldSlot{0, {0, 0, 0}, 0, 0, 0, 0});
  std::vector<int> row0(d.np, 0);
  for (int p = 1; p < d.np; ++p) row0[p] = row0[p - 1] + 4 * row_groups(G(p - 1));
  f.outs.assign(f.rows, FoldOut{{-1, -1, -1, -1, -1, -1, -1, -1}, 0, 0, {0, 0}});
  for (int p = 0; p < d.np; ++p) {
    int len[3] = {1, 1, 1}, cnt = 1;
    for (int a = 0; a < dim; ++a) {
      len[a] = axis_len(q, a < nf, (p >> a) & 1);
      cnt *= len[a];
    }
    for (int e = 0; e < vw * cnt; ++e) {
      int rem = e % cnt, idx[3] = {0, 0, 0};
      for (int a = dim - 1; a >= 0; --a) {
        idx[a] = rem % len[a];
        rem /= len[a];
      }
      FoldSlot s{0, {0, 0, 0}, 0, (uint8_t)p, 1, 0};
      int base = (e / cnt) * n;
      for (int a = 0; a < dim; ++a) {
        base += idx[a] * stride[a];
        if (a < nf && q - 1 - idx[a] != idx[a]) {
          s.amask |= (uint8_t)(1 << a);
          s.d[a] = (int16_t)((q - 1 - 2 * idx[a]) * stride[a]);
        }
      }
      s.base = (int16_t)base;
      const int pos = (int)((d.ppos >> (4 * p)) & 15), r = e / 4;
      const int kg = (int)((d.kgs[r / 8] >> (8 * (r % 8))) & 255) + pos;
      f.slots[(size_t)kg * 4 + e % 4] = s;
      for (uint32_t J = 0; J < 8; ++J) {  // the output rows this entry is part of
        if (J & ~(uint32_t)s.amask) continue;
        int row = base;
        for (int a = 0; a < dim; ++a)
          if ((J >> a) & 1) row += s.d[a];
        f.outs[row].row[p] = (int16_t)(row0[p] + e);
        f.outs[row].flips = (uint8_t)J;
        f.outs[row].shift = (uint8_t)__builtin_popcount(s.amask);
      }
    }
  }
  // what a wave computes and loads per chunk (fold_kernel.h)
  auto cnt_of = [&](int r) { return r < d.rounds ? (int)((d.cnt >> (4 * r)) & 15) : 0; };
  auto kgs_of = [&](int r) { return (int)((d.kgs[r / 8] >> (8 * (r % 8))) & 255); };
  f.maxc = 1;
  for (int m = 0; m <= nf; ++m) f.maxc = std::max(f.maxc, fold_chunks(d, m));
  const int np = d.np;
  f.lut_u.assign((size_t)8 * f.maxc * np * 2, make_uint4(0, 0, 0, 0));
  f.lut_l.assign((size_t)2 * 4 * f.maxc * np, make_uint2(0, 0));
  for (int z = 0; z < np; ++z) {
    const int m = __builtin_popcount(z), rpc = kFoldUnits >> m;
    int bit[3] = {0, 0, 0};
    for (int a = 0, k = 0; a < nf; ++a)
      if ((z >> a) & 1) bit[k++] = 1 << a;
    for (int c = 0; c < fold_chunks(d, m); ++c)
      for (int w = 0; w < np; ++w) {
        uint32_t u8[kFoldUnits];
        for (int u = 0; u < kFoldUnits; ++u) {
          const int rr = u >> m, j = u & ((1 << m) - 1), round = c * rpc + rr;
          int s = 0;
          for (int k = 0; k < m; ++k)
            if ((j >> k) & 1) s |= bit[k];
          const int pi = (int)((d.ppos >> (4 * (w ^ s ^ (int)d.sp))) & 15);
          const int unit = j * (np * rpc) + rr * np + pi;
          u8[u] = pi < cnt_of(round) ? (uint32_t)(1 << 16 | (kgs_of(round) + pi) << 8 | unit) : 0;
        }
        uint4* q = &f.lut_u[(((size_t)z * f.maxc + c) * np + w) * 2];
        q[0] = make_uint4(u8[0], u8[1], u8[2], u8[3]);
        q[1] = make_uint4(u8[4], u8[5], u8[6], u8[7]);
      }
  }
  for (int cv = 0; cv < 2; ++cv)  // tiles of 16, 32 columns
    for (int m = 0; m <= nf; ++m)
      for (int c = 0; c < fold_chunks(d, m); ++c)
        for (int w = 0; w < np; ++w) {
          uint64_t b = 0;
          for (int u = 0; u < 8; ++u) {
            const int q8 = w + np * u, kgl = cv == 1 ? q8 : 2 * q8;
            if (kgl >= (kFoldUnits * np) >> m) continue;
            const int round = c * (kFoldUnits >> m) + kgl / np, pi = kgl % np;
            if (pi < cnt_of(round)) b |= (uint64_t)(kgs_of(round) + pi) << (8 * u);
          }
          f.lut_l[(((size_t)cv * 4 + m) * f.maxc + c) * np + w] =
              make_uint2((uint32_t)b, (uint32_t)(b >> 32));
        }
  return true;
}

// Densities per tile: the split of R over tiles of `cols` columns that leaves
// the fewest columns idle (R = 24 over 64 columns: 3 x 8 densities of 8 boxes,
// all columns in use; 59: 15 x 4), at a cost by the densities themselves:
// neighbouring boxes in a tile share their sources' cache lines, so a run of
// 128 bytes or more per box and K group (4, 8) is best, one density per tile
// reads a quarter line per box (13 % slower at 64 densities), and counts that
// are no power of two straddle lines.  Measured, us at 1 / 2 / 4 / 8 densities
// per tile: 3D q = 6, 4096 boxes, 64 densities 3020 / 2750 / 2651 / 2663; 2D q =
// 6, 4096 boxes 277 / 245 / 249 / 252.  Prime counts then take 2 or 4 with a few
// columns idle and not 1: 13 densities, 3D q = 4, 4096 boxes 183 / 164; 29, 2D q
// = 3, 16384 boxes 346 / 279; 11, 3D q = 6, 4096 boxes 558 / 531.  Narrow tiles
// run at one workgroup per CU or less, where fewer tiles count for more (7
// densities, 3D q = 3, 512 boxes: 26 at 1 per tile, 29 at 4).  Large trees
// take as many as the kernel's 32-bit offsets reach (3D q = 6: 8 densities up
// to 299,591 boxes, 4 up to 599,184).
FoldTile fold_tile(const FoldDims& d, int nb, int n_tgt, int R, int nct) {
  const int Rq = std::min(R, 64);  // larger counts are whole multiples of 64
  int rc_max = Rq;
  while (rc_max > 1 && !fold_fits(d, nb, rc_max)) --rc_max;
  auto pick = [&](int nct) {
    const int cols = 16 * nct;
    FoldTile t;
    t.nct = nct;
    double best = -1.0;
    for (int rc = std::min(rc_max, cols); rc >= 1; --rc) {
      const int nrc = (Rq + rc - 1) / rc, B = cols / rc;
      double u = (double)Rq * B / (nrc * cols);
      if (nct == 1) {
        u -= rc < 8 ? 0.02 * std::log2(8.0 / rc) : (rc > 8 ? 1e-3 : 0.0);
      } else {
        switch (rc) {
          case 8: break;
          case 4: u *= 0.995; break;
          case 2: u *= 0.965; break;
          case 1: u *= 0.87; break;
          default: u *= (rc & (rc - 1)) == 0 ? 0.97 : 0.92;
        }
      }
      if (u > best) {
        best = u;
        t.Rc = rc;
        t.B = B;
      }
    }
    return t;
  };
  if (nct) return pick(nct);
  // 32 columns, unless that leaves some of the 256 CUs at one workgroup or
  // none; then 16 (q = 4, 4096 boxes, one density: three calls 141 us with 32,
  // 122 us with 16; graded q = 5, 446 tiles: 477 us with 32, 563 us with 16)
  const FoldTile t = pick(2);
  const int64_t tiles = (int64_t)((n_tgt + t.B - 1) / t.B) * ((R + t.Rc - 1) / t.Rc);
  return tiles <= 256 ? pick(1) : t;
}

size_t fold_x_size(const FoldDims& d, const FoldTile& t, int nb, int R) {
  // one K group more: narrow tiles load groups in pairs
  return (size_t)((R + t.Rc - 1) / t.Rc) * (nb + 1) * d.kg * t.Rc * 4 + t.Rc * 4;
}
size_t fold_dl_size(const FoldTile& t, int nb, int R) {
  return (size_t)((R + t.Rc - 1) / t.Rc) * (nb + 1) * t.Rc;
}

// ---------------------------------------------------------------- kernels
// A[cls][kg][16 G_p' ...]: M_hat[p', i][p, k] = sum_{J' <= amask_i}
// sum_{J <= amask_k} (-1)^{|p' & J'| + |p & J|} M[row_J'][col_J] /
// 2^{|amask_k|}, rows of parity p' as 16 x 4 fragments of
// v_mfma_f64_16x16x4f64 (lane l: row l % 16, k = l / 16) followed by the
// remaining groups as 4 x 4 fragments ([k][row]).
__global__ void __launch_bounds__(256)
    fold_table_kernel(FoldDims d, int n_cls, const FoldSlot* __restrict__ slots,
                      const int32_t* __restrict__ rep_blk, int MP, int KP, int n_rg, int rg_size,
                      const double* __restrict__ M, double* __restrict__ A) {
  const int64_t stride = (int64_t)d.kg * d.rows4 * 4;
  const int64_t total = stride * n_cls;
  for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < total;
       o += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(o / stride);
    int rem = (int)(o % stride);
    const int kg = rem / (d.rows4 * 4);
    rem %= d.rows4 * 4;
    int p = 0, G = 0;  // parity of the row
    for (;; ++p) {
      G = (int)((d.groups_lo >> (8 * p)) & 255);
      if (rem < 16 * G) break;
      rem -= 16 * G;
    }
    int i, k;  // entry of the parity, K entry of the group
    if (rem < 64 * (G / 4)) {
      i = 16 * (rem / 64) + rem % 16;
      k = (rem % 64) / 16;
    } else {
      const int q = rem - 64 * (G / 4);
      i = 16 * (G / 4) + 4 * (q / 16) + q % 4;
      k = (q % 16) / 4;
    }
    // the row's entry: K group r of parity p (a padding group has none)
    const int pos = (int)((d.ppos >> (4 * p)) & 15), r = i / 4;
    FoldSlot row{0, {0, 0, 0}, 0, 0, 0, 0};
    if (r < d.rounds && pos < (int)((d.cnt >> (4 * r)) & 15))
      row = slots[((int)((d.kgs[r / 8] >> (8 * (r % 8))) & 255) + pos) * 4 + i % 4];
    const FoldSlot col = slots[kg * 4 + k];
    double v = 0.0;
    if (row.valid && col.valid) {
      for (unsigned jr = 0; jr < 8; ++jr) {
        if (jr & ~(unsigned)row.amask) continue;
        int rr = row.base;
        for (int a = 0; a < 3; ++a)
          if ((jr >> a) & 1) rr += row.d[a];
        const double* mr = M + ((int64_t)(rep_blk[c] * n_rg + rr / rg_size) * MP + rr % rg_size) * KP;
        double s = 0.0;
        for (unsigned jc = 0; jc < 8; ++jc) {
          if (jc & ~(unsigned)col.amask) continue;
          int cc = col.base;
          for (int a = 0; a < 3; ++a)
            if ((jc >> a) & 1) cc += col.d[a];
          const double m = mr[cc];
          s += (__popc(col.par & jc) & 1) ? -m : m;
        }
        v += (__popc(row.par & jr) & 1) ? -s : s;
      }
      v = ldexp(v, -__popc(col.amask));
    }
    A[o] = v;
  }
}

// mx[c] = largest |entry| of class c's representative (infinite if one is not
// finite); rows past a group are zero in M.
__global__ void __launch_bounds__(256)
    fold_max_kernel(int64_t per, const int32_t* __restrict__ rep_blk, const double* __restrict__ M,
                    double* __restrict__ mx) {
  __shared__ double red[256];
  const double* m0 = M + rep_blk[blockIdx.x] * per;
  double m = 0.0;
  bool bad = false;
  for (int64_t i = threadIdx.x; i < per; i += 256) {
    const double v = fabs(m0[i]);
    bad = bad || !(v <= 1.7e308);
    m = fmax(m, v);
  }
  red[threadIdx.x] = bad ? __builtin_huge_val() : m;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) mx[blockIdx.x] = red[0];
}

// Check b: block blk[b] against class cls[b]'s representative reflected along
// flips[b].
__global__ void __launch_bounds__(256)
    fold_check_kernel(int dim, int q, int n, int rows, uint32_t sp, const double* __restrict__ M,
                      int MP, int KP, int n_rg, int rg_size, const int32_t* __restrict__ rep_blk,
                      const int32_t* __restrict__ blk_of, const int32_t* __restrict__ cls,
                      const int32_t* __restrict__ flips, int n_checks, const double* __restrict__ blk_max, int32_t* __restrict__ flag) {
  const int64_t total = (int64_t)n_checks * rows * rows;
  auto at = [&](int blk, int t, int s) {
    return M[((int64_t)(blk * n_rg + t / rg_size) * MP + t % rg_size) * KP + s];
  };
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int s = (int)(i % rows), t = (int)((i / rows) % rows);
    const int b = (int)(i / ((int64_t)rows * rows));
    const int c = cls[b], J = flips[b];
    const double want = at(rep_blk[c], t, s);
    const double got = at(blk_of[b], t / n * n + reflect_node(dim, q, t % n, J),
                          s / n * n + reflect_node(dim, q, s % n, J));
    const double e = (__popc((unsigned)J & sp) & 1) ? got + want : got - want;
    // finite sums of a block's 64 entries, so that an absent source adds 0
    if (!(fabs(e) <= 1e-14 * blk_max[c]) || !(blk_max[c] <= 1.7e308 / 64)) atomicOr(flag, 1);
  }
}

// Densities into the folded basis: X[rc][box][kg][r][4] = alpha(box) x the
// signed sums of the box's values, dl[rc][box][r] = the box's 2D log term;
// box nb gets zeros (the absent sources of a class).  A block takes `bx` boxes
// and `rs` densities of a tile column group at a time: 2^lw lanes read the
// values of one (box, density), with the box's node ids read once for all
// densities and kStageK values in flight per lane, into LDS in mode order; then
// a thread keeps one entry of the basis, reads its up to 8 terms at once and
// writes in output order (values that are not finite: see kFoldFinite;
// consecutive threads, consecutive doubles; 4 x 2^re
// threads for the densities of a K group, 2^gl K groups, the rest of the block
// for other boxes: 8.5 -> 5.9 us at q = 4, 4096 boxes, one density).
// Bound: memory, once the loads overlap: 4096 boxes, q = 6, 24 densities (350
// MB) 213 us with one value in flight per lane and divisions for the indices,
// 126 us so.
constexpr int kStageK = 4;
__global__ void __launch_bounds__(256)
    fold_stage_kernel(FoldDims d, int nm, int cplx, int rows, int Rc, int nb, int R, int bx, int rs,
                      int lw, int rl, int re, int gl, const FoldSlot* __restrict__ slots,
                      const double* __restrict__ f, int64_t ldf,
                      const int32_t* __restrict__ mode_point,
                      const int32_t* __restrict__ box_starts,
                      const double* __restrict__ box_alpha, const double* __restrict__ box_disp,
                      const double* __restrict__ nmlz, int log_disp, double* __restrict__ X,
                      double* __restrict__ dl) {
  extern __shared__ double sv[];  // [bx][rs][rows + 1]
  const int b0 = blockIdx.x * bx, rcx = blockIdx.y;
  const int nbx = min(bx, nb + 1 - b0);
  const int LS = rows + 1;
  const int tid = threadIdx.x;
  const int ln = tid & ((1 << lw) - 1), rln = (tid >> lw) & ((1 << rl) - 1);
  const int bln = tid >> (lw + rl), bstep = 256 >> (lw + rl);
  const int ek = tid & 3, er = (tid >> 2) & ((1 << re) - 1);
  const int ekg = (tid >> (2 + re)) & ((1 << gl) - 1), kgstep = 1 << gl;
  const int ebx = tid >> (2 + re + gl), bxstep = 64 >> (re + gl);
  for (int q0 = 0; q0 < Rc; q0 += rs) {
    const int nr = min(rs, Rc - q0);
    double finite = 0.0;
    for (int b = bln; b < nbx; b += bstep) {
      const int box = b0 + b;
      const double al = box < nb ? box_alpha[box] : 0.0;
      for (int k0 = ln; k0 < rows; k0 += kStageK << lw) {
        int64_t at[kStageK];
#pragma unroll
        for (int j = 0; j < kStageK; ++j) {
          const int k = min(k0 + (j << lw), rows - 1);
          // complex: consecutive lanes read (re, im) pairs
          const int64_t pt = mode_point[(int64_t)min(box, nb - 1) * nm + (cplx ? k >> 1 : k)];
          at[j] = cplx ? 2 * pt + (k & 1) : pt;
        }
        for (int r = rln; r < nr; r += 1 << rl) {
          const int rg = rcx * Rc + q0 + r;
          const double* fr = f + (int64_t)min(rg, R - 1) * ldf;
          const bool in = al != 0.0 && rg < R;
          double v[kStageK];
#pragma unroll
          for (int j = 0; j < kStageK; ++j) v[j] = fr[at[j]];
#pragma unroll
          for (int j = 0; j < kStageK; ++j) {
            const int k = k0 + (j << lw);
            if (k < rows)
              sv[(b * rs + r) * LS + (cplx ? (k & 1) * nm + (k >> 1) : k)] = in ? al * v[j] : 0.0;
          }
        }
      }
      if (log_disp)  // the lanes of a line take the same branches
        for (int r = rln; r < nr; r += 1 << rl) {
          const int rg = rcx * Rc + q0 + r;
          double dot = 0.0;
          const bool in = al != 0.0 && rg < R;
          if (in) {
            const double* src = f + (int64_t)rg * ldf + box_starts[box];
            for (int k = ln; k < nm; k += 1 << lw) dot = fma(nmlz[k], src[k], dot);
          }
          for (int h = 1; h < (1 << lw); h <<= 1) dot += __shfl_xor(dot, h);
          if (ln == 0) dl[((int64_t)rcx * (nb + 1) + box) * Rc + q0 + r] = in ? box_disp[box] * dot : 0.0;
        }
    }
    __syncthreads();
    if (er < nr)
      for (int kg = ekg; kg < d.kg; kg += kgstep) {
        const FoldSlot s = slots[kg * 4 + (ek ^ (ek >> 1))];  // stored in the order k = 0 1 3 2
        // axis by axis: pairs along axis 0, then 1, then 2
        auto pair = [&](double a, double c, int bit) {
          return a + ((s.amask & bit) ? ((s.par & bit) ? -c : c) : 0.0);
        };
        for (int b = ebx; b < nbx; b += bxstep) {
          const int box = b0 + b;
          const double* x = sv + (b * rs + er) * LS + s.base;
          double v = pair(pair(x[0], x[s.d[0]], 1), pair(x[s.d[1]], x[s.d[1] + s.d[0]], 1), 2);
          if (d.nf > 2) {
            const double* z = x + s.d[2];
            v = pair(v, pair(pair(z[0], z[s.d[0]], 1), pair(z[s.d[1]], z[s.d[1] + s.d[0]], 1), 2), 4);
          }
          X[(((int64_t)rcx * (nb + 1) + box) * d.kg + kg) * Rc * 4 + (q0 + er) * 4 + ek] =
              s.valid ? v : 0.0;
          finite = fma(v, 0.0, finite);
        }
      }
    if (finite != 0.0 && er < nr)  // NaN: some sum of this thread's is not finite
      for (int kg = ekg; kg < d.kg; kg += kgstep) {
        const FoldSlot s = slots[kg * 4 + (ek ^ (ek >> 1))];
        for (int b = ebx; b < nbx; b += bxstep) {
          double* at = X + (((int64_t)rcx * (nb + 1) + b0 + b) * d.kg + kg) * Rc * 4 + (q0 + er) * 4 + ek;
          if (fabs(*at) <= kFoldMax) continue;
          // the node of sign pattern par itself
          int node = s.base;
          for (int a = 0; a < d.nf; ++a)
            if ((s.par >> a) & 1) node += s.d[a];
          const double own = sv[(b * rs + er) * LS + node];
          *at = fabs(own) <= kFoldMax ? __longlong_as_double(kFoldFinite)
                                      : (own != own ? __builtin_nan("") : own);
        }
      }
    __syncthreads();
  }
}

// --------------------------------------------------------------- launches
hipError_t fold_build_launch(FoldPlan& f, int dim, int q, const double* M, int MP, int KP, int n_rg,
                             int rg_size, int32_t* flag, hipStream_t s) {
  // one allocation for the tables, the class lists and the check's scratch
  std::vector<char> h;
  auto put = [&](const void* src, size_t bytes) {
    const size_t at = h.size();
    h.resize((at + bytes + 255) / 256 * 256);
    if (src) std::memcpy(h.data() + at, src, bytes);
    return at;
  };
  // every key against its representative, then every representative against
  // itself along its zero axes
  const int n_keys = (int)f.key_cls.size();
  std::vector<int32_t> blk(n_keys), cls(f.key_cls), flips(f.key_flips);
  for (int k = 0; k < n_keys; ++k) blk[k] = k;
  for (int c = 0; c < f.n_cls; ++c)
    for (int a = 0; a < f.d.nf; ++a)
      if (!((f.zmask[c] >> a) & 1)) {
        blk.push_back(f.rep_blk[c]);
        cls.push_back(c);
        flips.push_back(1 << a);
      }
  const size_t o_u = put(f.lut_u.data(), f.lut_u.size() * sizeof(uint4));
  const size_t o_l = put(f.lut_l.data(), f.lut_l.size() * sizeof(uint2));
  const size_t o_s = put(f.slots.data(), f.slots.size() * sizeof(FoldSlot));
  const size_t o_o = put(f.outs.data(), f.outs.size() * sizeof(FoldOut));
  const size_t o_r = put(f.rep_blk.data(), f.rep_blk.size() * 4);
  const size_t o_b = put(blk.data(), blk.size() * 4);
  const size_t o_c = put(cls.data(), cls.size() * 4);
  const size_t o_f = put(flips.data(), flips.size() * 4);
  const size_t o_m = put(nullptr, (size_t)f.n_cls * 8);
  const size_t o_g = put(nullptr, 4);
  const size_t o_k = put(nullptr, sizeof(FoldBlocks));
  f.cls_stride = (int64_t)f.d.kg * f.d.rows4 * 4;
  const int64_t total = f.cls_stride * f.n_cls;
  hipError_t e = f.A.alloc((size_t)total * sizeof(double));
  if (e == hipSuccess) e = upload(f.lut, h.data(), h.size(), s);
  if (e != hipSuccess) return e;
  char* d = f.lut.as<char>();
  f.u_lut = reinterpret_cast<const uint4*>(d + o_u);
  f.l_lut = reinterpret_cast<const uint2*>(d + o_l);
  f.slot_lut = reinterpret_cast<const FoldSlot*>(d + o_s);
  f.out_lut = reinterpret_cast<const FoldOut*>(d + o_o);
  const auto* rep = reinterpret_cast<const int32_t*>(d + o_r);
  auto* mx = reinterpret_cast<double*>(d + o_m);
  auto* dflag = reinterpret_cast<int32_t*>(d + o_g);
  auto blocks = [](int64_t n) { return dim3((unsigned)std::min<int64_t>((n + 255) / 256, 65536)); };
  hipLaunchKernelGGL(fold_max_kernel, dim3(f.n_cls), dim3(256), 0, s, (int64_t)n_rg * MP * KP, rep, M,
                     mx);
  hipLaunchKernelGGL(fold_check_kernel, blocks((int64_t)blk.size() * f.rows * f.rows), dim3(256), 0, s, dim,
                     q, f.nm, f.rows, f.d.sp, M, MP, KP, n_rg, rg_size, rep,
                     reinterpret_cast<const int32_t*>(d + o_b),
                     reinterpret_cast<const int32_t*>(d + o_c),
                     reinterpret_cast<const int32_t*>(d + o_f), (int)blk.size(), mx, dflag);
  hipLaunchKernelGGL(fold_table_kernel, blocks(total), dim3(256), 0, s, f.d, f.n_cls, f.slot_lut, rep,
                     MP, KP, n_rg, rg_size, M, f.A.as<double>());
  e = hipGetLastError();
  const FoldBlocks blocks_of{f.slot_lut, M, rep, dim, q, MP, KP, n_rg, rg_size};
  f.blocks = reinterpret_cast<const FoldBlocks*>(d + o_k);
  if (e == hipSuccess)
    e = hipMemcpyAsync(d + o_k, &blocks_of, sizeof(blocks_of), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(flag, dflag, 4, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  return e;
}

hipError_t fold_stage_launch(const FoldPlan& f, const FoldTile& t, int nb, int R, const double* fin,
                             int64_t ldf, const int32_t* mode_point, const int32_t* box_starts,
                             const double* box_alpha, const double* box_disp, const double* nmlz,
                             int log_disp, double* X, double* dl, hipStream_t s) {
  // about 2048 values per block in LDS (16 KB): several blocks per CU
  const int rs = std::max(1, std::min({t.Rc, 64, 2048 / f.rows}));
  const int bx = std::max(1, std::min(16, 2048 / (f.rows * rs)));
  const size_t lds = sizeof(double) * (size_t)bx * rs * (f.rows + 1);
  auto log2_up = [](int n) {
    int l = 0;
    while ((1 << l) < n) ++l;
    return l;
  };
  // lanes per (box, density): all values in flight if the lanes allow
  const int lw = std::max(2, std::min(6, log2_up((f.rows + kStageK - 1) / kStageK)));
  const int rl = std::min(8 - lw, log2_up(rs)), re = log2_up(rs);
  const int gl = std::min(6 - re, log2_up(f.d.kg));
  const dim3 grid((unsigned)((nb + bx) / bx), (unsigned)((R + t.Rc - 1) / t.Rc));
  hipLaunchKernelGGL(fold_stage_kernel, grid, dim3(256), lds, s, f.d, f.nm, f.cplx, f.rows, t.Rc, nb,
                     R, bx, rs, lw, rl, re, gl, f.slot_lut, fin, ldf, mode_point, box_starts,
                     box_alpha, box_disp, nmlz, log_disp, X, dl);
  return hipGetLastError();
}

namespace {
// groups of a parity with 0..nf odd axes; counts past nf repeat the last one
void odd_groups(const FoldDims& d, int g[4]) {
  for (int k = 0; k < 4; ++k) g[k] = groups_of(d, (1 << std::min(k, d.nf)) - 1);
}
}  // namespace

bool fold_has_kernel(const FoldDims& d) {
  int g[4];
  odd_groups(d, g);
  FoldParams none{};
  none.d = d;
  // no tiles: the launchers only look the instance up
  return (d.np == 8 ? fold_launch_3d(none, 1, g, nullptr) : fold_launch_2d(none, 1, g, nullptr)) ==
         hipSuccess;
}

hipError_t fold_contract_launch(const FoldParams& p, const FoldTile& t, hipStream_t s) {
  if (!fold_fits(p.d, p.nb, p.Rc)) return hipErrorInvalidValue;
  int g[4];
  odd_groups(p.d, g);
  return p.d.np == 8 ? fold_launch_3d(p, t.nct, g, s) : fold_launch_2d(p, t.nct, g, s);
}

}  // namespace vl1
