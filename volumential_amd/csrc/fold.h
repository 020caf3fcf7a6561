// Reflection-folded FP64 list-1 contraction: layouts shared by the plan
// (plan.hip) and the kernels (fold_f64.hip).
//
// The blocks of an arithmetic-orbit table are invariant under the reflection
// of any axis: with R_J the reflection of the box nodes along the axes J,
//     M_{R_J v} = eps_J R_J M_v R_J,    eps_J = -1 per reflected derivative axis
// (v: case vector).  In the even/odd basis of each folded axis
// (e_i = x_i + x_{q-1-i}, o_i = x_i - x_{q-1-i}; the middle node of an odd q
// is its own even part) R_J is diagonal, (-1)^{|p & J|} on the component of
// parity p.  The up to 2^m list-1 sources of a target whose case vectors
// differ only in the signs of their m nonzero folded components (a "class")
// then sum to
//     Y[p ^ s ^ sp] += A_s[p] S_s[p],
//     S_s = sum_j (-1)^{popcount(j & s)} X_j   (Walsh-Hadamard over the 2^m
//           sign slots j, an absent source being zero),
// s running over the subsets of the nonzero axes and sp the derivative axes:
// each of the 2^m sums meets one (n / 2^d) square block per parity, where the
// unfolded form multiplies every source by the full n x n block.  On a
// uniform tree that is 1 / 2^d of the multiplications (27 n^2 / 8 in 3D,
// 9 n^2 / 4 in 2D per target and density), for one extra FP64 addition per
// axis and value on the way in and out.
#pragma once

#include <cstdint>
#include <vector>

#include "internal.h"

namespace vl1 {

constexpr int kFoldMaxGroups = 16;  // row groups of 4 per parity (64 rows)

// One entry of the folded basis: the sum over J in amask of
// (-1)^{popcount(par & J)} x[base + sum_{a in J} d[a]].
struct FoldSlot {
  int16_t base, d[3];
  uint8_t amask, par, valid, pad;
};

// One output row t of a box: 2^-shift sum over the parities p with row[p] >= 0
// of (-1)^{popcount(p & flips)} yhat[row[p]].
struct FoldOut {
  int16_t row[8];
  uint8_t flips, shift, pad[2];
};

// Shape of the folded basis.  Parity p has byte p of `groups_lo` groups of 4
// rows in the table blocks (its entries, padded); parities are ordered by
// falling size (nibble p of ppos: the place of parity p).
// K group kg = kgstart(round) + position enumerates (round, parity): round r
// holds the r-th group of the cnt(r) parities that have one.
struct FoldDims {
  int np = 0, nf = 0, kg = 0, rounds = 0;
  int rows4 = 0;  // 4 x row groups over all parities
  uint32_t ppos = 0, sp = 0;
  uint64_t groups_lo = 0;          // byte p: row groups of parity p
  uint64_t cnt = 0;                // nibble r: parities in round r
  uint64_t kgs[2] = {0, 0};        // byte r: first K group of round r
};

// A tile's place in the lists, and its first chunk words (one scalar load).
struct FoldTileInfo {
  int32_t step, n_steps, chunk, n_chunks;
  uint32_t words[4];
};

// The blocks themselves, for outputs that are not finite (fold_nonfinite): read
// through one pointer, so that the tile kernel keeps none of it in registers.
struct FoldBlocks {
  const FoldSlot* slots;   // [kg][4]
  const double* M;         // [blocks x n_rg][MP][KP]
  const int32_t* rep_blk;  // block of a class's representative
  int dim, q, MP, KP, n_rg, rg_size;
};

struct FoldParams {
  FoldDims d;
  int B, Rc, R;            // boxes per tile, densities per tile, densities in all
  int nb;                  // boxes; index nb of X holds zeros
  int n_box_tiles;
  int nm, cplx, rows;      // modes per box; rows per box (2 nm if complex)
  const FoldTileInfo* tiles;        // [n_box_tiles]
  const int32_t* tile_boxes;        // [n_box_tiles][B] target box or -1
  const uint32_t* chunks;           // chunk words, kFoldPad more at the end
  const int32_t* step_src;          // [n_steps + kFoldPad][B][np] source boxes (nb: none)
  const uint4* lut_u;               // [nonzero axes][maxc][parity][2] units of a wave
  const uint2* lut_l;               // [width][m][maxc][wave] K groups a wave loads (bytes)
  int maxc;
  int slot_doubles;                 // LDS slot (set by the launcher)
  const double* A;                 // [class][kg][16 x row groups]
  int64_t cls_stride;              // doubles per class
  const double* X;                 // [r chunk][nb + 1][kg][Rc][4], the 4 as k = 0 1 3 2
  const double* dl;                // [r chunk][nb + 1][Rc] log-term sums, or null
  const FoldOut* out;              // [rows]
  const int32_t* mode_point;
  double* y;
  int64_t ldy;
  const struct FoldBlocks* blocks;  // device: for outputs that are not finite
  double* est;                     // their densities' error estimates [R][2], or null
};

// A value of a density that is not finite makes all sums of its mirror nodes
// so.  Their places in X then hold the nodes' own values instead: infinities
// and NaN as they are, finite ones as this NaN.
constexpr double kFoldMax = 1.7976931348623157e308;
constexpr uint64_t kFoldFinite = 0x7ff8000000f01d00ull;

__device__ inline int reflect_node(int dim, int q, int node, int flips) {
  int out = 0, stride = 1;
  for (int a = dim - 1; a >= 0; --a) {
    const int i = node % q;
    node /= q;
    out += (((flips >> a) & 1) ? q - 1 - i : i) * stride;
    stride *= q;
  }
  return out;
}

// A chunk of a step: class, its nonzero folded axes z and their number m, the
// chunk within the step, and whether it is the step's first.
__host__ __device__ inline uint32_t fold_chunk_word(int cls, int z, int m, int c, bool first) {
  return (uint32_t)cls << 12 | (uint32_t)first << 11 | (uint32_t)m << 9 | (uint32_t)z << 6 | (uint32_t)c;
}
__host__ __device__ inline int fold_chunk_c(uint32_t w) { return (int)(w & 63); }
__host__ __device__ inline int fold_chunk_z(uint32_t w) { return (int)(w >> 6 & 7); }
__host__ __device__ inline int fold_chunk_m(uint32_t w) { return (int)(w >> 9 & 3); }
__host__ __device__ inline bool fold_chunk_first(uint32_t w) { return (w >> 11 & 1) != 0; }
__host__ __device__ inline int fold_chunk_cls(uint32_t w) { return (int)(w >> 12); }
constexpr int kFoldPad = 8;    // list entries the kernel may prefetch past the last tile
constexpr int kFoldUnits = 8;  // units per wave and chunk
// Chunks of a step with m nonzero axes: kFoldUnits >> m rounds each.
inline int fold_chunks(const FoldDims& d, int m) {
  return (d.rounds + (kFoldUnits >> m) - 1) / (kFoldUnits >> m);
}

struct FoldTile {
  int nct = 0, Rc = 0, B = 0;  // 16-column tiles; densities and boxes per tile
};

// The folded form of one plan: host geometry, device tables.
struct FoldPlan {
  FoldDims d;
  int nm = 0, cplx = 0, rows = 0;
  std::vector<FoldSlot> slots;  // [kg][4]
  std::vector<FoldOut> outs;    // [rows]
  std::vector<uint4> lut_u;
  std::vector<uint2> lut_l;
  int maxc = 0;
  DevBuf lut, A;  // lut: the tables, and the class lists of the build
  const FoldSlot* slot_lut = nullptr;  // device, in lut
  const FoldOut* out_lut = nullptr;
  const FoldBlocks* blocks = nullptr;
  const uint4* u_lut = nullptr;
  const uint2* l_lut = nullptr;
  int64_t cls_stride = 0;
  int n_cls = 0;
  // per class: nonzero folded axes, the plan block of its representative; per
  // plan key: class, negative folded axes, sign slot
  std::vector<uint8_t> zmask;
  std::vector<int32_t> rep_blk, key_cls, key_flips, key_slot;
  // list-1 classes per target: entry e in [start[t], start[t + 1])
  std::vector<int32_t> start, cls, src;  // src [entry][np], -1: none
};

// Folded basis of q^dim nodes (2 values per node if complex); false: sizes the
// kernel does not take.  `few_axes`: the basis with fewer folded axes that many
// columns are faster in, false where there is none.
bool fold_layout(FoldPlan& f, int dim, int q, int cplx, uint32_t sign_mask, bool few_axes = false);
// Whether the tile kernel's 32-bit byte offsets reach all nb boxes and the zero
// box at Rc densities per tile (a box holds kg K groups of 32 Rc bytes; a lane
// reads up to one box past its own offset).
inline bool fold_fits(const FoldDims& d, int nb, int Rc) {
  return ((uint64_t)nb + 2) * (uint64_t)d.kg * (uint64_t)Rc * 32 <= (uint64_t)1 << 32;
}
// Tile shape for R densities over n_tgt of nb boxes (16 nct columns; 0:
// choose); nb boxes must fit at one density per tile.
FoldTile fold_tile(const FoldDims& d, int nb, int n_tgt, int R, int nct = 0);
// X and dl sizes in doubles for one evaluation.
size_t fold_x_size(const FoldDims& d, const FoldTile& t, int nb, int R);
size_t fold_dl_size(const FoldTile& t, int nb, int R);
// A[class] from the representatives' blocks in M [blocks x n_rg][MP][KP], and
// *flag = 1 unless every key's block is the reflection of its class's
// representative by the folded axes key_flips[key], and every representative
// its own reflection along each folded axis on which its case vector is zero
// (the product has no terms between the parities of such an axis), to 1e-14 of
// the representative's largest entry.  Keeps M for outputs that are not finite.
// Returns after the device has finished.
hipError_t fold_build_launch(FoldPlan& f, int dim, int q, const double* M, int MP, int KP, int n_rg,
                             int rg_size, int32_t* flag, hipStream_t s);
hipError_t fold_stage_launch(const FoldPlan& f, const FoldTile& t, int nb, int R, const double* fin,
                             int64_t ldf, const int32_t* mode_point, const int32_t* box_starts,
                             const double* box_alpha, const double* box_disp, const double* nmlz,
                             int log_disp, double* X, double* dl, hipStream_t s);
hipError_t fold_contract_launch(const FoldParams& p, const FoldTile& t, hipStream_t s);
// ... by the group counts g[k] of a parity with k odd axes; hipErrorInvalidValue
// for counts without an instance
hipError_t fold_launch_2d(const FoldParams& p, int nct, const int g[4], hipStream_t s);
hipError_t fold_launch_2dc(const FoldParams& p, int nct, const int g[4], hipStream_t s);
hipError_t fold_launch_3d(const FoldParams& p, int nct, const int g[4], hipStream_t s);
hipError_t fold_launch_3dodd(const FoldParams& p, int nct, const int g[4], hipStream_t s);
bool fold_has_kernel(const FoldDims& d);

}  // namespace vl1
