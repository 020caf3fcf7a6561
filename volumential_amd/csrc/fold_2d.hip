// Instances of the folded tile kernel with at most four parities (real data,
// and 3D order 3 with fewer axes folded).
#include "fold_kernel.h"

namespace vl1 {

namespace {

template <int NP, int G0, int G1, int G2, int G3>
hipError_t pick(const FoldParams& p, int nct, hipStream_t s) {
  if (p.n_box_tiles == 0) return hipSuccess;
  if (nct == 1) return launch_fold<NP, 1, G0, G1, G2, G3>(p, s);
  if (nct == 2) return launch_fold<NP, 2, G0, G1, G2, G3>(p, s);
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t fold_launch_2d(const FoldParams& p, int nct, const int g[4], hipStream_t s) {
  switch (p.d.np << 20 | fold_key(g[0], g[1], g[2], g[3])) {
    case 1 << 20 | fold_key(1, 1, 1, 1): return pick<1, 1, 1, 1, 1>(p, nct, s);  // 2D q = 2
    case 1 << 20 | fold_key(8, 8, 8, 8): return pick<1, 8, 8, 8, 8>(p, nct, s);  // 3D q = 3, unfolded
    case 2 << 20 | fold_key(1, 1, 1, 1): return pick<2, 1, 1, 1, 1>(p, nct, s);  // 2D q = 2 complex, 3D q = 2
    case 4 << 20 | fold_key(1, 1, 1, 1): return pick<4, 1, 1, 1, 1>(p, nct, s);  // 2D q = 3, 4; 3D q = 2 complex
    case 4 << 20 | fold_key(4, 2, 1, 1): return pick<4, 4, 2, 1, 1>(p, nct, s);  // 2D q = 5
    case 4 << 20 | fold_key(4, 4, 4, 4): return pick<4, 4, 4, 4, 4>(p, nct, s);  // 2D q = 6, 7, 8
    case 4 << 20 | fold_key(6, 4, 2, 2): return pick<4, 6, 4, 2, 2>(p, nct, s);  // 3D q = 3 complex
    default: return fold_launch_2dc(p, nct, g, s);
  }
}

}  // namespace vl1
