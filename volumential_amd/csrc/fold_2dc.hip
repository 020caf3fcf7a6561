// Instances of the folded tile kernel with four parities: complex data and
// the largest real orders.
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

hipError_t fold_launch_2dc(const FoldParams& p, int nct, const int g[4], hipStream_t s) {
  switch (p.d.np << 20 | fold_key(g[0], g[1], g[2], g[3])) {
    case 4 << 20 | fold_key(2, 1, 1, 1): return pick<4, 2, 1, 1, 1>(p, nct, s);  // 2D q = 3 complex
    case 4 << 20 | fold_key(2, 2, 2, 2): return pick<4, 2, 2, 2, 2>(p, nct, s);  // 2D q = 4 complex
    case 4 << 20 | fold_key(5, 4, 2, 2): return pick<4, 5, 4, 2, 2>(p, nct, s);  // 2D q = 5 complex
    case 4 << 20 | fold_key(5, 5, 5, 5): return pick<4, 5, 5, 5, 5>(p, nct, s);  // 2D q = 6 complex
    case 4 << 20 | fold_key(8, 6, 5, 5): return pick<4, 8, 6, 5, 5>(p, nct, s);  // 2D q = 7 complex
    case 4 << 20 | fold_key(8, 8, 8, 8): return pick<4, 8, 8, 8, 8>(p, nct, s);  // 2D q = 10, q = 8 complex
    case 4 << 20 | fold_key(8, 5, 4, 4): return pick<4, 8, 5, 4, 4>(p, nct, s);  // 2D q = 9
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vl1
