// Instances of the folded tile kernel with eight parities, even orders (and
// order 3).
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

hipError_t fold_launch_3d(const FoldParams& p, int nct, const int g[4], hipStream_t s) {
  switch (p.d.np << 20 | fold_key(g[0], g[1], g[2], g[3])) {
    case 8 << 20 | fold_key(2, 1, 1, 1): return pick<8, 2, 1, 1, 1>(p, nct, s);  // q = 3
    case 8 << 20 | fold_key(2, 2, 2, 2): return pick<8, 2, 2, 2, 2>(p, nct, s);  // q = 4
    case 8 << 20 | fold_key(8, 8, 8, 8): return pick<8, 8, 8, 8, 8>(p, nct, s);  // q = 6
    case 8 << 20 | fold_key(16, 16, 16, 16): return pick<8, 16, 16, 16, 16>(p, nct, s);  // q = 8
    case 8 << 20 | fold_key(4, 4, 4, 4): return pick<8, 4, 4, 4, 4>(p, nct, s);  // q = 4 complex
    case 8 << 20 | fold_key(14, 14, 14, 14): return pick<8, 14, 14, 14, 14>(p, nct, s);  // q = 6 complex
    default: return fold_launch_3dodd(p, nct, g, s);
  }
}

}  // namespace vl1
