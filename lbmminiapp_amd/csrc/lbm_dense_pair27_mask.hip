// lbm_dense_pair27_mask.hip -- instantiates the D3Q27 two-step kernels for masked boxes.
#include "lbm_dense_pair.hpp"

namespace lbm {
PairKernel pick_pair27_mask(int storage, bool force, bool nt, bool narrow, bool small, int v) {
  return pick_pair_q<27, true>(storage, force, nt, narrow, small, v);
}
}  // namespace lbm
