// lbm_dense_pair19_mask.hip -- instantiates the D3Q19 two-step kernels for masked boxes.
#include "lbm_dense_pair.hpp"

namespace lbm {
PairKernel pick_pair19_mask(int storage, bool force, bool nt, bool narrow, bool small, int v) {
  return pick_pair_q<19, true>(storage, force, nt, narrow, small, v);
}
}  // namespace lbm
