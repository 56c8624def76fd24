// lbm_dense_pair19.hip -- instantiates the D3Q19 two-step kernels.
#include "lbm_dense_pair.hpp"

namespace lbm {
PairKernel pick_pair19(int storage, bool force, bool nt, bool narrow, bool small, int v) {
  return pick_pair_q<19, false>(storage, force, nt, narrow, small, v);
}
}  // namespace lbm
