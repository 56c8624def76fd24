// lbm_dense_pair27.hip -- instantiates the D3Q27 two-step kernels.
#include "lbm_dense_pair.hpp"

namespace lbm {
PairKernel pick_pair27(int storage, bool force, bool nt, bool narrow, bool small, int v) {
  return pick_pair_q<27, false>(storage, force, nt, narrow, small, v);
}
}  // namespace lbm
