// Instantiations of the split GEMM kernel for dense, K-contiguous A operands.
#include "gemm_split.hpp"

namespace mh {
namespace gemm {

bool launch_split_dense(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi, int batch) {
    return launch_split<kDense, kProNone>(ctx, p, wt, epi, batch);
}

}  // namespace gemm
}  // namespace mh
