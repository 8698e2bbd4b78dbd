// Instantiations of the split GEMM kernel for dense operands with a prologue:
// the GroupNorm affine applied as the rows load, and the folded LayerNorm with
// its row statistics from the producer's partials.
#include "gemm_split.hpp"

namespace mh {
namespace gemm {

bool launch_split_dense_pro(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi) {
    return launch_split<kDense, kProAffine>(ctx, p, wt, epi, 1);
}

bool launch_split_dense_ln(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi) {
    return p.lnp_in && launch_split<kDense, kProLnPart>(ctx, p, wt, epi, 1);
}

}  // namespace gemm
}  // namespace mh
