// Instantiations of the split GEMM kernel for the 3x3 conv's gathered A operand,
// with and without the GroupNorm prologue.
#include "gemm_split.hpp"

namespace mh {
namespace gemm {

bool launch_split_conv(Context &ctx, GemmArgs &p, WeightType wt, int mode, bool pro) {
    switch (mode) {
        case kConvAligned:
            return pro ? launch_split<kConvAligned, kProAffine>(ctx, p, wt, GemmEpilogue::None, 1)
                       : launch_split<kConvAligned, kProNone>(ctx, p, wt, GemmEpilogue::None, 1);
        case kConvVec:
            return pro ? launch_split<kConvVec, kProAffine>(ctx, p, wt, GemmEpilogue::None, 1)
                       : launch_split<kConvVec, kProNone>(ctx, p, wt, GemmEpilogue::None, 1);
        default:
            return false;
    }
}

}  // namespace gemm
}  // namespace mh
