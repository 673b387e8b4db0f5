// Instantiates the fused sampler for the GaussMany32 integrand: the
// dimensions that many_pays names.
#include "vgx_fused.h"

namespace vgx {

template <>
int launch_fused<GaussMany32>(const IterGeom& g, const FusedPtrs& io, const GaussMany32& fcn, int blocks,
                       size_t lds, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    switch (g.dim) {
        case 5: return launch_fused_dim<5>(g, io, fcn, blocks, lds, st, ev0, ev1);
        case 6: return launch_fused_dim<6>(g, io, fcn, blocks, lds, st, ev0, ev1);
        case 7: return launch_fused_dim<7>(g, io, fcn, blocks, lds, st, ev0, ev1);
        case 8: return launch_fused_dim<8>(g, io, fcn, blocks, lds, st, ev0, ev1);
        case 9: return launch_fused_dim<9>(g, io, fcn, blocks, lds, st, ev0, ev1);
        default: return VGX_EINVAL;
    }
}

}  // namespace vgx
