// The prompt tile kernel over the codebook formats.
#include "gemm_tile.h"

namespace pllm {

int launch_tiles_codebook(int type_id, const TileCall& c, int nt, int workgroups, hipStream_t stream) {
    switch (type_id) {
        case PLLM_TYPE_IQ2_XXS: return launch_tiles<TIQ2XXS>(c, nt, workgroups, stream);
        case PLLM_TYPE_IQ2_XS: return launch_tiles<TIQ2XS>(c, nt, workgroups, stream);
        case PLLM_TYPE_IQ3_XXS: return launch_tiles<TIQ3XXS>(c, nt, workgroups, stream);
        case PLLM_TYPE_IQ1_M: return launch_tiles<TIQ1M>(c, nt, workgroups, stream);
        default: return PLLM_ERR_UNSUPPORTED;
    }
}

}  // namespace pllm
