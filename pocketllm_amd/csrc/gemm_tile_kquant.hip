// The prompt tile kernel over Q2_K, Q4_K, Q5_K, Q6_K, IQ4_XS and FP8 weights.
#include "gemm_tile.h"

namespace pllm {

int launch_tiles_kquant(int type_id, const TileCall& c, int nt, int workgroups, hipStream_t stream) {
    switch (type_id) {
        case PLLM_TYPE_Q4_K: return launch_tiles<TQ4K>(c, nt, workgroups, stream);
        case PLLM_TYPE_Q5_K: return launch_tiles<TQ5K>(c, nt, workgroups, stream);
        case PLLM_TYPE_Q2_K: return launch_tiles<TQ2K>(c, nt, workgroups, stream);
        case PLLM_TYPE_Q6_K: return launch_tiles<TQ6K>(c, nt, workgroups, stream);
        case PLLM_TYPE_IQ4_XS: return launch_tiles<TIQ4XS>(c, nt, workgroups, stream);
        case kFp8Tiles: return launch_tiles<TFP8, false>(c, nt, workgroups, stream);
        default: return PLLM_ERR_UNSUPPORTED;
    }
}

}  // namespace pllm
