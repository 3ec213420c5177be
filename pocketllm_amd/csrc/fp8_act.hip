// FP8 activation quantizer: per (row, 128 values) s = max(amax, eps) / 448, optionally rounded up to
// a power of two, code = E4M3 (round to nearest even) of clamp(x / s, +-448).
#include "pllm_device.h"
#include "pllm_internal.h"

namespace pllm {
namespace {

constexpr int kThreads = 256;
constexpr size_t kMaxGrid = size_t{1} << 20;              // (more blocks than that: the groups walk on)

// Sixteen lanes per 128-value block, eight neighbouring values each.  Rows, codes and scales are contiguous and k is a multiple of
// 128, so the matrix is one sequence of blocks.  Large calls are bound by the bytes (2048 rows of 17408 bf16 values: 107 MB read and written
// in 20.7 us, 5.2 TB/s, what a large copy reaches), small ones by the start of a launch and the latency of one load (512 x 5120 bf16: 7.9 MB in
// 3.3 us back to back, 4.6 us as a call; one wave per block, two values per lane: 7.8).  A lane asks for its share in one 16-byte load (two for
// float32) and writes its codes in one 8-byte store.  WIDE needs x on 16 and codes on 8 bytes: other addresses (views the C entry is
// handed) go value by value, two codes per store.
template <int DT, bool WIDE>
__global__ __launch_bounds__(kThreads) void fp8_act_quant_kernel(
    const void* __restrict__ x, uint8_t* __restrict__ codes, float* __restrict__ scales, size_t blocks, float eps, int pow2) {
    const size_t stride = static_cast<size_t>(gridDim.x) * (kThreads / 16);
    for (size_t blk = static_cast<size_t>(blockIdx.x) * (kThreads / 16) + (threadIdx.x >> 4); blk < blocks; blk += stride) {
        const size_t base = blk * 128 + 8 * (threadIdx.x & 15);
        float v[8];
        if constexpr (!WIDE) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = load_any(x, DT, base + i);
        } else if constexpr (DT == PLLM_F32) {
            const float4 lo = *reinterpret_cast<const float4*>(static_cast<const float*>(x) + base);
            const float4 hi = *reinterpret_cast<const float4*>(static_cast<const float*>(x) + base + 4);
            v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
            v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
        } else {
            const uint4 raw = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(x) + base);
            const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t h = (i & 1) ? words[i / 2] >> 16 : words[i / 2] & 0xffffu;
                v[i] = DT == PLLM_BF16 ? __uint_as_float(h << 16) : f16_bits_to_float(h);
            }
        }
        float amax = fabsf(v[0]);
#pragma unroll
        for (int i = 1; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
        amax = group_max<16>(amax);                                          // (the sixteen lanes of a block leave the loop together)
        float s = fmaxf(amax, eps) / 448.0f;
        if (pow2) {
            int e;
            const float m = frexpf(fmaxf(s, 1.17549435e-38f), &e);          // s = m * 2^e, m in [0.5, 1)
            s = ldexpf(1.0f, m == 0.5f ? e - 1 : e);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = fminf(fmaxf(v[i] / s, -448.0f), 448.0f);
        int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false), hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], 0, false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
        if constexpr (WIDE) {
            *reinterpret_cast<uint2*>(codes + base) = make_uint2(static_cast<uint32_t>(lo), static_cast<uint32_t>(hi));
        } else {
            uint16_t* out = reinterpret_cast<uint16_t*>(codes + base);
            out[0] = static_cast<uint16_t>(lo); out[1] = static_cast<uint16_t>(static_cast<uint32_t>(lo) >> 16);
            out[2] = static_cast<uint16_t>(hi); out[3] = static_cast<uint16_t>(static_cast<uint32_t>(hi) >> 16);
        }
        if ((threadIdx.x & 15) == 0) scales[blk] = s;
    }
}

template <int DT>
void launch_fp8_act_quant(const void* x, uint8_t* codes, float* scales, size_t blocks, float eps, int pow2, hipStream_t stream) {
    const size_t groups = (blocks + kThreads / 16 - 1) / (kThreads / 16);
    const dim3 grid(static_cast<unsigned>(groups < kMaxGrid ? groups : kMaxGrid));
    const bool wide = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(codes) & 7u) == 0;
    if (wide) hipLaunchKernelGGL((fp8_act_quant_kernel<DT, true>), grid, dim3(kThreads), 0, stream, x, codes, scales, blocks, eps, pow2);
    else hipLaunchKernelGGL((fp8_act_quant_kernel<DT, false>), grid, dim3(kThreads), 0, stream, x, codes, scales, blocks, eps, pow2);
}

}  // namespace
}  // namespace pllm

extern "C" int pllm_fp8_act_quant(const void* x, int x_dtype, int64_t rows, int64_t k, uint8_t* codes, float* scales,
                                  float eps, int round_scale_pow2, void* stream) {
    if (!x || !codes || !scales || rows <= 0 || k <= 0 || (k % 128) != 0) return PLLM_ERR_INVALID_ARGUMENT;
    if (x_dtype != PLLM_F32 && x_dtype != PLLM_F16 && x_dtype != PLLM_BF16) return PLLM_ERR_INVALID_ARGUMENT;
    if (rows > 65535 || k / 128 > 0x7fffffffLL) return PLLM_ERR_UNSUPPORTED;
    const size_t blocks = static_cast<size_t>(rows) * static_cast<size_t>(k / 128);
    const hipStream_t st = static_cast<hipStream_t>(stream);
    if (x_dtype == PLLM_F32) pllm::launch_fp8_act_quant<PLLM_F32>(x, codes, scales, blocks, eps, round_scale_pow2, st);
    else if (x_dtype == PLLM_F16) pllm::launch_fp8_act_quant<PLLM_F16>(x, codes, scales, blocks, eps, round_scale_pow2, st);
    else pllm::launch_fp8_act_quant<PLLM_BF16>(x, codes, scales, blocks, eps, round_scale_pow2, st);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}
