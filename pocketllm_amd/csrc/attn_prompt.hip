// Attention of several new tokens per sequence against a key/value store (a prompt, or its continuation), three launches:
//     1. RMS normalisation of q and k over their whole width, rotary phases, the new keys and values into their stores (a workgroup per token);
//     2. the values of positions 0 .. length - 1 turned into rows of positions per head dimension;
//     3. causal grouped-query softmax attention on the 16-bit matrix cores with a running maximum, nothing of size steps x length in memory.
// What the reference does between its q / k / v projections and its output projection (src/models/minimax_m2/architecture.py:158-266).
// As framework operators steps 1 and 2 were 18 launches that moved the rows through memory ten times (1024 tokens of 48 / 8 heads: 110 us,
// here 17), and step 3 ran in the framework's library (85.8 us, here 38).
//
// Step 3: a workgroup of four waves takes 128 queries of a head, a wave 32 of them; 64 keys and values at a time come to LDS by
// direct-to-LDS loads, double-buffered.  The wave forms S^T = K Q^T (v_mfma_f32_32x32x16: matrix rows are keys, columns are queries), so a
// lane holds half of one query's scores: maximum and sum are registers and one exchange with the lane of the other half, and what
// the score product leaves in a lane is, rounded to 16 bits, what O^T = V^T P^T wants from it as its second operand: within 16 keys, lane
// half h holds keys 4 h .. 4 h + 3 and 8 + 4 h .. 8 + 4 h + 3.  The rows of step 2 hold their positions in that order.  Each tile costs a wave
// 32 matrix instructions, 32 KB of LDS reads and 32 exponentials per lane, which take a compute unit about the same time each.
// 16-byte pieces of a row lie permuted in LDS (key rows: by row % 16, value rows: by row / 2 % 8), so 16 neighbouring rows read at one
// piece meet no bank twice.  The longest query blocks start first; the heads of a group, which share keys, run on one XCD.
// A block's time is the chain of its tiles.  Two groups of waves that take every other tile where blocks leave places free (1024 tokens of 48 and 8 heads, all
// three steps: 50.4 -> 44.5 us; 128 behind 2000: 69.7 -> 52.4) round the softmax weights against other maxima: a sequence's outputs would then depend on the
// batch that it is in, and lanes of the second group that see no key send the whole wave through the products for very large scores.
#include "block_mfma.h"
#include "pllm_internal.h"

#include <float.h>
#include <math.h>

namespace pllm {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kDim = 128;                       // head dimension
constexpr int kTile = 64;                       // keys per step
constexpr int kMaxHeads = 64, kMaxKvHeads = 32;
constexpr int kRowThreads = 256, kQPieces = kMaxHeads * kDim / (8 * kRowThreads), kKPieces = kMaxKvHeads * kDim / (8 * kRowThreads);
constexpr int kWaves = 4, kBlockRows = 32 * kWaves;
constexpr int kTileBytes = kTile * kDim * 2;

struct PromptArgs {
    const uint16_t* q;                          // [batch * steps][heads * 128], as the projection left it
    const uint16_t* k;
    const uint16_t* v;
    const float* q_weight;                      // null: no normalisation
    const float* k_weight;
    const float* cos_rows;                      // [steps][128], null: no rotary part
    const float* sin_rows;
    uint16_t* k_store;
    uint16_t* v_store;
    uint16_t* q_rows;                           // workspace: q normalized and turned
    uint16_t* v_turned;                         // workspace: [batch * kv_heads][128][padded]
    uint16_t* out;
    size_t batch_stride, head_stride;           // of the stores, in elements
    float eps;
    int batch, steps, heads, kv_heads, first_pos, padded, rope_half;
};

template <bool BF16> __device__ __forceinline__ float half_value(uint32_t bits) {
    if constexpr (BF16) return __uint_as_float(bits << 16);
    else return f16_bits_to_float(bits);
}
template <bool BF16> __device__ __forceinline__ uint32_t half_pair(float a, float b) {
    if constexpr (BF16) {
        typedef __bf16 v2b __attribute__((ext_vector_type(2)));
        const v2b p = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
        return __builtin_bit_cast(uint32_t, p);
    } else {
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        const v2h p = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
        return __builtin_bit_cast(uint32_t, p);
    }
}
template <bool BF16> __device__ __forceinline__ float round_to_store(float v) {
    if constexpr (BF16) return static_cast<float>(static_cast<__bf16>(v));
    else return static_cast<float>(static_cast<_Float16>(v));
}
template <bool BF16> __device__ __forceinline__ v16f prompt_mfma(uint4 a, uint4 b, v16f c) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// One token: q and k normalized and turned, k and v into the stores.  IN_BF16: the type of q, k and v as they come; BF16: that of the stores and
// of what leaves.  Float32 arithmetic; the normalized values are rounded to the stores' type before they turn, where the separate
// operators (and the decode step) round.
template <bool IN_BF16, bool BF16>
__global__ __launch_bounds__(kRowThreads) void attn_prompt_rows_kernel(PromptArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[8];
    float* rows = reinterpret_cast<float*>(smem);                    // the q row, then the k row
    const int token = blockIdx.x, b = token / a.steps, s = token % a.steps, tid = threadIdx.x;
    const int qw = a.heads * kDim, kw = a.kv_heads * kDim;
    const uint16_t* q = a.q + static_cast<size_t>(token) * qw;
    const uint16_t* k = a.k + static_cast<size_t>(token) * kw;
    const uint16_t* v = a.v + static_cast<size_t>(token) * kw;
    uint4 qp[kQPieces], kp[kKPieces], vp[kKPieces];
    // everything the token needs in one batch of loads: the rows, the weights behind them, the phases of the thread's place in a head (asked for where
    // they are used, 1024 tokens of 48 and 8 heads took 22.1 us, this way 12.3)
    const int d0 = (8 * tid) % kDim;
    const bool inside = d0 < 2 * a.rope_half, eights = a.rope_half % 8 == 0;
    float4 qg[kQPieces][2], kg[kKPieces][2], cs[4];
    const auto pair = [](const float* p, float4* o) {                // (weights and phases may begin at any value)
        typedef float v4w __attribute__((ext_vector_type(4), aligned(4)));
        const v4w lo = *reinterpret_cast<const v4w*>(p), hi = *reinterpret_cast<const v4w*>(p + 4);
        o[0] = make_float4(lo[0], lo[1], lo[2], lo[3]);
        o[1] = make_float4(hi[0], hi[1], hi[2], hi[3]);
    };
#pragma unroll
    for (int i = 0; i < kQPieces; ++i)
        if (8 * kRowThreads * i < qw) qp[i] = *reinterpret_cast<const uint4*>(q + min(8 * (tid + kRowThreads * i), qw - 8));
#pragma unroll
    for (int i = 0; i < kKPieces; ++i)
        if (8 * kRowThreads * i < kw) {
            kp[i] = *reinterpret_cast<const uint4*>(k + min(8 * (tid + kRowThreads * i), kw - 8));
            vp[i] = *reinterpret_cast<const uint4*>(v + min(8 * (tid + kRowThreads * i), kw - 8));
        }
    if (a.q_weight)
#pragma unroll
        for (int i = 0; i < kQPieces; ++i)
            if (8 * kRowThreads * i < qw) pair(a.q_weight + min(8 * (tid + kRowThreads * i), qw - 8), qg[i]);
    if (a.k_weight)
#pragma unroll
        for (int i = 0; i < kKPieces; ++i)
            if (8 * kRowThreads * i < kw) pair(a.k_weight + min(8 * (tid + kRowThreads * i), kw - 8), kg[i]);
    if (a.rope_half > 0) {
        pair(a.cos_rows + static_cast<size_t>(s) * kDim + d0, cs);
        pair(a.sin_rows + static_cast<size_t>(s) * kDim + d0, cs + 2);
    }
    auto value = [](const uint4& p, int j) {
        const uint32_t w = j < 2 ? p.x : j < 4 ? p.y : j < 6 ? p.z : p.w;
        return half_value<IN_BF16>((j & 1) ? w >> 16 : w & 0xffffu);
    };
    float sq = 0.0f, sk = 0.0f;
#pragma unroll
    for (int i = 0; i < kQPieces; ++i)
        if (8 * (tid + kRowThreads * i) < qw)
#pragma unroll
            for (int j = 0; j < 8; ++j) sq += value(qp[i], j) * value(qp[i], j);
#pragma unroll
    for (int i = 0; i < kKPieces; ++i)
        if (8 * (tid + kRowThreads * i) < kw)
#pragma unroll
            for (int j = 0; j < 8; ++j) sk += value(kp[i], j) * value(kp[i], j);
    sq = group_sum<64>(sq);
    sk = group_sum<64>(sk);
    if ((tid & 63) == 0) { red[tid >> 6] = sq; red[4 + (tid >> 6)] = sk; }
    __syncthreads();
    sq = (red[0] + red[1]) + (red[2] + red[3]);
    sk = (red[4] + red[5]) + (red[6] + red[7]);
    const float rq = a.q_weight ? rsqrtf(sq / static_cast<float>(qw) + a.eps) : 1.0f, rk = a.k_weight ? rsqrtf(sk / static_cast<float>(kw) + a.eps) : 1.0f;
    const auto component = [](const float4* v, int j) { const float4 f = v[j >> 2]; return (j & 3) == 0 ? f.x : (j & 3) == 1 ? f.y : (j & 3) == 2 ? f.z : f.w; };
    auto normalize = [&](const uint4& p, int at, float r, bool on, const float4* weight, float* row) {
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = round_to_store<BF16>(on ? value(p, j) * r * component(weight, j) : value(p, j));
        *reinterpret_cast<float4*>(row + at) = make_float4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<float4*>(row + at + 4) = make_float4(o[4], o[5], o[6], o[7]);
    };
#pragma unroll
    for (int i = 0; i < kQPieces; ++i)
        if (8 * (tid + kRowThreads * i) < qw) normalize(qp[i], 8 * (tid + kRowThreads * i), rq, a.q_weight != nullptr, qg[i], rows);
#pragma unroll
    for (int i = 0; i < kKPieces; ++i)
        if (8 * (tid + kRowThreads * i) < kw) normalize(kp[i], 8 * (tid + kRowThreads * i), rk, a.k_weight != nullptr, kg[i], rows + qw);
    __syncthreads();
    // values `at` .. at + 7 of a row (all in one head) turned by the token's phases; their partners are eight neighbours too where the rotary
    // part is a multiple of 16 (read value by value they meet the same banks eight at a time: 28.1 us for 1024 tokens, this way 23.0)
    auto eight = [](const float* p, float* o) {
        const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
        o[0] = lo.x; o[1] = lo.y; o[2] = lo.z; o[3] = lo.w; o[4] = hi.x; o[5] = hi.y; o[6] = hi.z; o[7] = hi.w;
    };
    auto turned = [&](const float* row, int at) {
        float o[8], other[8];
        eight(row + at, o);
        if (inside) {
            if (eights) {
                eight(row + (d0 < a.rope_half ? at + a.rope_half : at - a.rope_half), other);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int d = d0 + j;
                    other[j] = row[at - d0 + (d < a.rope_half ? d + a.rope_half : (d < 2 * a.rope_half ? d - a.rope_half : d))];
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf(other[j], component(cs + 2, j), o[j] * component(cs, j));
        }
        return make_uint4(half_pair<BF16>(o[0], o[1]), half_pair<BF16>(o[2], o[3]), half_pair<BF16>(o[4], o[5]), half_pair<BF16>(o[6], o[7]));
    };
#pragma unroll
    for (int i = 0; i < kQPieces; ++i) {
        const int at = 8 * (tid + kRowThreads * i);
        if (at < qw) *reinterpret_cast<uint4*>(a.q_rows + static_cast<size_t>(token) * qw + at) = turned(rows, at);
    }
#pragma unroll
    for (int i = 0; i < kKPieces; ++i) {
        const int at = 8 * (tid + kRowThreads * i);
        if (at >= kw) continue;
        const size_t o = static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(at / kDim) * a.head_stride + static_cast<size_t>(a.first_pos + s) * kDim + at % kDim;
        *reinterpret_cast<uint4*>(a.k_store + o) = turned(rows + qw, at);
        *reinterpret_cast<uint4*>(a.v_store + o) =
            IN_BF16 == BF16 ? vp[i] : make_uint4(half_pair<BF16>(value(vp[i], 0), value(vp[i], 1)), half_pair<BF16>(value(vp[i], 2), value(vp[i], 3)),
                                                 half_pair<BF16>(value(vp[i], 4), value(vp[i], 5)), half_pair<BF16>(value(vp[i], 6), value(vp[i], 7)));
    }
}

// 64 positions of one key/value head: [position][dimension] -> [dimension][position], the positions of every 16 in operand order,
// zeros behind the last one.
__global__ __launch_bounds__(256) void attn_prompt_turn_kernel(PromptArgs a) {
    constexpr int kPitch = kDim + 2;
    __shared__ uint32_t tile[kTile * kPitch / 2];
    const int p0 = blockIdx.x * kTile, kvh = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, length = a.first_pos + a.steps;
    const uint16_t* src = a.v_store + static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(kvh) * a.head_stride;
    const int row = tid >> 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int piece = (tid & 3) + 4 * i;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (p0 + row < length) v = *reinterpret_cast<const uint4*>(src + static_cast<size_t>(p0 + row) * kDim + 8 * piece);
        uint32_t* t = tile + row * (kPitch / 2) + 4 * piece;
        t[0] = v.x; t[1] = v.y; t[2] = v.z; t[3] = v.w;
    }
    __syncthreads();
    const uint16_t* halves = reinterpret_cast<const uint16_t*>(tile);
    const int d = tid >> 1;
    uint16_t* dst = a.v_turned + ((static_cast<size_t>(b) * a.kv_heads + kvh) * kDim + d) * a.padded + p0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int piece = 4 * (tid & 1) + i, first = 16 * (piece >> 1) + 4 * (piece & 1);    // lane half piece % 2 of keys 16 (piece / 2) ..
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = first + 2 * (j & 1) + 8 * (j >> 1);
            w[j] = halves[k * kPitch + d] | (static_cast<uint32_t>(halves[(k + 1) * kPitch + d]) << 16);
        }
        *reinterpret_cast<uint4*>(dst + 8 * piece) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

template <bool BF16>
__global__ __launch_bounds__(64 * kWaves, 2) void attn_prompt_kernel(PromptArgs a) {
    extern __shared__ __align__(1024) unsigned char smem[];          // [2][64 keys, then 64 positions of the turned values]
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int head = a.heads % 8 == 0 ? static_cast<int>(blockIdx.x & 7) * (a.heads / 8) + static_cast<int>(blockIdx.x >> 3) : static_cast<int>(blockIdx.x);
    const int kvh = head / (a.heads / a.kv_heads), b = blockIdx.z;
    const int block0 = static_cast<int>(gridDim.y - 1 - blockIdx.y) * kBlockRows, q0 = block0 + 32 * wave;
    const int length = a.first_pos + a.steps;
    const int tiles = (a.first_pos + min(a.steps, block0 + kBlockRows) + kTile - 1) / kTile;
    const int wave_end = q0 < a.steps ? a.first_pos + min(a.steps, q0 + 32) : 0;             // keys below this are seen by one of the wave's queries
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte_ptr)smem));
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(a.k_store + static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(kvh) * a.head_stride);
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(a.v_turned + (static_cast<size_t>(b) * a.kv_heads + kvh) * kDim * a.padded);
    auto fetch = [&](int t, int buf) {
        const uint32_t dst = lds0 + buf * 2 * kTileBytes + wave * (kTileBytes / kWaves);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 16 * wave + 4 * i + (lane >> 4), key = min(kTile * t + row, length - 1);
            lds_dma16_at(kbase, static_cast<uint32_t>(key) * (2 * kDim) + 16u * ((lane & 15) ^ (row & 15)), dst + 1024 * i);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 32 * wave + 8 * i + (lane >> 3);
            lds_dma16_at(vbase, static_cast<uint32_t>(d) * (2u * a.padded) + 2u * kTile * t + 16u * ((lane & 7) ^ ((d >> 1) & 7)), dst + kTileBytes + 1024 * i);
        }
    };
    fetch(0, 0);
    uint4 qf[8];
    {
        const uint16_t* q = a.q_rows + (static_cast<size_t>(b) * a.steps + min(q0 + r, a.steps - 1)) * a.heads * kDim + head * kDim + 8 * h;
#pragma unroll
        for (int i = 0; i < 8; ++i) qf[i] = *reinterpret_cast<const uint4*>(q + 16 * i);
    }
    const float scale = 0.08838834764831845f * 1.4426950408889634f;  // 1 / sqrt(128), base 2
    const v16f zero = {};
    v16f o[4] = {zero, zero, zero, zero};
    float m = -FLT_MAX, l = 0.0f;                                      // of the lane's query; l over its half of the keys
    wait_vm<0>();
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        if (t + 1 < tiles) fetch(t + 1, (t + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        if (kTile * t < wave_end) {
            const unsigned char* kt = smem + (t & 1) * 2 * kTileBytes;
            const unsigned char* vt = kt + kTileBytes;
            v16f s[2];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint4 kf = *reinterpret_cast<const uint4*>(kt + (32 * u + r) * (2 * kDim) + (((2 * i + h) ^ (r & 15)) << 4));
                    s[u] = prompt_mfma<BF16>(kf, qf[i], i == 0 ? zero : s[u]);
                }
            if (kTile * t + kTile - 1 > a.first_pos + q0) {           // keys behind a query (wave-uniform test)
                const int seen = a.first_pos + q0 + r - kTile * t - 4 * h;
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        if (32 * u + 8 * (v >> 2) + (v & 3) > seen) s[u][v] = -INFINITY;
            }
            float top = fmaxf(s[0][0], s[1][0]);
#pragma unroll
            for (int v = 1; v < 16; ++v) top = fmaxf(top, fmaxf(s[0][v], s[1][v]));
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(top), __float_as_uint(top), false, false);
            const float m_new = fmaxf(m, fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * scale);
            if (__any(m_new > m)) {
                const float back = __builtin_amdgcn_exp2f(m - m_new);
                l *= back;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[i][v] *= back;
                m = m_new;
            }
            // The fused product keeps the bits that the maximum's own rounding lost: up to 2^-25 of it, the same factor in every weight of a
            // query, which goes again with the division by their sum, but past the exponent's range from 2^31 on.  Scores that far out
            // are multiplied and rounded first.
            float factor = scale;
            if (__any(fabsf(m) > 0x1p20f)) {
                factor = 1.0f;
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[u][v] *= scale;
            }
            uint4 p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i >> 1][8 * (i & 1) + j], factor, -m));
                l += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
                p[i] = make_uint4(half_pair<BF16>(e[0], e[1]), half_pair<BF16>(e[2], e[3]), half_pair<BF16>(e[4], e[5]), half_pair<BF16>(e[6], e[7]));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint4 vf = *reinterpret_cast<const uint4*>(vt + (32 * u + r) * (2 * kTile) + (((2 * i + h) ^ ((r >> 1) & 7)) << 4));
                    o[u] = prompt_mfma<BF16>(vf, p[i], o[u]);
                }
        }
        wait_vm<0>();
        __syncthreads();                                              // the next tile is there, this one has been read
    }
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    const float inv = 1.0f / (__uint_as_float(halves[0]) + __uint_as_float(halves[1]));
    // lane: query r, dimensions 32 u + 8 (v / 4) + 4 h + v % 4; through the wave's own 8 KB to rows of 256 bytes
    unsigned char* turn = smem + wave * (32 * 2 * kDim);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<uint2*>(turn + r * (2 * kDim) + (((4 * u + g) ^ (r & 15)) << 4) + 8 * h) =
                make_uint2(half_pair<BF16>(o[u][4 * g] * inv, o[u][4 * g + 1] * inv), half_pair<BF16>(o[u][4 * g + 2] * inv, o[u][4 * g + 3] * inv));
    __builtin_amdgcn_wave_barrier();                                  // (one wave's LDS operations take effect in order)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = 4 * i + (lane >> 4), piece = lane & 15;
        const uint4 v = *reinterpret_cast<const uint4*>(turn + row * (2 * kDim) + ((piece ^ (row & 15)) << 4));
        if (q0 + row < a.steps) *reinterpret_cast<uint4*>(a.out + (static_cast<size_t>(b) * a.steps + q0 + row) * a.heads * kDim + head * kDim + 8 * piece) = v;
    }
}

template <bool BF16>
int launch_prompt(const PromptArgs& a, bool in_bf16, hipStream_t stream) {
    static SmemGrant granted;
    const size_t smem = 4 * kTileBytes;
    if (!grant_dynamic_smem(reinterpret_cast<const void*>(attn_prompt_kernel<BF16>), smem, granted)) return PLLM_ERR_UNSUPPORTED;
    auto rows = in_bf16 ? attn_prompt_rows_kernel<true, BF16> : attn_prompt_rows_kernel<false, BF16>;
    hipLaunchKernelGGL(rows, dim3(a.batch * a.steps), dim3(kRowThreads), (a.heads + a.kv_heads) * kDim * sizeof(float), stream, a);
    if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    hipLaunchKernelGGL(attn_prompt_turn_kernel, dim3(a.padded / kTile, a.kv_heads, a.batch), dim3(256), 0, stream, a);
    if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    hipLaunchKernelGGL(attn_prompt_kernel<BF16>, dim3(a.heads, (a.steps + kBlockRows - 1) / kBlockRows, a.batch), dim3(64 * kWaves), smem, stream, a);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

int padded_positions(int64_t length) { return static_cast<int>((length + kTile - 1) / kTile * kTile); }
size_t q_rows_bytes(int64_t batch, int64_t steps, int64_t heads) { return align256(static_cast<size_t>(batch) * steps * heads * kDim * 2); }

}  // namespace
}  // namespace pllm

extern "C" {

size_t pllm_attention_prompt_workspace_bytes(int64_t batch, int64_t steps, int64_t heads, int64_t kv_heads, int64_t first_pos) {
    if (batch <= 0 || steps <= 0 || heads <= 0 || kv_heads <= 0 || first_pos < 0) return 0;
    return pllm::q_rows_bytes(batch, steps, heads) + static_cast<size_t>(batch) * kv_heads * pllm::kDim * pllm::padded_positions(first_pos + steps) * 2;
}

int pllm_attention_prompt(const void* q, const void* k_new, const void* v_new, int new_dtype, int dtype, const float* q_norm_weight, const float* k_norm_weight, float eps,
                          const float* cos_rows, const float* sin_rows, int64_t rope_dim, void* k_store, void* v_store, int64_t store_batch_stride,
                          int64_t store_head_stride, int64_t batch, int64_t steps, int64_t heads, int64_t kv_heads, int64_t head_dim, int64_t first_pos,
                          void* out, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace pllm;
    if (!q || !k_new || !v_new || !k_store || !v_store || !out || (dtype != PLLM_F16 && dtype != PLLM_BF16) || (new_dtype != PLLM_F16 && new_dtype != PLLM_BF16))
        return PLLM_ERR_INVALID_ARGUMENT;
    if (batch <= 0 || steps <= 0 || heads <= 0 || kv_heads <= 0 || first_pos < 0 || rope_dim < 0 || (rope_dim > 0 && (!cos_rows || !sin_rows)))
        return PLLM_ERR_INVALID_ARGUMENT;
    if (store_batch_stride < 0 || store_head_stride < (first_pos + steps) * head_dim) return PLLM_ERR_INVALID_ARGUMENT;
    // 32-bit offsets inside a head's rows, one workgroup per token and one grid row per sequence
    if (head_dim != kDim || heads > kMaxHeads || kv_heads > kMaxKvHeads || heads % kv_heads != 0 || rope_dim > kDim || rope_dim % 2 != 0 || batch > 65535 ||
        first_pos + steps > 131072 || batch * steps > 0x7fffffff)
        return PLLM_ERR_UNSUPPORTED;
    const uintptr_t align = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_new) | reinterpret_cast<uintptr_t>(v_new) |
                            reinterpret_cast<uintptr_t>(k_store) | reinterpret_cast<uintptr_t>(v_store) | reinterpret_cast<uintptr_t>(out);
    if ((align & 15u) != 0 || store_batch_stride % 8 != 0 || store_head_stride % 8 != 0) return PLLM_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < pllm_attention_prompt_workspace_bytes(batch, steps, heads, kv_heads, first_pos)) return PLLM_ERR_WORKSPACE;
    PromptArgs a{};
    a.q = static_cast<const uint16_t*>(q);
    a.k = static_cast<const uint16_t*>(k_new);
    a.v = static_cast<const uint16_t*>(v_new);
    a.q_weight = q_norm_weight;
    a.k_weight = k_norm_weight;
    a.cos_rows = cos_rows;
    a.sin_rows = sin_rows;
    a.k_store = static_cast<uint16_t*>(k_store);
    a.v_store = static_cast<uint16_t*>(v_store);
    a.q_rows = static_cast<uint16_t*>(workspace);
    a.v_turned = reinterpret_cast<uint16_t*>(static_cast<unsigned char*>(workspace) + q_rows_bytes(batch, steps, heads));
    a.out = static_cast<uint16_t*>(out);
    a.batch_stride = static_cast<size_t>(store_batch_stride);
    a.head_stride = static_cast<size_t>(store_head_stride);
    a.eps = eps;
    a.batch = static_cast<int>(batch);
    a.steps = static_cast<int>(steps);
    a.heads = static_cast<int>(heads);
    a.kv_heads = static_cast<int>(kv_heads);
    a.first_pos = static_cast<int>(first_pos);
    a.padded = padded_positions(first_pos + steps);
    a.rope_half = static_cast<int>(rope_dim / 2);
    return dtype == PLLM_BF16 ? launch_prompt<true>(a, new_dtype == PLLM_BF16, static_cast<hipStream_t>(stream)) : launch_prompt<false>(a, new_dtype == PLLM_BF16, static_cast<hipStream_t>(stream));
}

}  // extern "C"
