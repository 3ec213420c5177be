// Attention of one new token per sequence against a key/value store (decode step), two launches:
//     RMS normalisation of q and k over the whole projection width, rotary phases, store of the new key / value row,
//     scores against slices of 64 stored keys, softmax statistics and the weighted value sums of a run of slices;
//     then the runs of a head are merged (the usual running-maximum form of a split softmax).
// What the reference does between its q / k / v projections and its output projection (src/models/minimax_m2/
// architecture.py:158-266: q_norm, k_norm, apply_rotary_emb, cache update, scaled_dot_product_attention with the key/value
// heads shared by groups of query heads), for one query position.  None of it is quantized; it is here because a decoder
// block's step was dominated by the ~17 small framework launches this replaces, not by its matmuls.
//
// Layout: q [batch, heads * 128], k_new / v_new [batch, kv_heads * 128] in fp16 or bf16; stores [batch, kv_heads, capacity, 128]
// of the same type (batch and head strides in elements); out [batch, heads * 128].  Head dimension 128, up to 8 query heads per
// key/value head.  Arithmetic in float32 on the stored 16-bit values; the new key is rounded to the store's type before it is
// used, so a later step reads the same bits this step multiplied with.
//
// A workgroup of eight waves owns one or more runs of slices of 64 keys, one after the other: keys and values of the next slice are on their way while this one's are used.  Scores are
// matrix products of the 16-bit values (exact, float32 sums; the scale goes on behind them), softmax weights and value sums plain float32.
// Bound: short contexts by the two launches and the chain of one slice (loads, norm, five barriers), long ones by HBM (2 x length x kv_heads x 256 B:
// 100001 positions 4.3 TB/s).  us with both launches, replayed; four waves, scores by multiply-adds and a slice per workgroup / this form, 48 query and 8 key/value
// heads, bf16: 64 positions 7.9 / 6.1, 2048 11.1 / 9.4, 4096 13.5 / 11.5, 16384 42.2 / 22.5, 100001 245 / 95, sixteen rows of 1024 37.8 / 22.5; 64 and 8, four rows of
// 8192: 138 / 40.4; 32 and 32 heads, 701 positions 9.2 / 9.3.
#include "pllm_device.h"
#include "pllm_internal.h"

#include <algorithm>
#include <cfloat>

namespace pllm {
namespace {

constexpr int kHeadDim = 128;
constexpr int kSliceKeys = 64;
constexpr int kMaxGroup = 8;
constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kMaxHeads = 64;                  // q rows of up to 64 x 128 values (two 16-byte pieces per thread)
constexpr int kQPieces = kMaxHeads * kHeadDim / (8 * kThreads), kKPieces = 1;   // k rows of up to 32 x 128 values
constexpr int kPartFloats = kHeadDim + 2;     // a slice's result per query head: 128 weighted sums, running maximum, sum of weights

template <bool BF16> struct HalfBits {
    static __device__ __forceinline__ float to_float(uint32_t bits) {
        if constexpr (BF16) return __uint_as_float(bits << 16);
        else return f16_bits_to_float(bits);
    }
    static __device__ __forceinline__ uint16_t from(float v) {
        if constexpr (BF16) return from_float<bf16_t>(v).bits;
        else {
            union { _Float16 h; uint16_t u; } c;
            c.h = static_cast<_Float16>(v);
            return c.u;
        }
    }
};
#define half_bits_to_float(bits, bf16) HalfBits<bf16>::to_float(bits)
#define float_to_half_bits(v, bf16) HalfBits<bf16>::from(v)
template <bool bf16>
__device__ __forceinline__ void unpack8(const uint4& u, float v[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = half_bits_to_float(w[i] & 0xffffu, bf16);
        v[2 * i + 1] = half_bits_to_float(w[i] >> 16, bf16);
    }
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
template <bool BF16> __device__ __forceinline__ v4f half_mfma(const uint4& a, const uint4& b, v4f c) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// the rotary partner of value d of a head: the other half of the rotary part, itself behind it
__device__ __forceinline__ int rotary_partner(int d, int half) { return d < half ? d + half : (d < 2 * half ? d - half : d); }

// sum over the workgroup of two values at once; everybody gets both
__device__ __forceinline__ void block_sum2(float& a, float& b, float* red) {
    a = group_sum<64>(a);
    b = group_sum<64>(b);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[wave] = a; red[kWaves + wave] = b; }
    __syncthreads();
    const auto eight = [](const float* v) { return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])); };
    a = eight(red);
    b = eight(red + kWaves);
}

// a score with the scale on the query's values
template <bool BF16> __device__ __forceinline__ float scaled_first(const uint16_t* q, const uint16_t* k, float scale) {
    float s = 0.0f;
#pragma unroll 1
    for (int d = 0; d < kHeadDim; d += 8) {
        float qv[8], kv[8];
        unpack8<BF16>(*reinterpret_cast<const uint4*>(q + d), qv);
        unpack8<BF16>(*reinterpret_cast<const uint4*>(k + d), kv);
#pragma unroll
        for (int i = 0; i < 8; ++i) s = __builtin_fmaf(qv[i] * scale, kv[i], s);
    }
    return s;
}

__device__ const float kOne = 1.0f;

struct DecodeArgs {
    const uint16_t* q; const uint16_t* k_new; const uint16_t* v_new;
    const float* q_weight; const float* k_weight;               // RMS normalisation weights over the whole q / k width, or null
    const float* cos_row; const float* sin_row;                 // 128 floats each for this position, or null (no rotary part)
    uint16_t* k_store; uint16_t* v_store;
    size_t batch_stride, head_stride;                           // of the stores, in elements
    float* part;                                                // [batch][heads][runs][kPartFloats]
    uint16_t* out;
    float eps, scale;
    int bf16, heads, kv_heads, rope_half, pos, slices, per, runs, together;     // per: slices of a run; together: runs of a workgroup
};

// GROUP: the query heads per key/value head the loops are unrolled for (at least the launch's heads / kv_heads)
template <bool bf16, int GROUP>
__global__ __launch_bounds__(kThreads, 4) void attn_decode_slice_kernel(const DecodeArgs a) {
    __shared__ float red[2 * kWaves];
    __shared__ __align__(16) uint16_t qn[GROUP][kHeadDim + 8];                // normalized, turned queries of this key/value head's group, zeros behind them
    __shared__ __align__(16) uint16_t new_key[kHeadDim], new_value[kHeadDim]; // the new row as the store holds it
    __shared__ __align__(16) uint16_t raw_q[GROUP * kHeadDim], raw_k[kHeadDim];   // the group's q heads and this head's k as they came
    __shared__ float w_q[GROUP * kHeadDim], w_k[kHeadDim], rot_cos[kHeadDim], rot_sin[kHeadDim];
    __shared__ __align__(16) float weight[2][GROUP][kSliceKeys + 4];          // scores of the two halves of the head's columns; the first then the softmax weights
    __shared__ float stats[GROUP][2];
    __shared__ __align__(16) float sums[8][GROUP][kHeadDim];              // weighted value sums per wave's eight keys

    const int kvh = blockIdx.y, b = blockIdx.z;
    const int tid = threadIdx.x;
    const int group = a.heads / a.kv_heads;
    const int length = a.pos + 1;
    const int first_run = blockIdx.x * a.together, first = first_run * a.per, last = min(first + a.together * a.per, a.slices) - 1;
    const bool has_new = last == a.slices - 1;                                // the last slice holds the new position: its workgroup writes the stores
    const uint16_t* kbase = a.k_store + static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(kvh) * a.head_stride;
    const uint16_t* vbase = a.v_store + static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(kvh) * a.head_stride;

    // Stored keys and values of the slice first: they are the long round trip.  Keys come as matrix operands: wave w has keys 16 (w % 4) .. + 15,
    // columns 64 (w / 4) .. + 63, lane (key lane % 16, part lane / 16) the 16-byte pieces 2 part and 2 part + 1 of them; values: thread
    // (keys 4 (tid / 32) .. + 3, columns 4 (tid % 32) .. + 3).  The new position is not in memory yet.
    // Every load has a valid address whatever the thread's share (row numbers clamped to the new position, whose row exists and is
    // replaced below): no load stands under a condition, so all of them are in flight together.
    const int lane = tid & 63, wave = tid >> 6;
    const int key = 16 * (wave & 3) + (lane & 15), column = 64 * (wave >> 2) + 16 * (lane >> 4);
    const int kg = tid >> 5, dpart = tid & 31;
    uint4 kreg[2];
    uint2 vreg[4];
    auto load_keys = [&](int j0) {
        const uint4* src = reinterpret_cast<const uint4*>(kbase + static_cast<size_t>(min(j0 + key, a.pos)) * kHeadDim + column);
#pragma unroll
        for (int i = 0; i < 2; ++i) kreg[i] = src[i];
    };
    auto load_values = [&](int j0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            vreg[i] = *reinterpret_cast<const uint2*>(vbase + static_cast<size_t>(min(j0 + 4 * kg + i, a.pos)) * kHeadDim + 4 * dpart);
    };
    load_keys(first * kSliceKeys);
    load_values(first * kSliceKeys);

    // the q row, this head's k row, the group's normalisation weights and the rotary rows: requested in one batch behind the
    // stores' rows, staged in LDS as they are, so that the whole prologue costs one round trip to memory
    const uint16_t* qrow = a.q + static_cast<size_t>(b) * a.heads * kHeadDim;
    const uint16_t* krow = a.k_new + static_cast<size_t>(b) * a.kv_heads * kHeadDim;
    const int q_width = a.heads * kHeadDim, k_width = a.kv_heads * kHeadDim;
    uint4 qpiece[kQPieces], kpiece[kKPieces];
#pragma unroll
    for (int r = 0; r < kQPieces; ++r) qpiece[r] = *reinterpret_cast<const uint4*>(qrow + min(8 * (tid + kThreads * r), q_width - 8));
#pragma unroll
    for (int r = 0; r < kKPieces; ++r) kpiece[r] = *reinterpret_cast<const uint4*>(krow + min(8 * (tid + kThreads * r), k_width - 8));
    const float* qw_src = a.q_weight ? a.q_weight + kvh * group * kHeadDim : &kOne;    // null weights: read a one, stride zero
    const int qw_last = a.q_weight ? group * kHeadDim - 1 : 0;
    constexpr int kWeights = (GROUP * kHeadDim + kThreads - 1) / kThreads;
    float qw_reg[kWeights];
#pragma unroll
    for (int r = 0; r < kWeights; ++r) qw_reg[r] = qw_src[min(tid + kThreads * r, qw_last)];
    const float kw_reg = a.k_weight ? a.k_weight[kvh * kHeadDim + (tid & (kHeadDim - 1))] : 1.0f;
    const float rot_reg = a.cos_row ? (tid & kHeadDim ? a.sin_row : a.cos_row)[tid & (kHeadDim - 1)] : (tid < kHeadDim ? 1.0f : 0.0f);
    const uint16_t v_bits = a.v_new[static_cast<size_t>(b) * k_width + kvh * kHeadDim + (tid & (kHeadDim - 1))];

    // sums of squares of the whole q and k rows; the group's part of q and this head's k go to LDS on the way
    float ssq = 0.0f, ssk = 0.0f;
#pragma unroll
    for (int r = 0; r < kQPieces; ++r) {
        float v[8];
        unpack8<bf16>(qpiece[r], v);
        if (8 * (tid + kThreads * r) < q_width)
#pragma unroll
            for (int e = 0; e < 8; ++e) ssq += v[e] * v[e];
        const int at = 8 * (tid + kThreads * r) - kvh * group * kHeadDim;          // position inside the group's part
        if (at >= 0 && at < group * kHeadDim) *reinterpret_cast<uint4*>(&raw_q[at]) = qpiece[r];
    }
#pragma unroll
    for (int r = 0; r < kKPieces; ++r) {
        float v[8];
        unpack8<bf16>(kpiece[r], v);
        if (8 * (tid + kThreads * r) < k_width)
#pragma unroll
            for (int e = 0; e < 8; ++e) ssk += v[e] * v[e];
        const int at = 8 * (tid + kThreads * r) - kvh * kHeadDim;
        if (at >= 0 && at < kHeadDim) *reinterpret_cast<uint4*>(&raw_k[at]) = kpiece[r];
    }
#pragma unroll
    for (int r = 0; r < kWeights; ++r)
        if (tid + kThreads * r < group * kHeadDim) w_q[tid + kThreads * r] = qw_reg[r];
    if (tid < kHeadDim) { w_k[tid] = kw_reg; rot_cos[tid] = rot_reg; }
    else if (tid < 2 * kHeadDim) rot_sin[tid - kHeadDim] = rot_reg;
    block_sum2(ssq, ssk, red);                                                // (its barrier also covers the staging above)
    const float rstd_q = a.q_weight ? rsqrtf(ssq / static_cast<float>(q_width) + a.eps) : 1.0f;
    const float rstd_k = a.k_weight ? rsqrtf(ssk / static_cast<float>(k_width) + a.eps) : 1.0f;

    // one normalized value: x * rstd * weight, rounded to the activations' type like a separate normalisation's output; then the
    // turn out = x cos + partner sin, rounded again like a separate rotary operator's output
    auto normed = [&](const uint16_t* raw, const float* w, bool on, float rstd, int i) {
        const float x = half_bits_to_float(raw[i], bf16);
        return on ? half_bits_to_float(float_to_half_bits(x * rstd * w[i], bf16), bf16) : x;
    };
    auto turned = [&](const uint16_t* raw, const float* w, bool on, float rstd, int head_at, int d) {
        const float x = normed(raw, w, on, rstd, head_at + d);
        if (!a.cos_row) return x;
        const float xp = normed(raw, w, on, rstd, head_at + rotary_partner(d, a.rope_half));
        return half_bits_to_float(float_to_half_bits(__builtin_fmaf(xp, rot_sin[d], x * rot_cos[d]), bf16), bf16);
    };
    for (int e = tid; e < GROUP * kHeadDim; e += kThreads) {
        const int g = e / kHeadDim, d = e % kHeadDim;
        qn[g][d] = g < group ? float_to_half_bits(turned(raw_q, w_q, a.q_weight != nullptr, rstd_q, g * kHeadDim, d), bf16) : uint16_t{0};
    }
    if (has_new && tid < kHeadDim) {
        const uint16_t kb = float_to_half_bits(turned(raw_k, w_k, a.k_weight != nullptr, rstd_k, 0, tid), bf16);
        new_key[tid] = kb;
        new_value[tid] = v_bits;
        const size_t at = static_cast<size_t>(b) * a.batch_stride + static_cast<size_t>(kvh) * a.head_stride + static_cast<size_t>(a.pos) * kHeadDim + tid;
        a.k_store[at] = kb;
        a.v_store[at] = v_bits;
    }
    __syncthreads();

    constexpr int kOutputs = (GROUP * kHeadDim + kThreads - 1) / kThreads;
    float total[kOutputs], top[kOutputs], den[kOutputs];
    uint4 qreg[2];                                                            // head lane % 16, the columns of kreg
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        qreg[i] = *reinterpret_cast<const uint4*>(&qn[min(lane & 15, GROUP - 1)][column + 8 * i]);
        if ((lane & 15) >= GROUP) qreg[i] = make_uint4(0, 0, 0, 0);
    }
    int run = first_run, run_last = min(first + a.per, a.slices) - 1;
    bool fresh = true;                                                        // the slice is a run's first
    for (int slice = first; slice <= last; ++slice) {
        const int j0 = slice * kSliceKeys, nkeys = min(kSliceKeys, length - j0), next = min(slice + 1, last) * kSliceKeys;
        // scores on the matrix cores, products of the 16-bit values exact: rows the wave's keys, columns the group's heads
        if (j0 + key == a.pos) {
#pragma unroll
            for (int i = 0; i < 2; ++i) kreg[i] = *reinterpret_cast<const uint4*>(new_key + column + 8 * i);
        }
        {
            v4f s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 2; ++i) s = half_mfma<bf16>(kreg[i], qreg[i], s);
            if ((lane & 15) < group) *reinterpret_cast<v4f*>(&weight[wave >> 2][lane & 15][16 * (wave & 3) + 4 * (lane >> 4)]) = s;
        }
        load_keys(next);
        __syncthreads();

        // softmax statistics of the slice: a wave per head
        for (int g = wave; g < group; g += kWaves) {
            float s = weight[0][g][lane] + weight[1][g][lane];
            // (products of bf16 values can pass the largest float where the scaled score does not: there the scale goes on the query, in float32)
            if (bf16 && __any(lane < nkeys && !(fabsf(s) <= FLT_MAX))) s = scaled_first<bf16>(qn[g], j0 + lane >= a.pos ? new_key : kbase + static_cast<size_t>(j0 + lane) * kHeadDim, a.scale);
            else s *= a.scale;
            s = lane < nkeys ? s : -INFINITY;
            const float m = group_max<64>(s);
            const float p = lane < nkeys ? expf(s - m) : 0.0f;
            weight[0][g][lane] = p;
            const float l = group_sum<64>(p);
            if (lane == 0) { stats[g][0] = m; stats[g][1] = l; }
        }
        __syncthreads();

        // weighted sums of the values: four keys and four columns per thread, then the two halves of a wave
        {
            float acc[GROUP][4] = {}, p[GROUP][4];
#pragma unroll
            for (int g = 0; g < GROUP; ++g) {
                const float4 p4 = *reinterpret_cast<const float4*>(&weight[0][g < group ? g : 0][4 * kg]);
                p[g][0] = p4.x; p[g][1] = p4.y; p[g][2] = p4.z; p[g][3] = p4.w;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = 4 * kg + i;
                if (j < nkeys) {                 // uniform over the 32 threads of a key group
                    const uint2 fresh = *reinterpret_cast<const uint2*>(new_value + 4 * dpart);
                    const uint2 bits = j0 + j == a.pos ? fresh : vreg[i];
                    const float v0 = half_bits_to_float(bits.x & 0xffffu, bf16), v1 = half_bits_to_float(bits.x >> 16, bf16);
                    const float v2 = half_bits_to_float(bits.y & 0xffffu, bf16), v3 = half_bits_to_float(bits.y >> 16, bf16);
#pragma unroll
                    for (int g = 0; g < GROUP; ++g) {
                        acc[g][0] = __builtin_fmaf(p[g][i], v0, acc[g][0]);
                        acc[g][1] = __builtin_fmaf(p[g][i], v1, acc[g][1]);
                        acc[g][2] = __builtin_fmaf(p[g][i], v2, acc[g][2]);
                        acc[g][3] = __builtin_fmaf(p[g][i], v3, acc[g][3]);
                    }
                }
            }
#pragma unroll
            for (int g = 0; g < GROUP; ++g)
                if (g < group) {
                    float sum[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        float lower, upper;
                        swapped_pair<32>(acc[g][c], lower, upper);
                        sum[c] = lower + upper;
                    }
                    if ((kg & 1) == (g & 1)) *reinterpret_cast<float4*>(&sums[kg >> 1][g][4 * dpart]) = make_float4(sum[0], sum[1], sum[2], sum[3]);
                }
        }
        load_values(next);
        __syncthreads();
        // the slices of a run one after the other, in order: the usual running maximum
#pragma unroll
        for (int r = 0; r < kOutputs; ++r) {
            const int e = tid + kThreads * r, g = e / kHeadDim, d = e % kHeadDim;
            if (e >= group * kHeadDim) break;
            float o = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) o += sums[w][g][d];
            const float m = stats[g][0], l = stats[g][1];
            if (fresh) {
                total[r] = o;
                top[r] = m;
                den[r] = l;
            } else {
                const float now = fmaxf(top[r], m), before = expf(top[r] - now), here = expf(m - now);
                total[r] = total[r] * before + o * here;
                den[r] = den[r] * before + l * here;
                top[r] = now;
            }
        }
        fresh = slice == run_last;
        if (!fresh) continue;
        int thread = tid;
        asm volatile("" : "+v"(thread));             // (addresses worked out here: kept over the loop they push registers of eight heads to scratch memory)
#pragma unroll
        for (int r = 0; r < kOutputs; ++r) {
            const int e = thread + kThreads * r, g = e / kHeadDim, d = e % kHeadDim, head = kvh * group + g;
            if (e >= group * kHeadDim) break;
            if (a.runs == 1) {
                a.out[(static_cast<size_t>(b) * a.heads + head) * kHeadDim + d] = float_to_half_bits(total[r] / den[r], bf16);
            } else {
                float* dst = a.part + ((static_cast<size_t>(b) * a.heads + head) * a.runs + run) * kPartFloats;
                dst[d] = total[r];
                if (d == 0) { dst[kHeadDim] = top[r]; dst[kHeadDim + 1] = den[r]; }
            }
        }
        ++run;
        run_last = min(run_last + a.per, a.slices - 1);
    }
}

// out[b, head, :] = sum over slices of sums * exp(m - M) / sum over slices of l * exp(m - M), slices in order.
// The slices' statistics are fetched side by side (one round trip), the sums in batches of eight.
constexpr int kMaxSlices = 2048;                // stores of up to 131072 positions
__global__ __launch_bounds__(kHeadDim) void attn_decode_merge_kernel(const float* __restrict__ part, uint16_t* __restrict__ out, int slices, int bf16) {
    __shared__ float factor[kMaxSlices];
    __shared__ float wave_top[2], wave_den[2];
    const size_t row = blockIdx.x;                                            // b * heads + head
    const float* src = part + row * slices * kPartFloats;
    const int d = threadIdx.x;
    float top = -INFINITY;
    for (int s = d; s < slices; s += kHeadDim) { const float m = src[s * kPartFloats + kHeadDim]; factor[s] = m; top = fmaxf(top, m); }
    top = group_max<64>(top);
    if ((d & 63) == 0) wave_top[d >> 6] = top;
    __syncthreads();
    top = fmaxf(wave_top[0], wave_top[1]);
    float den = 0.0f;
    for (int s = d; s < slices; s += kHeadDim) {
        const float f = expf(factor[s] - top);
        factor[s] = f;
        den = __builtin_fmaf(src[s * kPartFloats + kHeadDim + 1], f, den);
    }
    den = group_sum<64>(den);
    if ((d & 63) == 0) wave_den[d >> 6] = den;
    __syncthreads();
    den = wave_den[0] + wave_den[1];
    float num = 0.0f;
    int s = 0;
    for (; s + 8 <= slices; s += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = src[(s + i) * kPartFloats + d];
#pragma unroll
        for (int i = 0; i < 8; ++i) num = __builtin_fmaf(v[i], factor[s + i], num);
    }
    for (; s < slices; ++s) num = __builtin_fmaf(src[s * kPartFloats + d], factor[s], num);
    out[row * kHeadDim + d] = bf16 ? HalfBits<true>::from(num / den) : HalfBits<false>::from(num / den);
}

}  // namespace

// Pieces of work of one workgroup: one workgroup per compute unit, or two, which hide each other's waits, from `two_from` pieces on.  Slices of a run: so that one
// sequence fills the machine, whatever the batch, so a sequence's sums (and bits) are the same in any; runs of a workgroup: by the whole batch
// (runs as long as a workgroup's share of the batch write and merge less: 48 and 8 heads, replayed, 16 rows of 1024 23.1 / 22.9 us, 32 of 2048 59.5 / 64.9, 256 of
// 200 62 / 76; a workgroup per run: 31 / 109 / 107; before workgroups walked over slices: 39 / 132 / 134).
// Slices: two workgroups per unit once each has two slices or more (48 query and 8 key/value heads, us with one / with two: 3000 positions 12.0 / 14.6, 4096
// 12.6 / 13.6, 16384 26.0 / 24.2, 100001 108 / 90; 32 and 8 heads, 6000 positions 12.9 / 15.7, 16384 22.2 / 20.8, four rows of 1024 positions 10.8 / 11.3,
// sixteen 22.5 / 20.7).  Runs of several slices: two as soon as there are more runs than units (8 and 8 heads, two rows of 3001 positions 11.6 / 10.8; 16 and 8 12.3 / 11.2).
static int pieces_per_workgroup(long long pieces, int rows, long long two_from) {
    const long long total = pieces * rows, units = compute_units(), places = total >= two_from ? 2 * units : units;
    return static_cast<int>(std::min(pieces, (total + places - 1) / places));
}

size_t attention_decode_workspace_bytes(int batch, int heads, int pos) {
    const int slices = pos / kSliceKeys + 1;
    return slices == 1 ? 0 : align256(static_cast<size_t>(batch) * heads * slices * kPartFloats * sizeof(float));
}

bool attention_decode_supports(int heads, int kv_heads, int head_dim, int rope_dim) {
    return head_dim == kHeadDim && kv_heads >= 1 && heads % kv_heads == 0 && heads / kv_heads <= kMaxGroup && heads <= kMaxHeads &&
           kv_heads * kHeadDim <= kKPieces * 8 * kThreads && rope_dim >= 0 && rope_dim <= kHeadDim && rope_dim % 2 == 0;
}

int attention_decode(const void* q, const void* k_new, const void* v_new, int dtype, const float* q_weight, const float* k_weight, float eps,
                     const float* cos_row, const float* sin_row, int rope_dim, void* k_store, void* v_store, size_t batch_stride,
                     size_t head_stride, int batch, int heads, int kv_heads, int pos, void* out, void* workspace, hipStream_t stream) {
    DecodeArgs a;
    a.q = static_cast<const uint16_t*>(q); a.k_new = static_cast<const uint16_t*>(k_new); a.v_new = static_cast<const uint16_t*>(v_new);
    a.q_weight = q_weight; a.k_weight = k_weight;
    a.cos_row = rope_dim > 0 ? cos_row : nullptr; a.sin_row = rope_dim > 0 ? sin_row : nullptr;
    a.k_store = static_cast<uint16_t*>(k_store); a.v_store = static_cast<uint16_t*>(v_store);
    a.batch_stride = batch_stride; a.head_stride = head_stride;
    a.part = static_cast<float*>(workspace);
    a.out = static_cast<uint16_t*>(out);
    a.eps = eps; a.scale = 1.0f / sqrtf(static_cast<float>(kHeadDim));
    a.bf16 = dtype == PLLM_BF16; a.heads = heads; a.kv_heads = kv_heads; a.rope_half = rope_dim / 2; a.pos = pos;
    a.slices = pos / kSliceKeys + 1;
    if (a.slices > kMaxSlices) return PLLM_ERR_UNSUPPORTED;
    const int group = heads / kv_heads;
    const long long units = compute_units();
    // One or two query heads per key/value head: a slice takes less than a workgroup's start, so runs of one slice where runs of two would leave units idle, as
    // far as the merge sums them in one batch (us, of two / of one: 16 and 16 heads, 1501 positions 9.4 / 9.0, two rows of them 11.1 / 10.3; 2048 positions, which fill the
    // machine by twos, 8.6 / 9.2; 8 and 8 heads, 3001 positions 8.7 / 10.7; the form of a slice per workgroup of four waves 8.7, 9.8, 8.8 and 10.6)
    const bool singles = group <= 2 && a.slices <= 32 && static_cast<long long>(a.slices) * kv_heads < 2 * units;
    a.per = singles ? 1 : pieces_per_workgroup(a.slices, kv_heads, 4 * units);
    a.runs = (a.slices + a.per - 1) / a.per;
    a.together = pieces_per_workgroup(a.runs, kv_heads * batch, a.per > 1 ? units + 1 : 4 * units);
    const dim3 grid((a.runs + a.together - 1) / a.together, kv_heads, batch);
#define PLLM_CASE(G) \
    if (group <= G) { \
        if (a.bf16) hipLaunchKernelGGL((attn_decode_slice_kernel<true, G>), grid, dim3(kThreads), 0, stream, a); \
        else hipLaunchKernelGGL((attn_decode_slice_kernel<false, G>), grid, dim3(kThreads), 0, stream, a); \
    } else
    PLLM_CASE(1) PLLM_CASE(2) PLLM_CASE(4) PLLM_CASE(6) PLLM_CASE(8) return PLLM_ERR_UNSUPPORTED;
#undef PLLM_CASE
    if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    if (a.runs > 1) {
        hipLaunchKernelGGL(attn_decode_merge_kernel, dim3(batch * heads), dim3(kHeadDim), 0, stream, a.part, a.out, a.runs, a.bf16);
        if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    }
    return PLLM_OK;
}

}  // namespace pllm
