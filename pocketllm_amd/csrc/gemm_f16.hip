// Prefill matmul y[T, N] = x[T, K] . dequant(W)[N, K]^T over raw super-blocks, on f16 MFMA: activation staging, plan of the tiles, their
// launches.  The kernel itself is gemm_tile.h, the block formats tile_formats.h.
//
// The activations go in as fp16.  fp16 rows that need no padding are read as the caller holds them; for the others a pre-pass scales
// every token row by a power of two so that its largest value sits just below 2^14, which keeps bf16 inputs exact and cannot
// overflow.
//
// The grid is one-dimensional.  Tiles that fill whole rounds of the machine (one workgroup per compute unit) run over all of K and store
// their result directly; the tiles left over, which would occupy a fraction of the machine for a full round, are cut along K in slices:
// every slice writes a float32 partial tile and a second kernel adds them in slice order, which keeps the result independent of
// scheduling.  Small token counts consist of left-over tiles only.
//
// Why fp16 tiles and not int8 MFMA here: with int8 activations every 32-wide group needs a float fix-up per output (two scales that
// change along K), which costs more vector instructions than the MFMA saves, and a single int8 activation term sits at ~5e-3 from the
// float statement of the operator.  Decoded-to-fp16 tiles need no fix-up, keep bf16 activations exact and land at ~2e-4.
#include "gemm_tile.h"

#include <algorithm>

namespace pllm {
namespace {

constexpr int kBN = kTileN;

// ---- activation pre-pass --------------------------------------------------------------------------
// xh[t, 0..kp) = fp16(x[t, :] * 2^-e_t) (zero beyond k), scale[t] = 2^e_t, amax_t * 2^-e_t in [2^13, 2^14)
__global__ __launch_bounds__(256) void act_f16_kernel(const void* __restrict__ x, int x_dtype, _Float16* __restrict__ xh,
                                                      float* __restrict__ scale, int k, int kp, const int64_t* __restrict__ row_map) {
    __shared__ float red[4];
    const size_t xoff = static_cast<size_t>(row_map ? row_map[blockIdx.x] : blockIdx.x) * k;      // row_map gathers source rows
    float am = 0.0f;
    for (int i = threadIdx.x; i < k; i += 256) am = fmaxf(am, fabsf(load_any(x, x_dtype, xoff + i)));
    am = group_max<64>(am);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = am;
    __syncthreads();
    am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int e = half_row_exponent<14>(am);
    const float down = ldexpf(1.0f, -e);
    _Float16* out = xh + static_cast<size_t>(blockIdx.x) * kp;
    for (int i = threadIdx.x; i < kp; i += 256)
        out[i] = static_cast<_Float16>(i < k ? load_any(x, x_dtype, xoff + i) * down : 0.0f);
    if (threadIdx.x == 0) scale[blockIdx.x] = ldexpf(1.0f, e);
}

// The same for rows of at most 8192 values with 16-bit inputs (the usual case): one wave per row
// keeps the row in registers between the maximum and the conversion, so x is read once.
// bits(v) = the value as float32: bf16 is the high half of a float32, fp16 converts in hardware.
// WPR = waves per row: 1 (four rows per workgroup) or 4 (one row per workgroup, for calls of few rows: four times the
// workgroups, a quarter of the row per wave; the waves meet in LDS for the maximum).
template <bool BF16, int WPR>
__global__ __launch_bounds__(256) void act_f16_rows_kernel(const uint16_t* __restrict__ x, _Float16* __restrict__ xh,
                                                           float* __restrict__ scale, int rows, int k, int kp, const int64_t* __restrict__ row_map) {
    __shared__ float wave_max[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = WPR == 1 ? blockIdx.x * 4 + wave : blockIdx.x, part = WPR == 1 ? 0 : wave;
    if (row >= rows) return;                       // (a whole workgroup when WPR = 4)
    const uint16_t* src = x + static_cast<size_t>(row_map ? row_map[row] : row) * k;
    constexpr int kMaxPieces = 16 / WPR;           // 16 pieces x 64 lanes x 8 values per row
    uint4 piece[kMaxPieces];
    float am = 0.0f;
    auto value = [](uint32_t word, int hi) -> float {
        const uint32_t h = hi ? (word >> 16) : (word & 0xffffu);
        if (BF16) return __uint_as_float(h << 16);
        return f16_bits_to_float(h);
    };
#pragma unroll
    for (int i = 0; i < kMaxPieces; ++i) {
        const int e0 = ((i * WPR + part) * 64 + lane) * 8;
        piece[i] = make_uint4(0, 0, 0, 0);
        if (e0 < k) piece[i] = *reinterpret_cast<const uint4*>(src + e0);          // k is a multiple of 8 here
        const uint32_t wds[4] = {piece[i].x, piece[i].y, piece[i].z, piece[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) am = fmaxf(am, fmaxf(fabsf(value(wds[j], 0)), fabsf(value(wds[j], 1))));
    }
    am = group_max<64>(am);
    if constexpr (WPR > 1) {
        if (lane == 0) wave_max[wave] = am;
        __syncthreads();
        am = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
    }
    const int e = half_row_exponent<14>(am);
    const float down = ldexpf(1.0f, -e);
    _Float16* out = xh + static_cast<size_t>(row) * kp;
#pragma unroll
    for (int i = 0; i < kMaxPieces; ++i) {
        const int e0 = ((i * WPR + part) * 64 + lane) * 8;
        if (e0 >= kp) continue;
        const uint32_t wds[4] = {piece[i].x, piece[i].y, piece[i].z, piece[i].w};
        half8 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o[2 * j] = static_cast<_Float16>(value(wds[j], 0) * down);
            o[2 * j + 1] = static_cast<_Float16>(value(wds[j], 1) * down);
        }
        *reinterpret_cast<half8*>(out + e0) = o;
    }
    if (lane == 0 && part == 0) scale[row] = ldexpf(1.0f, e);
}

// The same for longer rows and for float32 ones: a workgroup of eight waves keeps a row of up to 32768 values in registers, so x is read
// once, 16 bytes per load.  (The kernel above that, which walks the row twice one value at a time, remains for odd lengths and alignments:
// us, that one / this one, 1999 rows of 17408 fp16 values 88.1 / 28.4, 7 rows 37.1 / 4.9.)
constexpr int kLongThreads = 512, kLongPieces = 8, kLongRow = kLongThreads * 8 * kLongPieces;
template <int DT>
__global__ __launch_bounds__(kLongThreads) void act_f16_long_kernel(const void* __restrict__ x, _Float16* __restrict__ xh, float* __restrict__ scale,
                                                                    int k, int kp, const int64_t* __restrict__ row_map) {
    __shared__ float wave_max[kLongThreads / 64];
    constexpr int kVecs = DT == PLLM_F32 ? 2 : 1;
    const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned char* src = static_cast<const unsigned char*>(x) + static_cast<size_t>(row_map ? row_map[row] : row) * k * (8 * kVecs / 4);
    uint4 piece[kLongPieces][kVecs];
    auto value = [&](int i, int j) -> float {       // value j of piece i
        if constexpr (DT == PLLM_F32) {
            const uint4 v = piece[i][j >> 2];
            return __uint_as_float((j & 3) == 0 ? v.x : (j & 3) == 1 ? v.y : (j & 3) == 2 ? v.z : v.w);
        } else {
            const uint4 v = piece[i][0];
            const uint32_t w = j < 2 ? v.x : j < 4 ? v.y : j < 6 ? v.z : v.w, h = (j & 1) ? w >> 16 : w & 0xffffu;
            return DT == PLLM_BF16 ? __uint_as_float(h << 16) : f16_bits_to_float(h);
        }
    };
#pragma unroll
    for (int i = 0; i < kLongPieces; ++i) {
        const int e0 = (i * kLongThreads + threadIdx.x) * 8;
#pragma unroll
        for (int j = 0; j < kVecs; ++j) {
            piece[i][j] = make_uint4(0, 0, 0, 0);
            if (e0 < k) piece[i][j] = *reinterpret_cast<const uint4*>(src + static_cast<size_t>(e0) * (2 * kVecs) + 16 * j);      // k is a multiple of 8 here
        }
    }
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < kLongPieces; ++i)
        if (i * kLongThreads * 8 < k) {
#pragma unroll
            for (int j = 0; j < 8; ++j) am = fmaxf(am, fabsf(value(i, j)));
        }
    am = group_max<64>(am);
    if (lane == 0) wave_max[wave] = am;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kLongThreads / 64; ++i) am = fmaxf(am, wave_max[i]);
    const int e = half_row_exponent<14>(am);
    const float down = ldexpf(1.0f, -e);
    _Float16* out = xh + static_cast<size_t>(row) * kp;
#pragma unroll
    for (int i = 0; i < kLongPieces; ++i) {
        const int e0 = (i * kLongThreads + threadIdx.x) * 8;
        if (e0 >= kp) continue;
        half8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = static_cast<_Float16>(value(i, j) * down);
        *reinterpret_cast<half8*>(out + e0) = o;
    }
    if (threadIdx.x == 0) scale[row] = ldexpf(1.0f, e);
}

// Hidden activations of the routed experts: h = silu(min(g, L)) * clamp(u, +-L) * w_r (L <= 0: no clamp) from the float32 gate / up
// products, written as fp16 rows scaled like the ones above.
struct Hidden {
    float limit, route_weight;
    __device__ __forceinline__ float operator()(float g, float u) const {
        if (limit > 0.0f) {
            u = fminf(fmaxf(u, -limit), limit);
            g = fminf(g, limit);
        }
        return g / (1.0f + expf(-g)) * u * route_weight;
    }
};
// One workgroup per route, HELD pieces of four columns per thread (rows of up to 1024 HELD columns, a multiple of four): every product is read
// once, by loads that are all on their way together, and the exponential taken once.  Bound: the two float32 rows' bytes.  (One wave per route
// that walked its row twice: 27 us at 2048 routes of 1536 columns, 44 at 8192.)
template <int HELD>
__global__ __launch_bounds__(256) void swiglu_f16_held_kernel(const float* __restrict__ g, const float* __restrict__ u, const float* __restrict__ route_weights,
                                                              float limit, _Float16* __restrict__ hh, float* __restrict__ scale, int inter, int kp) {
    __shared__ float wave_max[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float4* gr = reinterpret_cast<const float4*>(g + static_cast<size_t>(row) * inter);
    const float4* ur = reinterpret_cast<const float4*>(u + static_cast<size_t>(row) * inter);
    const Hidden hidden{limit, route_weights[row]};
    float4 a[HELD], b[HELD];
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
        const int at = tid + 256 * j, from = 4 * at < inter ? at : 0;
        a[j] = gr[from];
        b[j] = ur[from];
    }
    float am = 0.0f;
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
        const bool in = 4 * (tid + 256 * j) < inter;
        a[j] = make_float4(hidden(a[j].x, b[j].x), hidden(a[j].y, b[j].y), hidden(a[j].z, b[j].z), hidden(a[j].w, b[j].w));
        if (!in) a[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        am = fmaxf(fmaxf(fmaxf(am, fabsf(a[j].x)), fmaxf(fabsf(a[j].y), fabsf(a[j].z))), fabsf(a[j].w));
    }
    am = group_max<64>(am);
    if ((tid & 63) == 0) wave_max[tid >> 6] = am;
    __syncthreads();
    const int e = half_row_exponent<14>(fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3])));
    const float down = ldexpf(1.0f, -e);
    _Float16* out = hh + static_cast<size_t>(row) * kp;
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
        const int col = 4 * (tid + 256 * j);
        if (col >= kp) continue;
        union { _Float16 h[4]; uint2 w; } o;
        o.h[0] = static_cast<_Float16>(a[j].x * down);
        o.h[1] = static_cast<_Float16>(a[j].y * down);
        o.h[2] = static_cast<_Float16>(a[j].z * down);
        o.h[3] = static_cast<_Float16>(a[j].w * down);
        *reinterpret_cast<uint2*>(out + col) = o.w;
    }
    if (tid == 0) scale[row] = ldexpf(1.0f, e);
}

// the same for rows of any length, one wave per route
__global__ __launch_bounds__(256) void swiglu_f16_rows_kernel(const float* __restrict__ g, const float* __restrict__ u,
                                                              const float* __restrict__ route_weights, float limit, _Float16* __restrict__ hh,
                                                              float* __restrict__ scale, int rows, int inter, int kp) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float* gr = g + static_cast<size_t>(row) * inter;
    const float* ur = u + static_cast<size_t>(row) * inter;
    const Hidden hidden{limit, route_weights[row]};
    float am = 0.0f;
    for (int i = lane; i < inter; i += 64) am = fmaxf(am, fabsf(hidden(gr[i], ur[i])));
    am = group_max<64>(am);
    const int e = half_row_exponent<14>(am);
    const float down = ldexpf(1.0f, -e);
    _Float16* out = hh + static_cast<size_t>(row) * kp;
    for (int i = lane; i < kp; i += 64) out[i] = static_cast<_Float16>(i < inter ? hidden(gr[i], ur[i]) * down : 0.0f);
    if (lane == 0) scale[row] = ldexpf(1.0f, e);
}

// 32 tokens x 64 columns (the share of one wave and token block, blockIdx.x) of split tile full_tiles + blockIdx.y:
// y[t, n] = xscale[t] * the sum, in slice order, of its slices' partial tiles, which lie as the lanes held them: [wave][token
// block][column / 32 of the wave][8-column group][half-wave: column / 4 of the group][token][column % 4].
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const TileCall c, int nt) {
    const int tile = c.full_tiles + blockIdx.y, bm = 32 * nt;
    int col_tile = tile / c.tiles_m, n = c.n;
    const uint8_t* unused = nullptr;
    void* y = c.y;
    c.more.pick(col_tile, unused, y, n);
    const int token = threadIdx.x >> 3, c8 = threadIdx.x & 7;               // eight columns per thread, a line per eight threads
    const int row = (tile % c.tiles_m) * bm + 32 * (blockIdx.x % nt) + token, col = col_tile * kBN + 64 * (blockIdx.x / nt) + 8 * c8;
    if (row >= c.t_rows || col >= n) return;
    const size_t tile_elems = static_cast<size_t>(bm) * kBN;
    const float* src = c.partial + static_cast<size_t>(blockIdx.y) * c.slices * tile_elems + (static_cast<size_t>(blockIdx.x) * 8 + c8) * 256 + token * 4;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int k = 0; k < c.slices; ++k) {
        const float4 lo = *reinterpret_cast<const float4*>(src + k * tile_elems), hi = *reinterpret_cast<const float4*>(src + k * tile_elems + 128);
        v[0] += lo.x; v[1] += lo.y; v[2] += lo.z; v[3] += lo.w;
        v[4] += hi.x; v[5] += hi.y; v[6] += hi.z; v[7] += hi.w;
    }
    const float sc = c.xscale ? c.xscale[row] : 1.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= sc;
    const size_t o = static_cast<size_t>(row) * n + col;
    if ((n & 7) == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 && !(c.y_dtype & kAccumulateInto)) {
        if (c.y_dtype == PLLM_F32) {
            float4* const dst = reinterpret_cast<float4*>(static_cast<float*>(y) + o);
            dst[0] = make_float4(v[0], v[1], v[2], v[3]);
            dst[1] = make_float4(v[4], v[5], v[6], v[7]);
        } else {
            uint32_t h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                h[i] = c.y_dtype == PLLM_BF16 ? from_float<bf16_t>(v[2 * i]).bits | (static_cast<uint32_t>(from_float<bf16_t>(v[2 * i + 1]).bits) << 16)
                                              : pack_halves(v[2 * i], v[2 * i + 1]);
            *reinterpret_cast<uint4*>(static_cast<uint16_t*>(y) + o) = make_uint4(h[0], h[1], h[2], h[3]);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (col + i < n) store_any(y, c.y_dtype, o + i, v[i]);
}

struct GemmPlan { int mi; int tiles_n; int tiles; int full_tiles; int slices; };

size_t partial_bytes(const GemmPlan& p) {
    return p.slices > 1 ? align256(static_cast<size_t>(p.tiles - p.full_tiles) * p.slices * 64 * p.mi * kBN * sizeof(float)) : 0;
}

GemmPlan tiles_of(int t_rows, int n, int mi) {
    GemmPlan p;
    const int cus = compute_units(), bm = 64 * mi;
    p.mi = mi;
    p.tiles_n = (n + kBN - 1) / kBN;
    p.tiles = ((t_rows + bm - 1) / bm) * p.tiles_n;
    p.full_tiles = (p.tiles / cus) * cus;
    p.slices = 1;
    return p;
}

// us that a tile takes per super-block of K: where every compute unit has one (`full`: the clock gives way, so half as many tiles at a time take
// half as long each) and where few have (`alone`: what a wave needs for its own chain).  Fitted to 363 sizes of 64 - 1999 rows, each at both
// heights and up to eleven numbers of slices; the choice by them is 1.0 % behind the best of those on average (heights by token count and
// slices by 8.8 us for every format: 4.0 % behind).  Long rows cost the lower tiles more per block (Q4_K 5120x17408 at 512 rows in three
// slices of 128-row tiles: 108.6 us, as much as 256-row tiles in six, where 17408x5120 gains a fifth), and any tile that runs by itself
// (Q5_K 5120x17408 at 1999 rows, 160 tiles whole 402 us, in three slices 382).
struct TileCost { double full, alone; };
TileCost tile_cost(int type_id, int mi) {
    switch (type_id) {
        case PLLM_TYPE_Q2_K: return mi == 2 ? TileCost{3.3, 2.9} : TileCost{7.0, 4.8};
        case PLLM_TYPE_Q4_K: return mi == 2 ? TileCost{3.45, 2.5} : TileCost{7.25, 4.7};
        case PLLM_TYPE_Q5_K: return mi == 2 ? TileCost{3.65, 3.0} : TileCost{7.65, 5.25};
        case PLLM_TYPE_Q6_K: return mi == 2 ? TileCost{4.95, 5.1} : TileCost{8.85, 7.1};
        case PLLM_TYPE_IQ4_XS: return mi == 2 ? TileCost{4.75, 3.95} : TileCost{7.9, 5.75};
        case PLLM_TYPE_IQ1_M: return mi == 2 ? TileCost{3.8, 3.9} : TileCost{8.0, 6.2};
        case PLLM_TYPE_IQ3_XXS: return mi == 2 ? TileCost{4.25, 4.6} : TileCost{8.35, 6.6};
        case kFp8Tiles: return mi == 2 ? TileCost{3.7, 3.0} : TileCost{7.8, 5.25};
        default: return mi == 2 ? TileCost{3.9, 3.45} : TileCost{7.8, 5.55};       // IQ2_XXS, IQ2_XS
    }
}

// The plan of this height that costs least: whole rounds, and the tiles beyond them in as many K slices as pay for their partial sums (a second
// launch, and the sums written and read) with the time that more workgroups save.
GemmPlan plan_tiles(int type_id, int t_rows, int n, int bpr, int mi, double& cost_us) {
    TileCost c = tile_cost(type_id, mi);
    const double long_rows = 1.0 + 0.18 * std::max(0, bpr - 20) / 48.0;
    if (mi < 4) c.full *= long_rows;
    c.alone *= long_rows;
    const double start_us = mi == 4 ? 5.0 : 3.0, sum_launch_us = 4.0, bytes_per_us = 10.0e6;
    const int cus = compute_units();
    GemmPlan p = tiles_of(t_rows, n, mi);
    const int rem = p.tiles - p.full_tiles;
    cost_us = p.full_tiles / cus * (c.full * bpr + start_us);
    if (rem == 0) return p;
    double best = 1e30;
    for (int s = 1; s <= 16 && s <= bpr && (s == 1 || rem * s <= 2 * cus); ++s) {
        const int units = rem * s, left = units % cus;
        const double blocks = static_cast<double>(bpr) / s;
        double cost = units / cus * (c.full * blocks + start_us);
        if (left) cost += blocks * std::max(c.alone * (s == 1 ? 1.1 : 1.0), c.full * left / cus) + start_us;
        if (s > 1) cost += sum_launch_us + 2.0 * units * 64 * mi * kBN * sizeof(float) / bytes_per_us;
        if (cost < best - 1e-9) { best = cost; p.slices = s; }
    }
    cost_us += best;
    return p;
}

// The plan of a caller with less workspace than its own plan takes, and of calls that the library's own array holds with this one only: 64 and 128
// rows up to that many tokens, above them 256, but 128 where 256-row tiles would leave the machine mostly empty (a quarter of the compute
// units or less) and where the last one would be half padding while the 128-row tiles still fit one round; slices as their sums' bytes
// at 5 TB/s allow beside 8.8 us per super-block and round.
GemmPlan plan_by_rows(int t_rows, int n, int bpr) {
    constexpr double kRoundUs = 8.8;
    const int cus = compute_units();
    int mi = t_rows <= 64 ? 1 : (t_rows <= 128 ? 2 : 4);
    if (t_rows > 128) {
        const int tiles_n = (n + kBN - 1) / kBN, tiles128 = (t_rows + 127) / 128, tiles256 = (t_rows + 255) / 256;
        if (tiles256 * tiles_n * 4 <= cus || ((tiles128 & 1) && tiles128 * tiles_n <= cus)) mi = 2;
    }
    GemmPlan p = tiles_of(t_rows, n, mi);
    const int rem = p.tiles - p.full_tiles;
    double best = 1e30;
    for (int s = 1; rem > 0 && s <= 16 && s <= bpr; ++s) {
        const double rounds = static_cast<double>((static_cast<long long>(rem) * s + cus - 1) / cus) / s;
        const double cost = rounds * kRoundUs * bpr + (s > 1 ? 2.0 * rem * s * 64 * mi * kBN * 4.0 / 5.0e6 : 0.0);
        if (cost < best - 1e-9) { best = cost; p.slices = s; }
    }
    return p;
}

// The cheaper height; up to 64 tokens the plan by token count (64-row tiles, three of them to a compute unit, take more and shorter slices than the
// costs say: FP8 17408x5120 at 64 rows 43.5 us, in three slices 47.1), up to 128 tokens 128-row tiles.  A call that the library's own array holds with the plan by token
// count keeps a plan that it holds: pllm_gguf_quant_gemm_static_scratch serves what fits the array, with the bits of the call with a
// workspace, which therefore runs the same plan.  FP8 weights have no such entry.
GemmPlan plan_gemm(int type_id, int t_rows, int n, int bpr) {
    double cost = 0.0, cost_high = 0.0;
    if (t_rows <= 64) return plan_by_rows(t_rows, n, bpr);
    GemmPlan p = plan_tiles(type_id, t_rows, n, bpr, 2, cost);
    if (t_rows > 128) {
        const GemmPlan high = plan_tiles(type_id, t_rows, n, bpr, 4, cost_high);
        if (cost_high < cost) p = high;
    }
    if (type_id == kFp8Tiles) return p;
    const size_t staged = gemm_f16_staged_bytes(t_rows, bpr);
    if (staged + partial_bytes(p) <= PLLM_STATIC_SCRATCH_BYTES) return p;
    const GemmPlan base = plan_by_rows(t_rows, n, bpr);
    return staged + partial_bytes(base) <= PLLM_STATIC_SCRATCH_BYTES ? base : p;
}

int launch_tiles_any(int type_id, const TileCall& c, int nt, int workgroups, hipStream_t stream) {
    const int st = launch_tiles_kquant(type_id, c, nt, workgroups, stream);
    return st == PLLM_ERR_UNSUPPORTED ? launch_tiles_codebook(type_id, c, nt, workgroups, stream) : st;
}

int launch_gemm(int type_id, const GemmPlan& p, TileCall c, hipStream_t stream) {
    c.tiles_m = p.tiles / p.tiles_n;
    c.full_tiles = p.slices > 1 ? p.full_tiles : p.tiles;               // unsplit left-over tiles are whole tiles too
    c.rest_tiles = p.tiles - c.full_tiles;
    c.slices = p.slices;
    const int nt = 2 * p.mi;
    const int st = launch_tiles_any(type_id, c, nt, c.full_tiles + c.rest_tiles * c.slices, stream);
    if (st != PLLM_OK || c.rest_tiles == 0) return st;
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3(4 * nt, c.rest_tiles), dim3(256), 0, stream, c, nt);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

}  // namespace

bool gemm_f16_supports(int type_id) {
    return type_id == PLLM_TYPE_Q4_K || type_id == PLLM_TYPE_Q5_K || type_id == PLLM_TYPE_Q2_K || type_id == PLLM_TYPE_IQ2_XXS ||
           type_id == PLLM_TYPE_IQ1_M || type_id == PLLM_TYPE_Q6_K || type_id == PLLM_TYPE_IQ4_XS || type_id == PLLM_TYPE_IQ2_XS ||
           type_id == PLLM_TYPE_IQ3_XXS;
}

size_t gemm_f16_workspace_bytes(int type_id, int rows, int n, int bpr) {
    return gemm_f16_staged_bytes(rows, bpr) + partial_bytes(plan_gemm(type_id, rows, n, bpr));
}

// (a caller with less than its plan takes gets the height by token count)
size_t gemm_f16_least_workspace_bytes(int type_id, int rows, int n, int bpr) {
    return std::min(gemm_f16_workspace_bytes(type_id, rows, n, bpr), gemm_f16_staged_bytes(rows, bpr) + partial_bytes(plan_by_rows(rows, n, bpr)));
}

namespace {
// fp16 rows that the tile kernel reads as the caller holds them: no padding, and 16-byte loads allowed (1999 rows of 17408: 28 us of staging saved).
// Their values, subnormal ones too, are exact operands, but the matrix core aligns the products of a sum by the exponents of the operands as
// stored, where a subnormal counts as 2^-14: sums over nothing but subnormal values lose the bits below.  Distance to float64 over
// the weights as halves, rows of 4096 N(0, 2^2e) values, Q4_K, as held / staged: e >= -14 1.3e-7 / 1.3e-7, -18 3.0e-7 / 1.1e-7, -20 1.3e-6 / 0.9e-7, -24
// (the least subnormal) 1.9e-5 / 0.4e-7; to the weights before that rounding 2.08e-4 either way, at -24 2.09e-4 / 2.08e-4.
bool rows_as_held(const void* x, int x_dtype, int k, int bpr) {
    return x_dtype == PLLM_F16 && k == bpr * 256 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
}

// activations -> fp16 rows + per-row scales at the head of the workspace; returns the partial-tile area
float* stage_activations(const void* x, int x_dtype, int rows, int k, int bpr, void* workspace, const _Float16*& xh_out, const float*& xscale_out,
                         hipStream_t stream, const int64_t* row_map = nullptr) {
    unsigned char* base = static_cast<unsigned char*>(workspace);
    _Float16* xh = reinterpret_cast<_Float16*>(base);
    base += align256(static_cast<size_t>(rows) * bpr * 256 * sizeof(_Float16));
    float* xscale = reinterpret_cast<float*>(base);
    base += align256(static_cast<size_t>(rows) * sizeof(float));
    const bool narrow = (x_dtype == PLLM_BF16 || x_dtype == PLLM_F16) && k % 8 == 0 && bpr * 256 <= 8192 &&
                        reinterpret_cast<uintptr_t>(x) % 16 == 0;
    const bool wide = k % 8 == 0 && bpr * 256 <= kLongRow && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    const bool few = rows <= 512;                  // one row per workgroup while that leaves the grid small
    const uint16_t* x16 = static_cast<const uint16_t*>(x);
    if (narrow && x_dtype == PLLM_BF16 && few)
        hipLaunchKernelGGL((act_f16_rows_kernel<true, 4>), dim3(rows), dim3(256), 0, stream, x16, xh, xscale, rows, k, bpr * 256, row_map);
    else if (narrow && x_dtype == PLLM_BF16)
        hipLaunchKernelGGL((act_f16_rows_kernel<true, 1>), dim3((rows + 3) / 4), dim3(256), 0, stream, x16, xh, xscale, rows, k, bpr * 256, row_map);
    else if (narrow && few)
        hipLaunchKernelGGL((act_f16_rows_kernel<false, 4>), dim3(rows), dim3(256), 0, stream, x16, xh, xscale, rows, k, bpr * 256, row_map);
    else if (narrow)
        hipLaunchKernelGGL((act_f16_rows_kernel<false, 1>), dim3((rows + 3) / 4), dim3(256), 0, stream, x16, xh, xscale, rows, k, bpr * 256, row_map);
    else if (wide && x_dtype == PLLM_BF16)
        hipLaunchKernelGGL((act_f16_long_kernel<PLLM_BF16>), dim3(rows), dim3(kLongThreads), 0, stream, x, xh, xscale, k, bpr * 256, row_map);
    else if (wide && x_dtype == PLLM_F16)
        hipLaunchKernelGGL((act_f16_long_kernel<PLLM_F16>), dim3(rows), dim3(kLongThreads), 0, stream, x, xh, xscale, k, bpr * 256, row_map);
    else if (wide && x_dtype == PLLM_F32)
        hipLaunchKernelGGL((act_f16_long_kernel<PLLM_F32>), dim3(rows), dim3(kLongThreads), 0, stream, x, xh, xscale, k, bpr * 256, row_map);
    else
        hipLaunchKernelGGL(act_f16_kernel, dim3(rows), dim3(256), 0, stream, x, x_dtype, xh, xscale, k, bpr * 256, row_map);
    xh_out = xh;
    xscale_out = xscale;
    return reinterpret_cast<float*>(base);
}

// the rows and the partial-tile area of a call (the area is where it is whether or not the rows are staged: one figure for all types)
int stage_call(TileCall& c, const void* x, int x_dtype, int k, void* workspace, hipStream_t stream) {
    if (rows_as_held(x, x_dtype, k, c.bpr)) {
        c.xh = static_cast<const _Float16*>(x);
        c.partial = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + gemm_f16_staged_bytes(c.t_rows, c.bpr));
        return PLLM_OK;
    }
    c.partial = stage_activations(x, x_dtype, c.t_rows, k, c.bpr, workspace, c.xh, c.xscale, stream);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}
}  // namespace

// columns of the tiles of `count` matrices of one launch (whole tiles each: the plan of a single matrix that wide is theirs)
static int multi_columns(const int* n, int count) {
    int cols = 0;
    for (int m = 0; m < count; ++m) cols += (n[m] + kBN - 1) / kBN * kBN;
    return cols;
}

size_t gemm_f16_multi_workspace_bytes(int type_id, int rows, const int* n, int count, int bpr) {
    return gemm_f16_workspace_bytes(type_id, rows, multi_columns(n, count), bpr);
}
size_t gemm_f16_multi_least_workspace_bytes(int type_id, int rows, const int* n, int count, int bpr) {
    return gemm_f16_least_workspace_bytes(type_id, rows, multi_columns(n, count), bpr);
}

// the plan of a call with this much workspace; false: too little for any
static bool plan_within(int type_id, int rows, int n, int bpr, const void* workspace, size_t workspace_bytes, GemmPlan& p) {
    if (!workspace || workspace_bytes < gemm_f16_least_workspace_bytes(type_id, rows, n, bpr)) return false;
    p = plan_gemm(type_id, rows, n, bpr);
    if (workspace_bytes < gemm_f16_staged_bytes(rows, bpr) + partial_bytes(p)) p = plan_by_rows(rows, n, bpr);
    return true;
}

int gemm_f16(const void* x, int x_dtype, const uint8_t* w, int type_id, void* y, int y_dtype,
             int rows, int k, int n, int bpr, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    return gemm_f16_multi(x, x_dtype, &w, type_id, &y, y_dtype, rows, k, &n, 1, bpr, workspace, workspace_bytes, stream);
}

// Up to four matrices of one format and row length on the same rows: staged once, one launch.  A matrix of few rows leaves most of the
// machine idle by itself (Q5_K, 1024 rows of 3072, 6144 + 1024 + 1024 matrix rows: 190 us one by one, 123 together).
int gemm_f16_multi(const void* x, int x_dtype, const uint8_t* const* ws, int type_id, void* const* ys, int y_dtype,
                   int rows, int k, const int* ns, int count, int bpr, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const int cols = multi_columns(ns, count), n = ns[0];
    const uint8_t* w = ws[0];
    void* y = ys[0];
    GemmPlan p;
    if (!plan_within(type_id, rows, cols, bpr, workspace, workspace_bytes, p)) return PLLM_ERR_WORKSPACE;
    TileCall c{};
    c.w = w; c.y = y; c.y_dtype = y_dtype; c.t_rows = rows; c.n = n; c.bpr = bpr;
    c.more.count = count - 1;
    int first = (n + kBN - 1) / kBN;
    for (int m = 1; m < count; ++m) {
        c.more.w[m - 1] = ws[m];
        c.more.y[m - 1] = ys[m];
        c.more.n[m - 1] = ns[m];
        c.more.first_tile[m - 1] = first;
        first += (ns[m] + kBN - 1) / kBN;
    }
    const int st = stage_call(c, x, x_dtype, k, workspace, stream);
    return st == PLLM_OK ? launch_gemm(type_id, p, c, stream) : st;
}

// FP8 weights [n, k] (k a multiple of 256), scales [ceil(n/128), k/128]
int gemm_f16_fp8(const void* x, int x_dtype, const uint8_t* w, const float* wscale, void* y, int y_dtype,
                 int rows, int k, int n, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (k % 256 != 0) return PLLM_ERR_UNSUPPORTED;
    const int bpr = k / 256;
    GemmPlan p;
    if (!plan_within(kFp8Tiles, rows, n, bpr, workspace, workspace_bytes, p)) return PLLM_ERR_WORKSPACE;
    TileCall c{};
    c.w = w; c.y = y; c.y_dtype = y_dtype; c.t_rows = rows; c.n = n; c.bpr = bpr;
    c.wscale = wscale; c.scale_kb = k / 128;
    const int st = stage_call(c, x, x_dtype, k, workspace, stream);
    return st == PLLM_OK ? launch_gemm(kFp8Tiles, p, c, stream) : st;
}

// ---- routed experts as a batch of tile matmuls ---------------------------------------------------------
size_t gemm_f16_staged_bytes(int rows, int bpr) {
    return align256(static_cast<size_t>(rows) * bpr * 256 * sizeof(_Float16)) + align256(static_cast<size_t>(rows) * sizeof(float));
}

// x rows gathered through row_map (route -> token) into fp16 rows + scales at `staged` (gemm_f16_staged_bytes bytes)
int gemm_f16_stage_rows(const void* x, int x_dtype, const int64_t* row_map, int rows, int k, int bpr, void* staged, hipStream_t stream) {
    const _Float16* xh;
    const float* xscale;
    (void)stage_activations(x, x_dtype, rows, k, bpr, staged, xh, xscale, stream, row_map);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

int gemm_f16_stage_swiglu(const float* g, const float* u, const float* route_weights, float limit, int rows, int inter, int bpr, void* staged,
                          hipStream_t stream) {
    _Float16* hh = static_cast<_Float16*>(staged);
    float* hscale = reinterpret_cast<float*>(static_cast<unsigned char*>(staged) + align256(static_cast<size_t>(rows) * bpr * 256 * sizeof(_Float16)));
    const int kp = bpr * 256;
    if (inter % 4 == 0 && kp <= 1024 * 2)
        hipLaunchKernelGGL(swiglu_f16_held_kernel<2>, dim3(rows), dim3(256), 0, stream, g, u, route_weights, limit, hh, hscale, inter, kp);
    else if (inter % 4 == 0 && kp <= 1024 * 8)
        hipLaunchKernelGGL(swiglu_f16_held_kernel<8>, dim3(rows), dim3(256), 0, stream, g, u, route_weights, limit, hh, hscale, inter, kp);
    else
        hipLaunchKernelGGL(swiglu_f16_rows_kernel, dim3((rows + 3) / 4), dim3(256), 0, stream, g, u, route_weights, limit, hh, hscale, rows, inter, kp);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

// rows of a group's tiles: one tile for most groups where the average allows it.  32 rows where few groups have more (their four workgroups to a
// compute unit wait for memory less; us, 32 / 64 rows: IQ2_XXS / Q2_K, 256 experts, 8 routes on average 655 / 712, 22 routes 747 / 766; where a
// fifth and more of the groups need two of them: Q4_K / Q6_K, 128 experts, 28 routes 582 / 509, Q4_K 32 routes 238 / 204)
static int grouped_height(int rows, int groups) {
    const int avg = (rows + groups - 1) / groups;
    return avg <= 20 ? 32 : avg <= 48 ? 64 : (avg <= 128 ? 128 : 256);
}

int gemm_f16_grouped_list(const int32_t* seg, int rows, int groups, void* list_ws, hipStream_t stream) {
    return moe_tile_list(seg, groups, grouped_height(rows, groups), rows, list_ws, stream);
}

// ys[m][r, :] (float32 [rows, n]) = staged row r, or row_map[r] of the `staged_rows` staged ones, . dequant(W_m,g)^T for the rows r of every group g, up
// to four matrices per group in one launch.  The grid counts row tiles, not groups times the rows that one group could have: 128 experts and
// 512 tokens had seven workgroups without work for each one with some, and two XCDs of eight without any.
int gemm_f16_grouped(const void* staged, int staged_rows, const int64_t* row_map, const uint8_t* const* ws, int type_id, size_t group_stride, const void* list_ws,
                     int groups, float* const* ys, int count, int rows, int n, int bpr, hipStream_t stream) {
    const int height = grouped_height(rows, groups), tiles_n = (n + kBN - 1) / kBN;
    TileCall c{};
    c.xh = static_cast<const _Float16*>(staged);
    c.xscale = reinterpret_cast<const float*>(static_cast<const unsigned char*>(staged) + align256(static_cast<size_t>(staged_rows) * bpr * 256 * sizeof(_Float16)));
    c.w = ws[0]; c.y = ys[0]; c.y_dtype = PLLM_F32; c.t_rows = rows; c.n = n; c.bpr = bpr;
    c.row_map = row_map; c.group_stride = group_stride;
    c.more.count = count - 1;
    for (int m = 1; m < count; ++m) {
        c.more.w[m - 1] = ws[m];
        c.more.y[m - 1] = ys[m];
        c.more.n[m - 1] = n;
        c.more.first_tile[m - 1] = m * tiles_n;
    }
    c.list = static_cast<const int4*>(list_ws);
    c.list_tiles = moe_tile_list_count(list_ws, rows);
    c.list_columns = count * tiles_n;
    const long long workgroups = (static_cast<long long>(moe_tile_list_most(rows, groups, height)) + 7) / 8 * 8 * c.list_columns;
    if (workgroups > INT32_MAX / kTileThreads) return PLLM_ERR_UNSUPPORTED;      // (a grid's threads are counted in 32 bits)
    return launch_tiles_any(type_id, c, height / 32, static_cast<int>(workgroups), stream);
}

}  // namespace pllm
