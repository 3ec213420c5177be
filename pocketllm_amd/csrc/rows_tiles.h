// What the kernels that multiply a few dozen activation rows with raw blocks share (gemm_q8_0.hip, gemm_kquant_rows.hip): a workgroup owns
// 32 MB matrix rows and 32 weight rows per wave over a slice of K, a step is 256 columns; sums of slices leave in lane order and are added
// in slice order by a second kernel.
#pragma once

#include "block_mfma.h"
#include "pllm_internal.h"

#include <algorithm>
#include <type_traits>

namespace pllm {
namespace {

constexpr int kWaveCols = 32;
constexpr int tile_waves(int mb) { return mb == 1 ? 4 : 8; }                     // (32 rows: two workgroups fit a compute unit's LDS)

template <int I, int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}
struct RowsArgs {
    const _Float16* rows;                            // matrix rows, kp halves each
    const float* unscale;                            // per activation row: 1 / its power of two (null: rows as the caller holds them)
    const uint8_t* w;
    void* y;
    float* partial;                                  // null: whole K per workgroup, results go to y
    int y_dtype, m_rows, n, blocks, kp, row_tiles, col_tiles, slices, steps, steps_more;
};

__device__ __forceinline__ float row_factor(const RowsArgs& a, int row) { return a.unscale ? a.unscale[row] : 1.0f; }

// fp16 rows that need no padding are read as the caller holds them, without the launch that scales rows by powers of two.  The sums keep all their bits for rows
// of any size: the matrix core aligns products by the exponents as stored, where a subnormal counts as 2^-14, with 24 bits below; the operands of these kernels are
// whole numbers of up to 2^12 and fp16 values multiples of 2^-24, so no product has a bit further down.  (Decoded weights have: sizes in gemm_f16.hip.)
// us, staged / as held: Q6_K 5120x17408 7 rows 30.0 / 26.0, 2048x3072 16 rows 11.7 / 8.8, 5120x5120 16 rows 17.1 / 14.3,
// 64 rows 24.3 / 21.8; IQ4_XS 17408x5120 16 rows 26.7 / 23.7; Q2_K 5120x5120 8 rows 15.2 / 11.8; Q8_0 4096x4096 32 rows 16.3 / 13.7, 203 rows 27.1 / 24.6.
inline bool rows_as_held(const void* x, int x_dtype, int k, int kp) { return x_dtype == PLLM_F16 && k == kp && reinterpret_cast<uintptr_t>(x) % 16 == 0; }

// sums of the slices, in slice order: thread = four matrix rows of one column
template <int MB, int TERMS>
__global__ __launch_bounds__(256) void rows_reduce_kernel(RowsArgs a) {
    constexpr int kWaves = tile_waves(MB), kCols = kWaves * kWaveCols;
    const size_t per_slice = static_cast<size_t>(a.col_tiles) * a.row_tiles * kWaves * MB * 4 * 64, i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= per_slice) return;
    const int lane = static_cast<int>(i & 63), q4 = static_cast<int>(i >> 6) & 3, m = static_cast<int>(i >> 8) % MB;
    const size_t wt = (i >> 8) / MB;
    const int wave = static_cast<int>(wt % kWaves), rt = static_cast<int>(wt / kWaves % a.row_tiles), ct = static_cast<int>(wt / kWaves / a.row_tiles);
    const int col = ct * kCols + wave * kWaveCols + (lane & 31), row0 = rt * 32 * MB + 32 * m + 8 * q4 + 4 * (lane >> 5);
    if (col >= a.n || row0 >= a.m_rows) return;
    const float4* src = reinterpret_cast<const float4*>(a.partial) + i;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // up to 16 slices requested together, added in slice order
    auto add = [&](auto batch) {
        constexpr int kBatch = decltype(batch)::value;
        for (int k0 = 0; k0 < a.slices; k0 += kBatch) {
            float4 v[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) v[k] = src[min(k0 + k, a.slices - 1) * per_slice];
#pragma unroll
            for (int k = 0; k < kBatch; ++k)
                if (k0 + k < a.slices) { s.x += v[k].x; s.y += v[k].y; s.z += v[k].z; s.w += v[k].w; }
        }
    };
    if (a.slices <= 4) add(std::integral_constant<int, 4>{});
    else if (a.slices <= 8) add(std::integral_constant<int, 8>{});
    else add(std::integral_constant<int, 16>{});
    const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
    for (int j = 0; j < 4; j += TERMS) {
        const int row = (row0 + j) / TERMS;
        const float t = TERMS == 2 ? v[j] + v[j + 1] : v[j];
        if (row0 + j < a.m_rows) store_any(a.y, a.y_dtype, static_cast<size_t>(row) * a.n + col, t * row_factor(a, row));
    }
}

// the activation rows of a tile (64 at most, 256 halves per step) are addressed with 32-bit byte offsets
inline bool rows_offsets_fit(int steps) { return static_cast<long long>(steps) * 256 * sizeof(_Float16) * 64 <= (1ll << 32); }

// us: a workgroup's start, a step at 32 and at 64 matrix rows
struct RowsCost { double start_us, step1_us, step2_us; };
struct RowsPlan { int mb, row_tiles, col_tiles, slices; };

inline RowsPlan plan_rows(int m_rows, int n, int steps, const RowsCost& cost_of) {
    RowsPlan p;
    p.mb = m_rows <= 32 ? 1 : 2;
    const int cols = tile_waves(p.mb) * kWaveCols;
    p.row_tiles = (m_rows + 32 * p.mb - 1) / (32 * p.mb);
    p.col_tiles = (n + cols - 1) / cols;
    const int tiles = p.row_tiles * p.col_tiles, places = (p.mb == 1 ? 2 : 1) * compute_units();
    // slices: rounds of the machine, whose workgroups take start + step us per 256 columns, against moving the partial sums (about
    // 4 TB/s out and in, and a launch)
    const double start_us = cost_of.start_us, step_us = p.mb == 2 ? cost_of.step2_us : cost_of.step1_us;
    p.slices = 1;
    double best = 1e30;
    for (int s = 1; s <= std::min(steps, 32); ++s) {
        const double rounds = static_cast<double>((static_cast<long long>(tiles) * s + places - 1) / places);
        const double move = s > 1 ? 4.0 + 2.0 * s * tiles * (32.0 * p.mb * cols * 4.0) / 4.0e6 : 0.0;
        const double cost = rounds * (start_us + step_us * ((steps + s - 1) / s)) + move;
        if (cost < best) { best = cost; p.slices = s; }
    }
    return p;
}

// activation rows and their scales, then the partial sums
struct RowsWorkspace { size_t unscale, partial, bytes; };
inline RowsWorkspace rows_workspace(int rows, int terms, int n, int steps, const RowsCost& cost) {
    const RowsPlan p = plan_rows(rows * terms, n, steps, cost);
    RowsWorkspace ws;
    ws.unscale = align256(static_cast<size_t>(rows) * terms * steps * 256 * sizeof(_Float16));
    ws.partial = ws.unscale + align256(static_cast<size_t>(rows) * sizeof(float));
    ws.bytes = ws.partial + (p.slices > 1 ? static_cast<size_t>(p.slices) * p.row_tiles * p.col_tiles * 32 * p.mb * tile_waves(p.mb) * kWaveCols * sizeof(float) : 0);
    return ws;
}

}  // namespace
}  // namespace pllm
