// The prompt tile kernel: y[T, N] = x[T, K] . dequant(W)[N, K]^T over raw super-blocks on f16 MFMA.  Formats: tile_formats.h; plan,
// activation staging and dispatch: gemm_f16.hip.
//
// A workgroup of four waves owns an output tile of 32 NT tokens (NT = 1 for lists, 2, 4, 8) x 256 weight rows and walks K in steps of 64.
//  * Weights stay in the wave that owns them: wave w has rows 64 w .. 64 w + 63, reads their raw blocks itself, a step or more ahead, and
//    decodes them in registers straight into the operands of v_mfma_f32_32x32x16_f16 (lane = row, half of the wave = half of a
//    sub-block).  No decoded weight passes through LDS and none is decoded twice in a tile.
//  * The tokens' fp16 rows go through a ring of four LDS stages that direct-to-LDS loads fill three steps ahead.  Rows lie 128 bytes apart,
//    unpadded (a wave instruction of such a load writes eight rows); the 16-byte pieces of row r are stored at piece ^ ((r / 2) % 8), which
//    keeps the 16-byte reads free of bank conflicts.  An operand read serves both 32-row blocks of the wave.
//  * One barrier per step, after its first quarter: by then the wave's loads of the next step have landed, and every read of the step before has
//    returned, so its stage can be filled again.
//  * Weights are decoded one instruction's operands ahead (16 registers of operands, not 32).  Between two matrix instructions (32 cycles
//    each) stand at most the decode of two weights, an operand read and a load: five vector
//    instructions are hidden behind one matrix instruction, and a wave that is alone on its SIMD (NT = 8: 256 accumulators) has
//    nobody else to hide them.  sched_barrier keeps the compiler from bunching them.
//  * Lanes hold tokens and registers hold weight rows (the weights are the matrix instruction's A rows), so four neighbouring outputs of
//    a token leave together, through LDS, in whole 128-byte lines.
// What bounds it, by the counters (cycles in which the matrix cores work, and the clock).  Launches that give every SIMD two waves: the clock, which
// gives way as the units fill (Q4_K 17408x5120 at 2048 rows 78 % at 1.37 GHz, 16384x5120 at 1024 rows 74 % at 1.41).  With one wave per SIMD: the
// wave's own chain of decode and operand reads, 56 - 59 % at 1.61 - 1.66 GHz (Q4_K and FP8, 512 rows), 66 % at 1.51 at NT = 8 (Q5_K 5120x17408).  Few
// or short tiles: fill, drain and that chain (Q5_K, 1024 rows: 256 tiles of 12 blocks 46 % at 1.76 GHz, 96 tiles in two slices of 12 blocks 35 % at
// 1.93).  us per call, the kernel before (decoded weights through LDS, eight waves) / this one: Q4_K 16384x5120 at 1024 rows 202 / 159, at 512 rows (NT = 4) 126 / 101, 17408x5120 at 2048 rows 445 / 347, Q6_K 16384x5120 at
// 1024 rows 227 / 190, Q4_K 17408x5120 at 512 rows 147 / 101.  Measured and not kept: other orders of the instructions, the weights as the
// second operand, whole blocks of weights loaded at once, staged rows laid out stage by stage (all within 1 %); token loads in the last
// quarter of a step (3 - 5 % slower than in the second).
#pragma once

#include "block_mfma.h"
#include "tile_formats.h"

#include <utility>

namespace pllm {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));

// fn(integral_constant 0), ..., fn(integral_constant N - 1): every index a constant, so that arrays stay in registers
template <typename Fn, int... I>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, Fn&& fn) { (fn(std::integral_constant<int, I>{}), ...); }
template <int N, typename Fn>
__device__ __forceinline__ void each(Fn&& fn) { each_of(std::make_integer_sequence<int, N>{}, fn); }

constexpr int kTileN = 256, kTileStages = 4, kTileRow = 144;      // kTileRow: bytes between rows of the store's staging area

// Further matrices of one launch, of the same format and row length on the same activation rows: the tiles along N run through the
// launch's first matrix and then through these.
struct MoreMatrices {
    const uint8_t* w[3];
    void* y[3];
    int n[3], first_tile[3], count;
    // the matrix of tile tn along N: w, y and n become its own, tn counts from its first tile
    __device__ __forceinline__ void pick(int& tn, const uint8_t*& mw, void*& my, int& mn) const {
        int from = 0;
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if (m < count && tn >= first_tile[m]) {
                mw = w[m];
                my = y[m];
                mn = n[m];
                from = first_tile[m];
            }
        tn -= from;
    }
};

// One launch.  Tiles are numbered with the token tiles of a column of tiles next to each other.  Workgroups [0, full_tiles) take whole
// tiles; the others one slice of K each of the tiles from full_tiles on, whose float32 sums go to `partial`.  xscale: factor of every
// token's row, or null.  With `list` the launch is a batch of products (routed experts): every group (expert) has its own matrix, `group_stride`
// bytes from the one before, and its own run of output rows; list = the row tiles of all groups {group, first row, rows, 0}, *list_tiles of them.
// row_map (with a list): output row -> activation row, or null where they are the same.
struct TileCall {
    const _Float16* xh;
    const float* xscale;
    const uint8_t* w;
    void* y;
    float* partial;
    const float* wscale;
    const int4* list;
    const int32_t* list_tiles;
    const int64_t* row_map;
    size_t group_stride;
    MoreMatrices more;
    int y_dtype, t_rows, n, bpr, tiles_m, full_tiles, rest_tiles, slices, scale_kb;
    int list_columns;                            // tiles along N of a list's launch, over all of its matrices
};

// Workgroup -> tile and slice.  Hardware deals workgroups to the eight XCDs in turn; numbered back, an XCD's workgroups are neighbours:
// they share the weights of a column of tiles (and the slice of them) in that XCD's L2.
struct TileOf { int tile, slice, slices, slot; };
__device__ __forceinline__ TileOf tile_of(const TileCall& c) {
    auto by_xcd = [](int i, int count) { const int per = count >> 3; return i < per * 8 ? (i & 7) * per + (i >> 3) : i; };
    const int wg = blockIdx.x;
    if (wg < c.full_tiles) return {by_xcd(wg, c.full_tiles), 0, 1, 0};
    const int r = by_xcd(wg - c.full_tiles, c.rest_tiles * c.slices), whole_cols = c.rest_tiles / c.tiles_m * c.tiles_m * c.slices;
    int t, s;
    if (r < whole_cols) {
        const int col = r / (c.tiles_m * c.slices), in = r % (c.tiles_m * c.slices);
        t = col * c.tiles_m + in % c.tiles_m;
        s = in / c.tiles_m;
    } else {
        const int left = c.rest_tiles % c.tiles_m, in = r - whole_cols;
        t = c.rest_tiles - left + in % left;
        s = in / left;
    }
    return {c.full_tiles + t, s, c.slices, t * c.slices + s};
}

template <typename F, int NT>
constexpr int tile_lds_bytes() {                  // the stages and the codebook; at the end the four waves' staging areas of the store
    constexpr int loop = kTileStages * 32 * NT * 128 + F::kTableBytes, store = 4 * 2 * 32 * kTileRow;
    return loop > store ? loop : store;
}

// Workgroups that a compute unit has registers for: one at NT = 8 (256 accumulators a lane), two at NT = 4 and 2 in every format, three at NT = 1.
// (IQ4_XS, whose parts are twice as large, with one at NT = 4: 17408x5120 at 512 rows 123 us, with two 116, at 777 rows 190 / 176, elsewhere level.)
template <typename F, int NT>
__global__ __launch_bounds__(kTileThreads, NT == 8 ? 1 : NT == 1 ? 3 : 2) void gemm_tile_kernel(const TileCall c) {
    constexpr int kBM = 32 * NT, kStage = kBM * 128, kSets = 4 / F::kPairs, kPerInstruction = NT <= 2 ? 4 / NT : 1;
    // Weight loads of the two steps before, one vector load per row block and part at least.  What the compiler makes of load_part is its own affair:
    // tests/test_tile_kernel_waits.py counts the loads behind every wait in the compiled kernels.
    constexpr int kNewerParts = 4 / F::kPairs;
    extern __shared__ __align__(1024) unsigned char smem[];
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte_ptr)smem));
    unsigned char* const table = smem + kTileStages * kStage;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 31, hs = lane >> 5;
    TileOf at;
    int col_tile, t0, t_rows = c.t_rows, n = c.n;
    size_t group_offset = 0;
    if (c.list) {
        // An XCD's workgroups (every eighth) take all columns of a row tile one after the other, so its activation rows are in that XCD's L2.
        // Workgroups past the end of the list come last.
        const int i = blockIdx.x >> 3, entry = i / c.list_columns * 8 + (blockIdx.x & 7);
        if (entry >= *c.list_tiles) return;
        const int4 t = c.list[entry];
        at = {0, 0, 1, 0};
        col_tile = i % c.list_columns;
        t0 = t.y;
        t_rows = t.y + t.z;
        group_offset = static_cast<size_t>(t.x) * c.group_stride;
    } else {
        at = tile_of(c);
        col_tile = at.tile / c.tiles_m;
        t0 = (at.tile % c.tiles_m) * kBM;
    }
    const bool whole = at.slices == 1;
    const uint8_t* w = c.w;
    void* y = c.y;
    c.more.pick(col_tile, w, y, n);
    w += group_offset;
    const int n0 = col_tile * kTileN, bpr = c.bpr;
    const int b0 = static_cast<int>(static_cast<long long>(at.slice) * bpr / at.slices);
    const int b1 = static_cast<int>(static_cast<long long>(at.slice + 1) * bpr / at.slices);

    // Token rows: the wave's kilobytes NT wave .. of a stage (eight rows each; lane = row in the piece, position in the row).  Offsets of 32 bits
    // from the wave's first row: 63 rows of less than 2^25 columns (mapped rows: from the first of all).
    const uint32_t x_pitch = static_cast<uint32_t>(bpr) * 512u;
    const int xrow0 = c.row_map ? 0 : min(t0 + 8 * NT * wave, t_rows - 1);
    uint32_t xoff[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int row = 8 * (NT * wave + j) + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        const int from = min(t0 + row, t_rows - 1);
        xoff[j] = static_cast<uint32_t>((c.row_map ? static_cast<int>(c.row_map[from]) : from) - xrow0) * x_pitch + 16u * piece;
    }
    const unsigned char* const xbase = reinterpret_cast<const unsigned char*>(c.xh) + static_cast<size_t>(xrow0) * x_pitch;
    // (Past the end the last step is fetched again and dropped: no branch around the loads.  Short slices are mostly ends, so what is dropped there
    // comes from one line: the lanes' offsets masked away, for the weights at every height.)
    auto x_step = [&](int step) { return xbase + static_cast<size_t>(min(step, 4 * b1 - 1)) * 128; };
    auto x_piece = [&](const unsigned char* src, uint32_t mask, int stage, int j) {
        lds_dma16_at(src, NT <= 2 ? xoff[j] & mask : xoff[j], lds0 + stage * kStage + (NT * wave + j) * 1024);
    };

    // weight rows of the lane: l and 32 + l of the wave's 64
    const uint32_t row_bytes = static_cast<uint32_t>(bpr) * F::kBlockBytes;
    const int wrow0 = min(n0 + 64 * wave, n - 1);
    const uint8_t* const wbase = w + static_cast<size_t>(wrow0) * row_bytes;
    uint32_t woff[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) woff[r] = static_cast<uint32_t>(min(n0 + 64 * wave + 32 * r + l, n - 1) - wrow0) * row_bytes;
    const float* const srow = c.wscale + static_cast<size_t>(wrow0 >> 7) * c.scale_kb;        // FP8 only (the wave's 64 rows share a scale block)

    const int swizzle = (l >> 1) & 7;
    uint32_t aoff[2][2];                         // [half step][instruction]: where the lane's eight values of a token stand in a stage
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i) aoff[e][i] = l * 128 + 16 * ((4 * e + 2 * hs + i) ^ swizzle);
    auto operand = [&](int stage, int e, int i, int tb) -> half8 {
        return *reinterpret_cast<const half8*>(smem + stage * kStage + tb * 4096 + aoff[e][i]);
    };

    floatx16 acc[NT][2];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    typename F::Head head[2];
    typename F::Expanded ex[2];
    typename F::Part part[kSets][2];
    typename F::Look look[2];
    typename F::Scale sc[2];
    const uint8_t* wb = wbase + static_cast<size_t>(b0) * F::kBlockBytes;
    // Token rows first, weights behind them: loads complete in order, so the first block's first part, which everything waits for, brings
    // three stages with it.
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const unsigned char* src = x_step(4 * b0 + s);
#pragma unroll
        for (int j = 0; j < NT; ++j) x_piece(src, ~0u, s, j);
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) F::load_head(head[r], wb + woff[r], hs, srow, b0);
#pragma unroll
    for (int s = 0; s < kSets; ++s)
#pragma unroll
        for (int r = 0; r < 2; ++r) F::load_part(part[s][r], wb + woff[r], s * F::kPairs, hs);
    if constexpr (F::kTableBytes > 0) {
        F::stage_table(table);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) F::expand(head[r], ex[r]);

    // A sub-step (p, e, i) is one matrix instruction of K = 16 per token and row block.  While one runs, the next one's eight weights per row
    // block are decoded in eight quanta of two weights: row block q / 4, weights 2 (q % 4) and the next one.  Codebook entries are looked up
    // four quanta ahead.
    uint32x4 b[2][2];                            // operands: [sub-step parity][row block]
    auto look_up = [&](int p, int e, int i, int r) {
        if constexpr (F::kLooks) F::look(look[r], part[p / F::kPairs][r], p, e, hs, i, table);
    };
    auto quantum = [&](auto qc, auto ic, int p, int e) {
        constexpr int q = decltype(qc)::value, i = decltype(ic)::value, r = q >> 2;
        const typename F::Part& codes = part[p / F::kPairs][r];
        if (q % 4 == 0 && i == 0) sc[r] = F::scale(ex[r], codes, p, e, hs);
        b[i][r][q & 3] = F::template pair<4 * i + (q & 3)>(ex[r], codes, look[r], sc[r], p, e, hs);
    };
    look_up(0, 0, 0, 0);
    look_up(0, 0, 0, 1);
    each<8>([&](auto qc) { quantum(qc, std::integral_constant<int, 0>{}, 0, 0); });
    look_up(0, 0, 1, 0);
    wait_vm<2 * (kSets - 1)>();                  // (the later parts' loads stand behind the stages')
    __syncthreads();
    half8 a[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) a[tb] = operand(0, 0, 0, tb);

    for (int blk = b0; blk < b1; ++blk) {
        const int nb = min(blk + 1, b1 - 1);
        const uint8_t* const wn = wbase + static_cast<size_t>(nb) * F::kBlockBytes;
        const uint32_t mask = blk + 1 < b1 ? ~0u : 0u;
        each<16>([&](auto sc_) {
            constexpr int s = decltype(sc_)::value, p = s >> 2, e = (s >> 1) & 1, i = s & 1;
            constexpr int dp = ((s + 1) & 15) >> 2, de = ((s + 1) >> 1) & 1, di = 1 - i;      // the sub-step decoded meanwhile
            constexpr int fp = ((s + 2) & 15) >> 2, fe = ((s + 2) >> 1) & 1;                  // and the one after it
            // Loads complete in order, so a wait for weights covers the token loads ahead of them: it stands here, before this step's
            // token loads, and not at the first use of either row block.
            if (e == 0 && i == 1 && ((p + 1) & 3) % F::kPairs == 0) {
#pragma unroll
                for (int r = 0; r < 2; ++r) F::hold(part[((p + 1) & 3) / F::kPairs][r]);
            }
            if (s == 15) {
#pragma unroll
                for (int r = 0; r < 2; ++r) F::expand(head[r], ex[r]);
            }
            const unsigned char* const src = x_step(4 * blk + p + 3);
            each<2 * NT>([&](auto mc) {
                constexpr int m = decltype(mc)::value, tb = m >> 1, rb = m & 1;
                __builtin_amdgcn_sched_barrier(0);
                acc[tb][rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, b[i][rb]), a[tb], acc[tb][rb], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (rb == 1) a[tb] = operand(dp, de, di, tb);
                each<kPerInstruction>([&](auto qc) {
                    constexpr int q = NT == 8 ? m / 2 : kPerInstruction * m + decltype(qc)::value;
                    if (NT == 8 && rb == 1) return;
                    if (q == 0) look_up(dp, de, di, 1);
                    if (q == 4) look_up(fp, fe, i, 0);
                    quantum(std::integral_constant<int, q>{}, std::integral_constant<int, di>{}, dp, de);
                });
                if (e == 0 && i == 1 && rb == 1) x_piece(src, p == 0 ? ~0u : mask, (p + 3) & 3, tb);
            });
            __builtin_amdgcn_sched_barrier(0);
            if (e == 0 && i == 0) {
                // This wave's loads of the next step have landed: behind them stand the tokens of the one after and the weights of two steps.  (With the
                // tokens alone counted, 64-row tiles waited for what they had asked for one step ago.)
                wait_vm<NT + kNewerParts>();
                __builtin_amdgcn_s_barrier();            // (everybody's; and every read of the step before has returned)
            }
            if (e == 1 && i == 0) {                      // (the pair's last weights are decoded)
                if (p == 1) {
#pragma unroll
                    for (int r = 0; r < 2; ++r) F::load_head(head[r], wn + (woff[r] & mask), hs, srow, nb);
                }
                if ((p + 1) % F::kPairs == 0) {
#pragma unroll
                    for (int r = 0; r < 2; ++r) F::load_part(part[p / F::kPairs][r], wn + (woff[r] & mask), p, hs);
                }
            }
        });
    }
    wait_vm<0>();                                        // the dropped loads past the end: nothing may arrive in LDS from here on

    // D[m][n]: the lane holds token n = l of block tb and weight rows m = 8 (v / 4) + 4 hs + v % 4 of row block r
    if (!whole) {                                        // raw sums of this slice, as the lanes hold them: [wave][tb][r][v / 4][lane][v % 4]
        float4* const dst = reinterpret_cast<float4*>(c.partial) + static_cast<size_t>(at.slot) * (kBM * kTileN / 4) + wave * (NT * 8 * 64) + lane;
        each<8 * NT>([&](auto ic) {
            if (t0 + 32 * (decltype(ic)::value / 8) + l >= t_rows) return;       // (nobody reads the sums of tokens past the end)
            constexpr int tb = decltype(ic)::value / 8, r = decltype(ic)::value / 4 % 2, q = decltype(ic)::value % 4;
            dst[decltype(ic)::value * 64] = make_float4(acc[tb][r][4 * q], acc[tb][r][4 * q + 1], acc[tb][r][4 * q + 2], acc[tb][r][4 * q + 3]);
        });
        return;
    }
    float xs[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) {
        const int row = min(t0 + 32 * tb + l, t_rows - 1);
        xs[tb] = c.xscale ? c.xscale[c.row_map ? c.row_map[row] : row] : 1.0f;
    }
    __syncthreads();                                     // (the stages are the waves' own from here on)
    unsigned char* const mine = smem + wave * (2 * 32 * kTileRow);
    const int y_dtype = c.y_dtype, c0 = n0 + 64 * wave, orow = lane >> 3, piece = lane & 7;
    const bool wide = y_dtype == PLLM_F32 ? (n & 3) == 0 : (n & 7) == 0;
    const bool vector_ok = wide && !(y_dtype & kAccumulateInto) && reinterpret_cast<uintptr_t>(y) % 16 == 0;
    if (vector_ok && y_dtype != PLLM_F32) {
        uint16_t* const out = static_cast<uint16_t*>(y) + c0 + 8 * piece;
        const bool col_ok = c0 + 8 * piece < n;
        each<NT>([&](auto tc) {
            constexpr int tb = decltype(tc)::value;
            unsigned char* const area = mine + (tb & 1) * (32 * kTileRow);
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float v0 = acc[tb][r][4 * q] * xs[tb], v1 = acc[tb][r][4 * q + 1] * xs[tb], v2 = acc[tb][r][4 * q + 2] * xs[tb], v3 = acc[tb][r][4 * q + 3] * xs[tb];
                    uint2 o;
                    if (y_dtype == PLLM_BF16) {
                        o.x = from_float<bf16_t>(v0).bits | (static_cast<uint32_t>(from_float<bf16_t>(v1).bits) << 16);
                        o.y = from_float<bf16_t>(v2).bits | (static_cast<uint32_t>(from_float<bf16_t>(v3).bits) << 16);
                    } else {
                        o = make_uint2(pack_halves(v0, v1), pack_halves(v2, v3));
                    }
                    *reinterpret_cast<uint2*>(area + l * kTileRow + 64 * r + 16 * q + 8 * hs) = o;
                }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint4 o = *reinterpret_cast<const uint4*>(area + (8 * j + orow) * kTileRow + 16 * piece);
                const int row = t0 + 32 * tb + 8 * j + orow;
                if (row < t_rows && col_ok) *reinterpret_cast<uint4*>(out + static_cast<size_t>(row) * n) = o;
            }
        });
        return;
    }
    each<2 * NT>([&](auto ic) {
        constexpr int tb = decltype(ic)::value / 2, r = decltype(ic)::value % 2;
        unsigned char* const area = mine + r * (32 * kTileRow);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(area + l * kTileRow + 32 * q + 16 * hs) =
                make_float4(acc[tb][r][4 * q] * xs[tb], acc[tb][r][4 * q + 1] * xs[tb], acc[tb][r][4 * q + 2] * xs[tb], acc[tb][r][4 * q + 3] * xs[tb]);
        const int col = c0 + 32 * r + 4 * piece;
        for (int j = 0; j < 4; ++j) {
            const float4 o = *reinterpret_cast<const float4*>(area + (8 * j + orow) * kTileRow + 16 * piece);
            const int row = t0 + 32 * tb + 8 * j + orow;
            if (row >= t_rows) continue;
            const size_t to = static_cast<size_t>(row) * n + col;
            if (vector_ok) {
                if (col < n) *reinterpret_cast<float4*>(static_cast<float*>(y) + to) = o;
            } else {
                if (col < n) store_any(y, y_dtype, to, o.x);
                if (col + 1 < n) store_any(y, y_dtype, to + 1, o.y);
                if (col + 2 < n) store_any(y, y_dtype, to + 2, o.z);
                if (col + 3 < n) store_any(y, y_dtype, to + 3, o.w);
            }
        }
    });
}

template <typename F, int NT>
int launch_tile_kernel(const TileCall& c, int workgroups, hipStream_t stream) {
    auto kern = gemm_tile_kernel<F, NT>;
    constexpr int lds = tile_lds_bytes<F, NT>();
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return PLLM_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(kern, dim3(workgroups), dim3(kTileThreads), lds, stream, c);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}
template <typename F, bool LISTS = true>
int launch_tiles(const TileCall& c, int nt, int workgroups, hipStream_t stream) {
    if constexpr (LISTS)
        if (nt == 1) return launch_tile_kernel<F, 1>(c, workgroups, stream);
    switch (nt) {
        case 2: return launch_tile_kernel<F, 2>(c, workgroups, stream);
        case 4: return launch_tile_kernel<F, 4>(c, workgroups, stream);
        default: return launch_tile_kernel<F, 8>(c, workgroups, stream);
    }
}

// by type id (kFp8Tiles: FP8 weights); two files, so that they compile side by side
int launch_tiles_kquant(int type_id, const TileCall& c, int nt, int workgroups, hipStream_t stream);      // Q2_K, Q4_K, Q5_K, Q6_K, IQ4_XS, FP8
int launch_tiles_codebook(int type_id, const TileCall& c, int nt, int workgroups, hipStream_t stream);    // IQ2_XXS, IQ2_XS, IQ3_XXS, IQ1_M

}  // namespace pllm
