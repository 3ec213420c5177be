// Routed experts of several tokens, IQ2_XXS gate / up and IQ1_M down: tiles of up to 64 routes against weights decoded in registers.
//
// The integer weights of both formats, code times group scale, are exact in half precision, and so are bf16 / fp16 activations
// scaled by a power of two per row (float32 rows go in as two half-precision terms = two matrix rows).  A workgroup takes a tile
// of one expert's routes, and every wave owns 64 weight rows (gate and up of the same 32 hidden columns, or 64 rows of the down
// projection) over all of K.  A weight's codes go from memory to the lane that needs them as a matrix operand and are decoded there
// once per tile: lane = one codebook entry (eight weights) of a weight row per matrix instruction, v_mfma_f32_32x32x16_f16 for
// tiles of 32 and 64 matrix rows, v_mfma_f32_16x16x32_f16 for tiles of 16.  The lanes of a row split its block into halves
// (quarters) and step through them side by side; the activation operand follows that order.  Activation rows come to LDS by
// direct-to-LDS loads, 512 bytes per row and block; 16-byte piece p of row r lies at position p ^ (r % 32), so rows read at one
// piece meet no bank twice.  The matrix cores sum over a block, whose scale goes on as the sums join the totals.
//
// Two forms.  Up to 12 matrix rows per expert on average: tiles of 16 rows, twelve waves, all of K of the activation rows in LDS
// before the loop (96 KB at 3072 columns), no barrier inside it.  Above: tiles of 64 (or 32) rows, eight waves, two blocks of
// activations in LDS, one barrier per block.  256 experts of 3072 -> 1536 -> 3072, us for gate / up + down: 2048 routes 303 + 139 in the
// first form, 372 + 157 in the second; 8192 routes 437 + 180 in the second.  (The form before, one decode per 16 routes with the
// activations in registers: 336 + 161 at 2048 routes, 1960 + 986 at 8192 unevenly spread ones, where an expert with many routes kept
// four workgroups busy long after the others had ended: the tiles of all experts now go into one list.)
//
// Bound: LDS reads (two codebook reads of 16 bytes per eight IQ2_XXS weights, one per eight IQ1_M weights, eight cycles each) and the
// vector ALU beside the matrix instructions; both are paid once per tile.  Gate / up at 2048 routes: LDS busy for 67 % of the time
// (nearly half of that counted as bank conflicts), vector ALU 59 %, matrix cores 13 %; at 8192 routes 44 %, 46 % and 25 %.
#include "block_mfma.h"
#include "pllm_internal.h"

#include <algorithm>
#include <type_traits>

namespace pllm {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kTileRows = 64;                       // matrix rows of a tile
constexpr int kWaveCols = 32;                       // hidden columns (gate / up) per wave; weight rows per wave: 64
// a wave's LDS for turning the bytes of a block: 32 weight rows at a time, 16 with twelve waves
constexpr int wave_slot(int waves) { return waves == 8 ? 32 * 64 : 16 * 64; }

__device__ __forceinline__ v8h as_v8h(uint4 u) { return __builtin_bit_cast(v8h, u); }
__device__ __forceinline__ uint32_t times(uint32_t pair, v2h scale) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, pair) * scale); }
// 2 s + 1 as a pair of halves: 1024 + 2 s + 1 by integer arithmetic on the bits, minus 1024
__device__ __forceinline__ v2h odd_scale(uint32_t s) {
    const v2h k1024 = {static_cast<_Float16>(1024.0f), static_cast<_Float16>(1024.0f)};
    return __builtin_bit_cast(v2h, s * 0x00020002u + 0x64016401u) - k1024;
}
// a << s, or >> -s
template <int S> __device__ __forceinline__ uint32_t shl(uint32_t v) {
    if constexpr (S > 0) return v << S;
    else if constexpr (S < 0) return v >> -S;
    else return v;
}
template <int I, int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// A format: the lane's half of a block in registers, its scale, and codebook entry i of that half as eight halves in two steps
// (look: the LDS reads; finish: what the vector ALU adds once they are there).
struct TileIQ2XXS {
    static constexpr int kBlockBytes = IQ2XXSm::kBlockBytes;
    static constexpr int kCopies = 8;               // of every entry side by side: lane l reads copy l % 8
    static constexpr int kTableBytes = 49152;       // 256 magnitudes (32 KB), 128 sign masks (16 KB)
    struct Raw { uint4 a, b; };                     // four sub-blocks of 8 bytes (ids, signs + scale)
    struct Look { uint4 mag, sgn; };
    static __device__ void stage_tables(unsigned char* lds, int tid, int threads) {
        for (int i = tid; i < (256 + 128) * kCopies; i += threads) {
            const int e = i / kCopies;
            uint32_t w[4];
            if (e < 256) {
                const uint64_t g = PLLM_IQ2XXS_GRID[e];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v2h c = {static_cast<_Float16>(static_cast<float>((g >> (16 * j)) & 0xffu)), static_cast<_Float16>(static_cast<float>((g >> (16 * j + 8)) & 0xffu))};
                    w[j] = __builtin_bit_cast(uint32_t, c);
                }
            } else {
                const uint64_t m = PLLM_IQ2XXS_SIGN_MASKS.v[e - 256];
#pragma unroll
                for (int j = 0; j < 4; ++j) w[j] = (((m >> (16 * j)) & 1u) ? 0x8000u : 0u) | (((m >> (16 * j + 8)) & 1u) ? 0x80000000u : 0u);
            }
            reinterpret_cast<uint4*>(lds)[i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    static __device__ __forceinline__ uint32_t table_lane(int lane) { return (lane & (kCopies - 1)) * 16; }
    static __device__ __forceinline__ uint32_t piece_off(int t) { return 2 + 16 * t; }
    static __device__ __forceinline__ uint4 load_piece(const uint8_t* block, uint32_t off) { return load16_a2(block + off); }
    // the bytes of the lane's share of a turned row: half `part` (LANES = 2) or quarter `part` (LANES = 4) of the block
    template <int LANES> static __device__ __forceinline__ void pick(Raw& r, const unsigned char* row, uint32_t swz, int part) {
        if constexpr (LANES == 2) {
            r.a = *reinterpret_cast<const uint4*>(row + ((32u * part) ^ swz));
            r.b = *reinterpret_cast<const uint4*>(row + ((32u * part + 16u) ^ swz));
        } else {
            r.a = *reinterpret_cast<const uint4*>(row + ((16u * part) ^ swz));
        }
    }
    // block scales: lane group g of the wave fetched those of set g; swaps of the groups hand them round
    static __device__ __forceinline__ uint32_t load_scale(const uint8_t* block, uint32_t off) { return *reinterpret_cast<const uint16_t*>(block + off); }
    template <int SETS> static __device__ __forceinline__ void scales(uint32_t d, const Raw*, float* out) {
        const auto half = __builtin_amdgcn_permlane32_swap(d, d, false, false);
        if constexpr (SETS == 2) {
            out[0] = 0.125f * f16_bits_to_float(half[0]);
            out[1] = 0.125f * f16_bits_to_float(half[1]);
        } else {
            const auto lo = __builtin_amdgcn_permlane16_swap(half[0], half[0], false, false), hi = __builtin_amdgcn_permlane16_swap(half[1], half[1], false, false);
            out[0] = 0.125f * f16_bits_to_float(lo[0]);
            out[1] = 0.125f * f16_bits_to_float(lo[1]);
            out[2] = 0.125f * f16_bits_to_float(hi[0]);
            out[3] = 0.125f * f16_bits_to_float(hi[1]);
        }
    }
    template <int I> static __device__ __forceinline__ uint32_t ids(const Raw& r) { return I < 4 ? r.a.x : I < 8 ? r.a.z : I < 12 ? r.b.x : r.b.z; }
    template <int I> static __device__ __forceinline__ uint32_t aux(const Raw& r) { return I < 4 ? r.a.y : I < 8 ? r.a.w : I < 12 ? r.b.y : r.b.w; }
    template <int I> static __device__ __forceinline__ void look(Look& l, const Raw& r, const unsigned char* lds, uint32_t copy) {
        constexpr int j = I & 3;
        const uint32_t id = (shl<7 - 8 * j>(ids<I>(r)) & 0x7f80u) | copy, sg = (shl<7 - 7 * j>(aux<I>(r)) & 0x3f80u) | copy;
        l.mag = *reinterpret_cast<const uint4*>(lds + id);
        l.sgn = *reinterpret_cast<const uint4*>(lds + sg + 32768);
    }
    template <int I> static __device__ __forceinline__ uint4 finish(const Look& l, const Raw& r) {
        const v2h s = odd_scale(aux<I>(r) >> 28);
        return make_uint4(times(l.mag.x ^ l.sgn.x, s), times(l.mag.y ^ l.sgn.y, s), times(l.mag.z ^ l.sgn.z, s), times(l.mag.w ^ l.sgn.w, s));
    }
};

struct TileIQ1M {
    static constexpr int kBlockBytes = IQ1Mm::kBlockBytes;
    static constexpr int kTableBytes = 65536;       // 4096 entries (index byte | qh nibble << 8) of eight finished codes
    struct Raw { uint4 q; uint2 qh; uint32_t sw; float d; };      // index bytes, qh nibbles and scale words of the lane's share, block scale
    struct Look { uint4 code; };
    static __device__ void stage_tables(unsigned char* lds, int tid, int threads) {
        for (int i = tid; i < 4096; i += threads) {
            const uint64_t v = PLLM_IQ1_DELTA_CODES.v[i];
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const v2h c = {static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(v >> (16 * j)))), static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(v >> (16 * j + 8))))};
                w[j] = __builtin_bit_cast(uint32_t, c);
            }
            reinterpret_cast<uint4*>(lds)[i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    static __device__ __forceinline__ uint32_t table_lane(int) { return 0; }
    static __device__ __forceinline__ uint32_t piece_off(int t) { return t < 3 ? 16 * t : 40; }           // (the last piece ends with the block)
    static __device__ __forceinline__ uint4 load_piece(const uint8_t* block, uint32_t off) {
        const uint2* p = reinterpret_cast<const uint2*>(block + off);                                    // blocks are 8-byte aligned
        const uint2 lo = p[0], hi = p[1];
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    template <int LANES> static __device__ __forceinline__ void pick(Raw& r, const unsigned char* row, uint32_t swz, int part) {
        const uint2 sc = *reinterpret_cast<const uint2*>(row + (48u ^ swz) + 8);
        r.d = 0.125f * f16_bits_to_float(((sc.x >> 12) & 0xfu) | ((sc.x >> 24) & 0xf0u) | ((sc.y >> 4) & 0xf00u) | ((sc.y >> 16) & 0xf000u));
        if constexpr (LANES == 2) {
            r.q = *reinterpret_cast<const uint4*>(row + ((16u * part) ^ swz));
            r.qh = *reinterpret_cast<const uint2*>(row + (32u ^ swz) + 8 * part);
            r.sw = part ? sc.y : sc.x;
        } else {
            const uint2 q = *reinterpret_cast<const uint2*>(row + ((16u * (part >> 1)) ^ swz) + 8 * (part & 1));
            r.q = make_uint4(q.x, q.y, 0u, 0u);
            r.qh = make_uint2(*reinterpret_cast<const uint32_t*>(row + (32u ^ swz) + 4 * part), 0u);
            r.sw = ((part >> 1) ? sc.y : sc.x) >> (16 * (part & 1));
        }
    }
    static __device__ __forceinline__ uint32_t load_scale(const uint8_t*, uint32_t) { return 0; }
    template <int SETS> static __device__ __forceinline__ void scales(uint32_t, const Raw* r, float* out) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) out[s] = r[s].d;
    }
    template <int I> static __device__ __forceinline__ void look(Look& l, const Raw& r, const unsigned char* lds, uint32_t) {
        constexpr int j = I & 3, t = I & 7;
        const uint32_t qw = I < 4 ? r.q.x : I < 8 ? r.q.y : I < 12 ? r.q.z : r.q.w, hw = I < 8 ? r.qh.x : r.qh.y;
        l.code = *reinterpret_cast<const uint4*>(lds + ((shl<4 - 8 * j>(qw) & 0xff0u) | (shl<12 - 4 * t>(hw) & 0xf000u)));
    }
    template <int I> static __device__ __forceinline__ uint4 finish(const Look& l, const Raw& r) {
        const v2h s = odd_scale(__builtin_amdgcn_ubfe(r.sw, 16 * (I >> 3) + 3 * ((I >> 1) & 3), 3));
        return make_uint4(times(l.code.x, s), times(l.code.y, s), times(l.code.z, s), times(l.code.w, s));
    }
};

struct TileArgs {
    const _Float16* rows;                           // activation rows, kp halves each
    const float* unscale;                           // per activation row group (token or route): 1 / its power of two
    const int64_t* route_tokens;
    const float* route_weights;
    const uint8_t* w0;                              // gate (or down)
    const uint8_t* w1;                              // up (gate / up launches)
    const int4* tiles;                              // {expert, first route, routes, 0}
    const int32_t* n_tiles;
    float* out;                                     // hidden values [routes][out_pitch], or partial outputs
    float* tile_max;                                // largest magnitude per route and 16 hidden columns
    float limit;
    int bpr, n, out_pitch, col_groups;
};

__device__ __forceinline__ v16f mfma(uint4 a, uint4 b, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(as_v8h(a), as_v8h(b), c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma(uint4 a, uint4 b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(as_v8h(a), as_v8h(b), c, 0, 0, 0); }

// How a wave's 64 weight rows meet the tile's matrix rows.  16 rows: v_mfma_f32_16x16x32_f16, four sets of 16 weight rows, a quarter of
// a block per lane; 32 or 64 rows: v_mfma_f32_32x32x16_f16, two sets of 32, half a block per lane.
template <int ROWS> struct TileShape {
    static constexpr bool kNarrow = ROWS == 16;
    static constexpr int kSets = kNarrow ? 4 : 2, kCols = kNarrow ? 16 : 32, kParts = kNarrow ? 4 : 2, kSteps = 32 / kParts, kM = kNarrow ? 1 : ROWS / 32, kRegs = kNarrow ? 4 : 16;
    using Acc = std::conditional_t<kNarrow, v4f, v16f>;
};

// One tile of up to ROWS matrix rows against the wave's 64 weight rows.  !mine (WHOLE_K): the wave only moves its share of the activations.
template <typename FMT, int ROWS, int WAVES, bool WHOLE_K, int TERMS, bool GATE_UP>
__device__ __forceinline__ void tile_pass(const TileArgs& a, const int4 t, int group, unsigned char* smem, uint32_t lds0, float* factors, int tid, int wave, bool mine) {
    using S = TileShape<ROWS>;
    using Acc = typename S::Acc;
    constexpr int kChunk = ROWS * 512, kPieces = ROWS / 2, kDma = (kPieces + WAVES - 1) / WAVES;      // (direct-to-LDS instructions per block of activations)
    constexpr int kActOff = FMT::kTableBytes + WAVES * wave_slot(WAVES);
    const int lane = tid & 63, r = lane % S::kCols, part = lane / S::kCols;
    const int kp = a.bpr * 256, row_bytes = a.bpr * FMT::kBlockBytes;
    const uint8_t* base0 = a.w0 + static_cast<size_t>(t.x) * a.n * row_bytes;
    const uint8_t* base1 = GATE_UP ? a.w1 + static_cast<size_t>(t.x) * a.n * row_bytes : base0;
    const int c0 = (group * WAVES + wave) * (GATE_UP ? kWaveCols : 2 * kWaveCols), c1 = GATE_UP ? c0 : c0 + kWaveCols;
    // A block's bytes are fetched with four neighbouring lanes on one weight row (instruction k of a half: rows 16 k .. 16 k + 15),
    // then turned in the wave's own LDS slot: asked for by the lanes that decode them, every instruction would touch 32 rows' lines
    // (the fetches then cost 100 of 383 us at 256 experts and 2048 routes).
    uint32_t woff[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int k = 0; k < 2; ++k) woff[s][k] = static_cast<uint32_t>(min((s ? c1 : c0) + 16 * k + (lane >> 2), a.n - 1)) * row_bytes + FMT::piece_off(lane & 3);
    // (the weight row of set `part` that the lane's column stands for)
    const uint32_t doff = static_cast<uint32_t>(min((lane >= 32 ? c1 : c0) + (lane & 31), a.n - 1)) * row_bytes;
    unsigned char* slot = smem + FMT::kTableBytes + wave * wave_slot(WAVES);
    const uint32_t slot_in = (lane >> 2) * 64u + (((lane & 3) ^ ((lane >> 4) & 3)) << 4), slot_swz = ((r >> 2) & 3) << 4;

    uint32_t xoff[kDma];                            // instruction i of the wave moves matrix rows 2 (wave + WAVES i) and the next one
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
        const int row = min(2 * (wave + WAVES * i), ROWS - 2) + (lane >> 5), route = t.y + min(row / TERMS, t.z - 1);
        const uint32_t src = GATE_UP ? static_cast<uint32_t>(a.route_tokens[route]) * TERMS + row % TERMS : static_cast<uint32_t>(route);
        xoff[i] = src * (2u * kp) + 16u * ((lane & 31) ^ (row & 31));
    }
    const unsigned char* xb = reinterpret_cast<const unsigned char*>(a.rows);
    auto dma = [&](const unsigned char* src, int buf) {
#pragma unroll
        for (int i = 0; i < kDma; ++i)
            if (kPieces % WAVES == 0 || wave + WAVES * i < kPieces) lds_dma16_at(src, xoff[i], lds0 + kActOff + buf * kChunk + (wave + WAVES * i) * 1024);
    };
    if (tid < ROWS / TERMS) {                       // the epilogue's factors per route
        const int route = t.y + min(tid, t.z - 1);
        factors[tid] = a.unscale[GATE_UP ? a.route_tokens[route] : route];
        factors[kTileRows + tid] = GATE_UP ? a.route_weights[route] : 1.0f;
    }
    uint4 fetched[2][2];
    uint32_t fetched_d, block_d;
    typename FMT::Raw raw[S::kSets];
    auto fetch = [&]() {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            fetched[0][k] = FMT::load_piece(base0, woff[0][k]);
            fetched[1][k] = FMT::load_piece(base1, woff[1][k]);
        }
        fetched_d = FMT::load_scale(lane >= 32 ? base1 : base0, doff);
    };
    auto turn = [&]() {                             // (one wave's LDS operations take effect in order: the slot serves one half after the other)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                *reinterpret_cast<uint4*>(slot + (S::kNarrow ? 0 : 1024 * k) + slot_in) = fetched[s][k];
                if constexpr (S::kNarrow) FMT::template pick<4>(raw[2 * s + k], slot + r * 64, slot_swz, part);
            }
            if constexpr (!S::kNarrow) FMT::template pick<2>(raw[s], slot + r * 64, slot_swz, part);
        }
        block_d = fetched_d;
    };
    if (!WHOLE_K || mine) fetch();
    if constexpr (WHOLE_K) {                        // all of K at once, no barrier in the loop over its blocks
        for (int b = 0; b < a.bpr; ++b) dma(xb + 512 * b, b);
    } else {
        dma(xb, 0);
    }
    Acc acc[S::kM][S::kSets];
#pragma unroll
    for (int m = 0; m < S::kM; ++m)
#pragma unroll
        for (int s = 0; s < S::kSets; ++s) acc[m][s] = Acc{};
    const uint32_t abase = kActOff + (static_cast<uint32_t>(r) * 512u | (static_cast<uint32_t>(r ^ (S::kSteps * part)) << 4));
    const uint32_t copy = FMT::table_lane(lane);
    const Acc zero = {};
    if (!WHOLE_K || mine) turn();
    wait_vm<0>();
    __syncthreads();
    for (int b = 0; b < (!WHOLE_K || mine ? a.bpr : 0); ++b) {
        const bool more = b + 1 < a.bpr;            // (past the end: the last block again, not used)
        base0 += more ? FMT::kBlockBytes : 0;
        base1 += more ? FMT::kBlockBytes : 0;
        fetch();
        if constexpr (!WHOLE_K) {
            xb += more ? 512 : 0;
            dma(xb, (b + 1) & 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* at = smem + (WHOLE_K ? b : b & 1) * kChunk;
        Acc c[S::kM][S::kSets];
        // codebook reads run two entries ahead (one with four sets: as many reads in flight), activation reads one
        constexpr int kAhead = S::kNarrow ? 1 : 2;
        typename FMT::Look look[kAhead][S::kSets];
        constexpr int kAv = S::kM == 1 ? 2 : 1;      // (64 rows: registers for one step's activations)
        uint4 bw[S::kSets], av[kAv][S::kM];
        static_for<0, kAhead + 1>([&](auto I) {
            constexpr int i = I;
#pragma unroll
            for (int s = 0; s < S::kSets; ++s) {
                if constexpr (i == kAhead) bw[s] = FMT::template finish<0>(look[0][s], raw[s]);
                FMT::template look<i>(look[i % kAhead][s], raw[s], smem, copy);
            }
            if constexpr (i == 0) {
#pragma unroll
                for (int m = 0; m < S::kM; ++m) av[0][m] = *reinterpret_cast<const uint4*>(at + abase + m * 16384);
            }
        });
        // step i: matrix instructions of entry i, the second half of the decode of entry i + 1, LDS reads for later entries
        static_for<0, S::kSteps>([&](auto I) {
            constexpr int i = I;
            if constexpr (kAv == 2 && i + 1 < S::kSteps) {
#pragma unroll
                for (int m = 0; m < S::kM; ++m) av[(i + 1) % kAv][m] = *reinterpret_cast<const uint4*>(at + (abase ^ ((i + 1) << 4)) + m * 16384);
            }
            static_for<0, S::kM * S::kSets>([&](auto U) {
                constexpr int u = U, m = u / S::kSets, s = u % S::kSets;
                c[m][s] = mfma(av[i % kAv][m], bw[s], i == 0 ? zero : c[m][s]);
                if constexpr (kAv == 1 && s == S::kSets - 1 && i + 1 < S::kSteps) av[0][m] = *reinterpret_cast<const uint4*>(at + (abase ^ ((i + 1) << 4)) + m * 16384);
                if constexpr (m == S::kM - 1 && i + 1 < S::kSteps) {
                    bw[s] = FMT::template finish<i + 1>(look[(i + 1) % kAhead][s], raw[s]);
                    if constexpr (i + 1 + kAhead < S::kSteps) FMT::template look<i + 1 + kAhead>(look[(i + 1) % kAhead][s], raw[s], smem, copy);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        float d[S::kSets];
        FMT::template scales<S::kSets>(block_d, raw, d);
#pragma unroll
        for (int s = 0; s < S::kSets; ++s)
#pragma unroll
            for (int m = 0; m < S::kM; ++m)
#pragma unroll
                for (int v = 0; v < S::kRegs; ++v) acc[m][s][v] += d[s] * c[m][s][v];
        turn();
        if constexpr (!WHOLE_K) {
            wait_vm<0>();
            __syncthreads();                        // the next block's rows are there, this one's have been read
        }
    }
    if constexpr (WHOLE_K) {
        __syncthreads();                            // (the next tile's rows go where this one's were read)
        if (!mine) return;
    }
    // lane: column r of each set; matrix rows 4 part + v of 16, or 8 (v / 4) + 4 part + v % 4 of each 32
#pragma unroll
    for (int m = 0; m < S::kM; ++m)
#pragma unroll
        for (int v = 0; v < S::kRegs; v += TERMS) {
            const int row = (S::kNarrow ? 4 * part + v : 32 * m + 8 * (v >> 2) + 4 * part + (v & 3)) / TERMS;
            const float f = factors[row];
            float* out = a.out + static_cast<size_t>(t.y + row) * a.out_pitch;
            auto total = [&](int s) { return (acc[m][s][v] + (TERMS == 2 ? acc[m][s][(v + 1) % S::kRegs] : 0.0f)) * f; };
#pragma unroll
            for (int s = 0; s < S::kSets; s += 1) {
                const int in_half = (s % (S::kSets / 2)) * S::kCols + r;
                if constexpr (GATE_UP) {
                    if (s >= S::kSets / 2) break;
                    const int col = c0 + in_half;
                    float g = total(s), u = total(s + S::kSets / 2);
                    if (a.limit > 0.0f) {
                        u = fminf(fmaxf(u, -a.limit), a.limit);
                        g = fminf(g, a.limit);
                    }
                    const float hv = col < a.n ? g / (1.0f + expf(-g)) * u * factors[kTileRows + row] : 0.0f;   // (padding columns: zeros)
                    const float am = group_max<16>(fabsf(hv));
                    if (row < t.z && col < a.out_pitch) {
                        out[col] = hv;
                        if ((r & 15) == 0) a.tile_max[static_cast<size_t>(t.y + row) * (a.out_pitch / 16) + (col >> 4)] = am;
                    }
                } else {
                    const int col = (s >= S::kSets / 2 ? c1 : c0) + in_half;
                    if (row < t.z && col < a.n) out[col] = total(s);
                }
            }
        }
}

// WAVES = 8: tiles of up to 64 matrix rows (two waves per SIMD); 12: of up to 16 (three)
template <typename FMT, int WAVES, bool WHOLE_K, int TERMS, bool GATE_UP>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void moe_tile_kernel(TileArgs a) {
    extern __shared__ __align__(1024) unsigned char smem[];
    __shared__ float factors[2][2 * kTileRows];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte_ptr)smem));
    const int units = a.n_tiles[0] * a.col_groups;
    // The units of a last round that would keep a few compute units busy for a whole round are dealt out by waves: `parts` workgroups
    // take WAVES / parts waves' columns each (a unit's waves share the LDS and the SIMDs of one compute unit otherwise).  2048 routes over 256
    // experts are 1024 units and a few for experts of more than 16 routes, whose fifth round took as long as the four before it each:
    // 256 tokens, gate / up and down with everything around them, 444 -> 428 us.  (Those experts as tiles of 32 rows among the twelve waves
    // instead: 511 us, the registers overflow.)
    const int whole_units = WHOLE_K ? units - units % static_cast<int>(gridDim.x) : units, left = units - whole_units;
    int parts = 1;
    if constexpr (WHOLE_K) {
        for (int p = 2; p <= WAVES; ++p)
            if (WAVES % p == 0 && left * p <= static_cast<int>(gridDim.x)) parts = p;
    }
    if (static_cast<int>(blockIdx.x) >= whole_units + left * parts) return;
    FMT::stage_tables(smem, tid, blockDim.x);       // (visible behind the first unit's barrier)
    int parity = 0;
    for (int at = blockIdx.x; at < whole_units + left * parts; at += gridDim.x, parity ^= 1) {
        const bool split = at >= whole_units;
        const int unit = split ? whole_units + (at - whole_units) / parts : at, part = split ? (at - whole_units) % parts : 0;
        const bool mine = !split || wave / (WAVES / parts) == part;
        const int4 t = a.tiles[unit / a.col_groups];
        if constexpr (WAVES == 8) {
            if (t.z * TERMS > 32) {
                tile_pass<FMT, 64, WAVES, false, TERMS, GATE_UP>(a, t, unit % a.col_groups, smem, lds0, factors[parity], tid, wave, mine);
                continue;
            }
        }
        tile_pass<FMT, WAVES == 8 ? 32 : 16, WAVES, WHOLE_K, TERMS, GATE_UP>(a, t, unit % a.col_groups, smem, lds0, factors[parity], tid, wave, mine);
    }
}

// the power of two that brings a row whose largest magnitude is am into [1024, 2048) (1 for rows of zeros or with non-finite values)
__device__ __forceinline__ float rows_scale(float am) { return ldexpf(1.0f, -half_row_exponent<11>(am)); }

// Activation rows as half-precision images: img[token][term][kpad] = x * s (zero beyond dim), s the power of two of rows_scale,
// unscale[token] = 1 / s.  TERMS = 2 adds the rounding residual as a second row.
// pieces of four values a thread keeps: rows of up to four times as many values as all threads hold are read once
constexpr int image_held(int threads) { return threads == 1024 ? 8 : 4; }
template <int TERMS, int THREADS>
__global__ __launch_bounds__(THREADS) void rows_image_kernel(const void* __restrict__ x, int x_dtype, int dim, int kpad, _Float16* __restrict__ img,
                                                         float* __restrict__ unscale) {
    constexpr int kImageHeld = image_held(THREADS);
    __shared__ float part[THREADS / 64];
    const int token = blockIdx.x, tid = threadIdx.x;
    const size_t base = static_cast<size_t>(token) * dim;
    const bool held = kpad <= 4 * kImageHeld * THREADS && dim % 4 == 0 &&
                      ((reinterpret_cast<uintptr_t>(x) + base * (x_dtype == PLLM_F32 ? 4 : 2)) & 15u) == 0;
    float v[kImageHeld][4];
    float am = 0.0f;
    if (held) {                                // all of the thread's pieces requested together (beyond the row: its first piece again, dropped)
        int e0[kImageHeld];
#pragma unroll
        for (int j = 0; j < kImageHeld; ++j) e0[j] = 4 * (tid + THREADS * j) < dim ? 4 * (tid + THREADS * j) : 0;
        load_rows4_batch(v, x, x_dtype, base, e0);
#pragma unroll
        for (int j = 0; j < kImageHeld; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (4 * (tid + THREADS * j) >= dim) v[j][i] = 0.0f;
                am = fmaxf(am, fabsf(v[j][i]));
            }
    } else {
        for (int k = tid; k < dim; k += THREADS) am = fmaxf(am, fabsf(load_any(x, x_dtype, base + k)));
    }
    am = group_max<64>(am);
    if ((tid & 63) == 0) part[tid >> 6] = am;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) am = fmaxf(am, part[w]);
    const float s = rows_scale(am);
    _Float16* row = img + static_cast<size_t>(token) * TERMS * kpad;
    if (held) {
#pragma unroll
        for (int j = 0; j < kImageHeld; ++j) {
            const int k0 = 4 * (tid + THREADS * j);
            if (k0 < kpad) {
                union { _Float16 h[4]; uint2 u; } hi, lo;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float w = v[j][i] * s;
                    hi.h[i] = static_cast<_Float16>(w);
                    lo.h[i] = static_cast<_Float16>(w - static_cast<float>(hi.h[i]));
                }
                *reinterpret_cast<uint2*>(row + k0) = hi.u;
                if constexpr (TERMS == 2) *reinterpret_cast<uint2*>(row + kpad + k0) = lo.u;
            }
        }
    } else {
        for (int k = tid; k < kpad; k += THREADS) {
            const float w = k < dim ? load_any(x, x_dtype, base + k) * s : 0.0f;
            const _Float16 h = static_cast<_Float16>(w);
            row[k] = h;
            if constexpr (TERMS == 2) row[kpad + k] = static_cast<_Float16>(w - static_cast<float>(h));
        }
    }
    if (tid == 0) unscale[token] = 1.0f / s;
}

// hidden rows of the down projection: h16[route][k] = h[route][k] * s, s the power of two of rows_scale for the route's
// largest magnitude; unscale[route] = 1 / s.  One workgroup per route.
__global__ __launch_bounds__(256) void rows_hidden_half_kernel(const float* __restrict__ h, const float* __restrict__ tile_max, int h_kpad,
                                                               _Float16* __restrict__ h16, float* __restrict__ unscale) {
    __shared__ float part[4];
    const int route = blockIdx.x, tid = threadIdx.x;
    float am = 0.0f;
    for (int t = tid; t < h_kpad / 16; t += 256) am = fmaxf(am, tile_max[static_cast<size_t>(route) * (h_kpad / 16) + t]);
    am = group_max<64>(am);
    if ((tid & 63) == 0) part[tid >> 6] = am;
    __syncthreads();
    const float s = rows_scale(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
    const float4* src = reinterpret_cast<const float4*>(h + static_cast<size_t>(route) * h_kpad);
    uint2* dst = reinterpret_cast<uint2*>(h16 + static_cast<size_t>(route) * h_kpad);
    for (int k = tid; k < h_kpad / 4; k += 256) {
        const float4 v = src[k];
        union { _Float16 h[4]; uint2 u; } c;
        c.h[0] = static_cast<_Float16>(v.x * s); c.h[1] = static_cast<_Float16>(v.y * s);
        c.h[2] = static_cast<_Float16>(v.z * s); c.h[3] = static_cast<_Float16>(v.w * s);
        dst[k] = c.u;
    }
    if (tid == 0) unscale[route] = 1.0f / s;
}

// the tiles of all experts: every expert's routes in runs of at most `per_tile`.  The products take a tile's rows as they stand in it, so whatever the
// table says, the list names no row outside [0, routes) and has no more than `most` tiles.
__global__ __launch_bounds__(256) void moe_tile_list_kernel(const int32_t* __restrict__ seg, int n_experts, int per_tile, int routes, int most,
                                                            int4* __restrict__ tiles, int32_t* __restrict__ n_tiles) {
    __shared__ int wave_sum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int done = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 256) {
        const int e = e0 + tid;
        const int r0 = e < n_experts ? min(max(seg[e], 0), routes) : 0, r1 = e < n_experts ? min(max(seg[e + 1], 0), routes) : 0;
        const int mine = (max(r1 - r0, 0) + per_tile - 1) / per_tile;
        int sum = mine;                             // inclusive sum over the wave
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(sum, o);
            if (lane >= o) sum += v;
        }
        if (lane == 63) wave_sum[wave] = sum;
        __syncthreads();
        int at = done + sum - mine;
        for (int w = 0; w < wave; ++w) at += wave_sum[w];
        for (int i = 0; i < mine && at + i < most; ++i) tiles[at + i] = make_int4(e, r0 + i * per_tile, min(per_tile, r1 - r0 - i * per_tile), 0);
        done += wave_sum[0] + wave_sum[1] + wave_sum[2] + wave_sum[3];
        __syncthreads();
    }
    if (tid == 0) n_tiles[0] = min(done, most);
}

template <typename FMT, int WAVES, bool WHOLE_K, int TERMS, bool GATE_UP>
int launch_tiles_waves(TileArgs a, int most_tiles, hipStream_t stream) {
    static SmemGrant granted;
    const size_t smem = FMT::kTableBytes + WAVES * wave_slot(WAVES) + (WHOLE_K ? a.bpr : 2) * (WAVES == 8 ? kTileRows : 16) * 512;
    if (smem + 2 * 2 * kTileRows * sizeof(float) > 160 * 1024) return PLLM_ERR_UNSUPPORTED;
    auto kern = moe_tile_kernel<FMT, WAVES, WHOLE_K, TERMS, GATE_UP>;
    if (!grant_dynamic_smem(reinterpret_cast<const void*>(kern), smem, granted)) return PLLM_ERR_UNSUPPORTED;
    const int group_cols = WAVES * (GATE_UP ? kWaveCols : 2 * kWaveCols);
    a.col_groups = ((GATE_UP ? a.out_pitch : a.n) + group_cols - 1) / group_cols;
    // (WHOLE_K: one workgroup per compute unit whatever the number of units, since the kernel deals out units by waves.  Gate / up and down with
    // everything around them, us, one workgroup per unit / per compute unit: 8 experts of 3072 -> 1536 with 16 routes 123 / 85, 16 with 96 126 /
    // 89, 32 with 64 126 / 104, 64 of 2048 -> 768 with 128 103 / 93; 64 of 2048 -> 1280 and larger sets alike)
    const long long units = static_cast<long long>(most_tiles) * a.col_groups;
    const int grid = WHOLE_K ? compute_units() : static_cast<int>(std::min<long long>(units, compute_units()));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WAVES), smem, stream, a);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}
template <typename FMT, int TERMS, bool GATE_UP>
int launch_tiles(const TileArgs& a, int most_tiles, bool small, hipStream_t stream) {
    if (!small) return launch_tiles_waves<FMT, 8, false, TERMS, GATE_UP>(a, most_tiles, stream);
    const int st = launch_tiles_waves<FMT, 12, true, TERMS, GATE_UP>(a, most_tiles, stream);
    return st != PLLM_ERR_UNSUPPORTED ? st : launch_tiles_waves<FMT, 12, false, TERMS, GATE_UP>(a, most_tiles, stream);
}

}  // namespace

// activation rows as half-precision matrix rows: img[row][term][kpad] (float32 rows: two terms) and 1 / scale per row
int half_rows_stage(const void* x, int x_dtype, int rows, int k, int kpad, void* img, float* unscale, hipStream_t stream) {
    // (1024 threads above 4096 values: 203 rows of 5120 bf16 values 12.2 us with 256, which then read every value twice)
    const bool two = x_dtype == PLLM_F32, wide = kpad > 4 * image_held(256) * 256;
    const auto kern = wide ? (two ? rows_image_kernel<2, 1024> : rows_image_kernel<1, 1024>) : (two ? rows_image_kernel<2, 256> : rows_image_kernel<1, 256>);
    hipLaunchKernelGGL(kern, dim3(rows), dim3(wide ? 1024 : 256), 0, stream, x, x_dtype, k, kpad, static_cast<_Float16*>(img), unscale);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

bool moe_tiles_supports(int w13_type, int w2_type, int dim, int inter, int tokens, int routes, const uint8_t* w1, const uint8_t* w3, const uint8_t* w2) {
    if (w13_type != PLLM_TYPE_IQ2_XXS || w2_type != PLLM_TYPE_IQ1_M || dim % 16 != 0 || inter % 16 != 0) return false;
    // (IQ2_XXS blocks are read at 2-byte alignment, IQ1_M blocks at 8)
    if (((reinterpret_cast<uintptr_t>(w1) | reinterpret_cast<uintptr_t>(w3)) & 1u) || (reinterpret_cast<uintptr_t>(w2) & 7u)) return false;
    // activation rows are addressed with 32-bit byte offsets, and so are the rows of one expert's matrices
    const unsigned long long kx = (static_cast<unsigned long long>(dim) + 255) / 256 * 256, kh = (static_cast<unsigned long long>(inter) + 255) / 256 * 256;
    const unsigned long long x_bytes = 4ull * tokens * kx, h_bytes = 2ull * routes * kh, w_bytes = std::max(kx * inter, kh * dim);
    return x_bytes < (1ull << 32) && h_bytes < (1ull << 32) && w_bytes < (1ull << 32);
}

size_t moe_rows_x_bytes(int64_t tokens, int64_t dim) {
    const size_t kpad = static_cast<size_t>((dim + 255) / 256) * 256;
    return align256(static_cast<size_t>(tokens) * 2 * kpad * sizeof(_Float16)) + align256(static_cast<size_t>(tokens) * sizeof(float));
}

// hidden rows of the routes: float32 values [routes][h_kpad], largest magnitudes per 16-row tile, half-precision rows, 1 / scale
struct RowsHidden { float* values; float* tile_max; _Float16* half_rows; float* unscale; size_t bytes; };

static RowsHidden rows_hidden(void* ws, int64_t routes, int64_t inter) {
    const size_t kpad = static_cast<size_t>((inter + 255) / 256) * 256, r = static_cast<size_t>(routes);
    unsigned char* p = static_cast<unsigned char*>(ws);
    RowsHidden h;
    h.values = reinterpret_cast<float*>(p);        p += align256(r * kpad * sizeof(float));
    h.tile_max = reinterpret_cast<float*>(p);      p += align256(r * (kpad / 16) * sizeof(float));
    h.half_rows = reinterpret_cast<_Float16*>(p);  p += align256(r * kpad * sizeof(_Float16));
    h.unscale = reinterpret_cast<float*>(p);       p += align256(r * sizeof(float));
    h.bytes = static_cast<size_t>(p - static_cast<unsigned char*>(ws));
    return h;
}

size_t moe_rows_h_bytes(int64_t routes, int64_t inter) { return rows_hidden(nullptr, routes, inter).bytes; }

size_t moe_tiles_list_bytes(int64_t routes) { return align256(static_cast<size_t>(routes) * sizeof(int4)) + 256; }

namespace {
// matrix rows per expert on average up to which tiles of 16 rows and twelve waves are taken (us for all experts, 16- / 64-row tiles:
// 8 rows on average 442 / 533, 16 rows ~640 / 575, as half of the experts then need two of the small tiles)
constexpr int kSmallTileRows = 12;
bool small_tiles(int terms, int routes, int n_experts) { return static_cast<long long>(routes) * terms <= static_cast<long long>(kSmallTileRows) * n_experts; }
TileArgs tile_args(void* list_ws, int routes) {
    TileArgs a{};
    a.tiles = static_cast<int4*>(list_ws);
    a.n_tiles = moe_tile_list_count(list_ws, routes);
    return a;
}
}  // namespace

int moe_tile_list_most(int routes, int n_experts, int per_tile) { return std::min(routes, std::min(routes, n_experts) + routes / per_tile); }
// (list_ws: the tiles, then their count)
const int32_t* moe_tile_list_count(const void* list_ws, int routes) {
    return reinterpret_cast<const int32_t*>(static_cast<const unsigned char*>(list_ws) + align256(static_cast<size_t>(routes) * sizeof(int4)));
}
int moe_tile_list(const int32_t* seg, int n_experts, int per_tile, int routes, void* list_ws, hipStream_t stream) {
    hipLaunchKernelGGL(moe_tile_list_kernel, dim3(1), dim3(256), 0, stream, seg, n_experts, per_tile, routes,
                       moe_tile_list_most(routes, n_experts, per_tile), static_cast<int4*>(list_ws),
                       const_cast<int32_t*>(moe_tile_list_count(list_ws, routes)));
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

// hidden values of all routes, SiLU(gate) * up * route weight, as half-precision rows in h_rows_ws
int moe_tiles_w13(const void* x, int x_dtype, int tokens, int dim, void* x_rows_ws, const int64_t* route_tokens, const int32_t* seg,
                  const float* route_weights, const uint8_t* w1, const uint8_t* w3, int inter, float limit, void* h_rows_ws, void* list_ws,
                  int n_experts, int routes, hipStream_t stream) {
    const int bpr = (dim + 255) / 256, kpad = bpr * 256, h_kpad = (inter + 255) / 256 * 256;
    _Float16* x_rows = static_cast<_Float16*>(x_rows_ws);
    const RowsHidden hid = rows_hidden(h_rows_ws, routes, inter);
    float* unscale = reinterpret_cast<float*>(static_cast<unsigned char*>(x_rows_ws) + align256(static_cast<size_t>(tokens) * 2 * kpad * sizeof(_Float16)));
    const int terms = x_dtype == PLLM_F32 ? 2 : 1;
    int st = half_rows_stage(x, x_dtype, tokens, dim, kpad, x_rows, unscale, stream);
    if (st != PLLM_OK) return st;
    TileArgs a = tile_args(list_ws, routes);
    a.rows = x_rows;
    a.unscale = unscale;
    a.route_tokens = route_tokens;
    a.route_weights = route_weights;
    a.w0 = w1;
    a.w1 = w3;
    a.out = hid.values;
    a.tile_max = hid.tile_max;
    a.limit = limit;
    a.bpr = bpr;
    a.n = inter;
    a.out_pitch = h_kpad;
    const bool small = small_tiles(terms, routes, n_experts);
    const int per_tile = (small ? 16 : kTileRows) / terms, tiles = moe_tile_list_most(routes, n_experts, per_tile);
    st = moe_tile_list(seg, n_experts, per_tile, routes, list_ws, stream);
    if (st != PLLM_OK) return st;
    st = terms == 2 ? launch_tiles<TileIQ2XXS, 2, true>(a, tiles, small, stream) : launch_tiles<TileIQ2XXS, 1, true>(a, tiles, small, stream);
    if (st != PLLM_OK) return st;
    hipLaunchKernelGGL(rows_hidden_half_kernel, dim3(routes), dim3(256), 0, stream, hid.values, hid.tile_max, h_kpad, hid.half_rows, hid.unscale);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

// partial [routes][dim] = W2_e times the half-precision hidden rows of every route
int moe_tiles_w2(void* h_rows_ws, void* list_ws, int x_dtype, int inter, const int32_t* seg, const uint8_t* w2, float* partial, int dim, int n_experts,
                 int routes, hipStream_t stream) {
    const RowsHidden hid = rows_hidden(h_rows_ws, routes, inter);
    TileArgs a = tile_args(list_ws, routes);
    a.rows = hid.half_rows;
    a.unscale = hid.unscale;
    a.w0 = w2;
    a.out = partial;
    a.bpr = (inter + 255) / 256;
    a.n = dim;
    a.out_pitch = dim;
    const bool small = small_tiles(1, routes, n_experts);
    const int per_tile = small ? 16 : kTileRows;
    if (x_dtype == PLLM_F32) {                       // (the gate / up launch had half as many routes per tile)
        const int st = moe_tile_list(seg, n_experts, per_tile, routes, list_ws, stream);
        if (st != PLLM_OK) return st;
    }
    return launch_tiles<TileIQ1M, 1, false>(a, moe_tile_list_most(routes, n_experts, per_tile), small, stream);
}

}  // namespace pllm
