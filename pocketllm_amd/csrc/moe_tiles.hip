// Routed experts of several tokens, IQ2_XXS gate / up and IQ1_M down: tiles of up to 64 routes against weights decoded in registers.
//
// The integer weights of both formats, code times group scale, are exact in half precision, and so are bf16 / fp16 activations
// scaled by a power of two per row (fp16 rows of whole blocks go in as the caller holds them, float32 rows as two half-precision terms = two matrix rows).  A workgroup takes a tile
// of one expert's routes, and every wave owns 64 weight rows (gate and up of the same 32 hidden columns, or 64 rows of the down
// projection) over all of K.  A weight's codes go from memory to the lane that needs them as a matrix operand and are decoded there
// once per tile: lane = one codebook entry (eight weights) of a weight row per matrix instruction, v_mfma_f32_32x32x16_f16 for
// tiles of 32 and 64 matrix rows, v_mfma_f32_16x16x32_f16 for tiles of 16.  The lanes of a row split its block into halves
// (quarters) and step through them side by side; the activation operand follows that order.  Activation rows come to LDS by
// direct-to-LDS loads, in an order in which rows read at one piece of 16 bytes meet no bank twice.  The matrix cores sum over a block,
// whose scale goes on as the sums join the totals.
//
// Two forms, of eight waves each: tiles of 16 rows up to 13 matrix rows per expert on average, tiles of 64 (or 32) above.  256 experts of
// 3072 -> 1536 -> 3072, us for gate / up + down: 2048 routes 272 + 130 in the first form, 331 + 143 in the second; 3072 routes 292 + 142
// and 338 + 147; 3584 routes 328 + 158 and 341 + 149; 8192 routes 399 + 183 in the second.
//
// A wave issues an instruction every five cycles at most, two waves a SIMD's every four or five, so instructions are what counts, then what a wave
// waits for.  Against the kernel before, with a workgroup's units apart from one another, sign masks and group scales of IQ2_XXS applied by
// two operations per pair and outputs stored behind a branch each (287 + 133 at 2048 routes, 485 + 195 at 8192): the next unit's weights, rows and first
// codebook reads are on their way during a unit's last blocks and its epilogue, whose stores need no branch and no reloaded address
// (8 - 11 us per unit before); signs times scales come from a table (454 vector instructions per block and wave before, 302 now); the L1 sees words
// (309 accesses per wave and block before, 160 now).  At 2048 routes the fetch alone (66 bytes per row and block from rows far apart: requests of
// 64 bytes, 3 TB/s) takes 200 us and the rest alone 230; LDS busy 71 %, vector ALU 42 %, matrix cores 14 %.
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
constexpr int kWaves = 8;
// a wave's LDS for turning the bytes of a block: 32 weight rows at a time, 16 for small tiles
constexpr int wave_slot(bool small) { return small ? 16 * 64 : 32 * 64; }

// 16 bytes at an LDS address (the kernel's shared memory is all dynamic and starts at 0)
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) v4u* lds_v4u_ptr;
__device__ __forceinline__ uint4 lds_read16(uint32_t at) {
    const v4u v = *reinterpret_cast<lds_v4u_ptr>(at);
    return make_uint4(v.x, v.y, v.z, v.w);
}
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
    // Two tables, both of eight halves: the signs of an entry times its group scale 2 s + 1 (16 scales of 128 sign patterns, 32 KB), so that the decode is
    // one multiplication per pair; and the 256 magnitudes (64 KB) in sixteen copies side by side, lane l reads copy l % 16: a 16-byte read serves
    // sixteen lanes at a time from the 64 banks, so no two of them meet a bank twice (cycles per read and compute unit at random entries: 3.8; eight
    // copies 7.0, one 9.9 - 10.5).
    static constexpr int kCopies = 16;
    static constexpr int kSignBytes = 16 * 128 * 16;
    static constexpr int kTableBytes = kSignBytes + 256 * 16 * kCopies;
    struct Raw { uint4 a, b; };                     // four sub-blocks of 8 bytes (ids, signs + scale)
    struct Look { uint4 mag, sgn; };
    static __device__ void stage_tables(unsigned char* lds, int tid) {
        if (tid < 256) {                            // a thread, an entry (copies one lane apart: the writes of 16 lanes meet no bank twice)
            const uint64_t g = PLLM_IQ2XXS_GRID[tid];
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const v2h c = {static_cast<_Float16>(static_cast<float>((g >> (16 * j)) & 0xffu)), static_cast<_Float16>(static_cast<float>((g >> (16 * j + 8)) & 0xffu))};
                w[j] = __builtin_bit_cast(uint32_t, c);
            }
#pragma unroll
            for (int c = 0; c < kCopies; ++c)
                reinterpret_cast<uint4*>(lds + kSignBytes)[tid * kCopies + ((c + tid) & (kCopies - 1))] = make_uint4(w[0], w[1], w[2], w[3]);
        } else if (tid < 256 + 128) {
            const uint64_t m = PLLM_IQ2XXS_SIGN_MASKS.v[tid - 256];
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = (((m >> (16 * j)) & 1u) ? 0x8000u : 0u) | (((m >> (16 * j + 8)) & 1u) ? 0x80000000u : 0u);
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const uint32_t x = __builtin_bit_cast(uint32_t, odd_scale(s));
                reinterpret_cast<uint4*>(lds)[s * 128 + tid - 256] = make_uint4(w[0] ^ x, w[1] ^ x, w[2] ^ x, w[3] ^ x);
            }
        }
    }
    static __device__ __forceinline__ uint32_t table_lane(int lane) { return (lane & (kCopies - 1)) * 16; }
    // Four neighbouring lanes fetch a block, 16 of its 64 bytes of codes each; `words`: it starts on a whole word and so do its 16-byte pieces, the
    // block scale among them; the lanes then take the last two bytes, and otherwise the block scale, by a load of their own.  (Loads of 16
    // bytes that start between two words take an access per lane and not per four lanes: 309 accesses of the L1 per wave and block against 160.)
    struct Piece { uint4 v; uint32_t x; };
    static constexpr int kLoads = 2;                // vector loads of load_piece
    static __device__ __forceinline__ void load_piece(Piece& p, const uint8_t* block, uint32_t row_off, int t, bool words) {
        p.v = load16_a2(block + (words ? 0 : 2) + (row_off + 16 * t));
        p.x = *reinterpret_cast<const uint16_t*>(block + (words ? 64 : 0) + row_off);
    }
    static __device__ __forceinline__ uint4 codes(const Piece& p, int t, bool words) {
        const uint32_t after = __builtin_amdgcn_mov_dpp(p.v.x, 0xf9, 0xf, 0xf, true), shift = words ? 16 : 0;      // (the next lane's first word)
        return make_uint4(__builtin_amdgcn_alignbit(p.v.y, p.v.x, shift), __builtin_amdgcn_alignbit(p.v.z, p.v.y, shift), __builtin_amdgcn_alignbit(p.v.w, p.v.z, shift),
                          __builtin_amdgcn_alignbit(t == 3 ? p.x : after, p.v.w, shift));
    }
    static __device__ __forceinline__ float block_scale(const Raw&) { return 0.0f; }
    static constexpr bool kScaleApart = true;       // the block scale is not among the codes: half a word in the first of the four lanes
    static __device__ __forceinline__ uint32_t scale(const Piece& p, bool words) {
        const uint32_t mask = words ? 0xffffffffu : 0u;
        return (p.v.x & mask) | (p.x & ~mask);
    }
    // the bytes of the lane's share of a turned row: half `part` (LANES = 2) or quarter `part` (LANES = 4) of the block
    template <int LANES> static __device__ __forceinline__ void pick(Raw& r, const unsigned char* row, uint32_t swz, int part) {
        if constexpr (LANES == 2) {
            r.a = *reinterpret_cast<const uint4*>(row + ((32u * part) ^ swz));
            r.b = *reinterpret_cast<const uint4*>(row + ((32u * part + 16u) ^ swz));
        } else {
            r.a = *reinterpret_cast<const uint4*>(row + ((16u * part) ^ swz));
        }
    }
    template <int I> static __device__ __forceinline__ uint32_t ids(const Raw& r) { return I < 4 ? r.a.x : I < 8 ? r.a.z : I < 12 ? r.b.x : r.b.z; }
    template <int I> static __device__ __forceinline__ uint32_t aux(const Raw& r) { return I < 4 ? r.a.y : I < 8 ? r.a.w : I < 12 ? r.b.y : r.b.w; }
    template <int I> static __device__ __forceinline__ void look(Look& l, const Raw& r, uint32_t copy) {
        constexpr int j = I & 3;
        // (magnitudes are 256 bytes apart: id j and the lane's copy are bytes 1 and 0 of the address)
        const uint32_t id = __builtin_amdgcn_perm(ids<I>(r), copy, 0x0c0c0400u + 0x100u * j);
        const uint32_t sg = (shl<4 - 7 * j>(aux<I>(r)) & 0x7f0u) | ((aux<I>(r) >> 17) & 0x7800u);
        l.mag = lds_read16(id + kSignBytes);
        l.sgn = lds_read16(sg);
    }
    static __device__ __forceinline__ uint4 finish(const Look& l) {
        const auto product = [](uint32_t x, uint32_t y) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, x) * __builtin_bit_cast(v2h, y)); };
        return make_uint4(product(l.mag.x, l.sgn.x), product(l.mag.y, l.sgn.y), product(l.mag.z, l.sgn.z), product(l.mag.w, l.sgn.w));
    }
};

struct TileIQ1M {
    static constexpr int kBlockBytes = IQ1Mm::kBlockBytes;
    static constexpr int kTableBytes = 65536;       // 4096 entries (index byte | qh nibble << 8) of eight finished codes
    struct Raw { uint4 q; uint2 qh; uint32_t sw; float d; };      // index bytes, qh nibbles and scale words of the lane's share, block scale
    struct Look { uint4 code; v2h scale; };
    static __device__ void stage_tables(unsigned char* lds, int tid) {
        // (a thread's entries requested together: one after the other they waited for memory eight times, down projection of 8 experts with 6 routes 16.4 us, now 13.9)
        constexpr int kThreads = 64 * kWaves, kEach = 4096 / kThreads;
        uint64_t v[kEach];
#pragma unroll
        for (int i = 0; i < kEach; ++i) v[i] = PLLM_IQ1_DELTA_CODES.v[tid + kThreads * i];
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const v2h c = {static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(v[i] >> (16 * j)))), static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(v[i] >> (16 * j + 8))))};
                w[j] = __builtin_bit_cast(uint32_t, c);
            }
            reinterpret_cast<uint4*>(lds)[tid + kThreads * i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    static __device__ __forceinline__ uint32_t table_lane(int) { return 0; }
    struct Piece { uint4 v; };
    static constexpr int kLoads = 1;
    static __device__ __forceinline__ void load_piece(Piece& p, const uint8_t* block, uint32_t row_off, int t, bool) {
        const uint2* from = reinterpret_cast<const uint2*>(block + (row_off + (t < 3 ? 16 * t : 40)));        // (the last piece ends with the block; 8-byte aligned)
        const uint2 lo = from[0], hi = from[1];
        p.v = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    static __device__ __forceinline__ uint4 codes(const Piece& p, int, bool) { return p.v; }
    static constexpr bool kScaleApart = false;
    static __device__ __forceinline__ float block_scale(const Raw& r) { return r.d; }
    static __device__ __forceinline__ uint32_t scale(const Piece&, bool) { return 0; }
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
    template <int I> static __device__ __forceinline__ void look(Look& l, const Raw& r, uint32_t) {
        constexpr int j = I & 3, t = I & 7;
        const uint32_t qw = I < 4 ? r.q.x : I < 8 ? r.q.y : I < 12 ? r.q.z : r.q.w, hw = I < 8 ? r.qh.x : r.qh.y;
        l.code = lds_read16((shl<4 - 8 * j>(qw) & 0xff0u) | (shl<12 - 4 * t>(hw) & 0xf000u));
        if constexpr ((I & 1) == 0) l.scale = odd_scale(__builtin_amdgcn_ubfe(r.sw, 16 * (I >> 3) + 3 * ((I >> 1) & 3), 3));      // (16 weights have one)
    }
    static __device__ __forceinline__ uint4 finish(const Look& l) {
        return make_uint4(times(l.code.x, l.scale), times(l.code.y, l.scale), times(l.code.z, l.scale), times(l.code.w, l.scale));
    }
};

struct TileArgs {
    const _Float16* rows;                           // activation rows, kp halves each
    const float* unscale;                           // per activation row group (token or route): 1 / its power of two; null: rows as the caller holds them
    const float* route_weights;
    const uint8_t* w0;                              // gate (or down)
    const uint8_t* w1;                              // up (gate / up launches)
    float* out;                                     // hidden values [routes][out_pitch], or partial outputs
    float limit;
    int bpr, n, out_pitch, wave_cols;               // wave_cols: columns in waves
};

__device__ __forceinline__ v16f mfma(uint4 a, uint4 b, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(as_v8h(a), as_v8h(b), c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma(uint4 a, uint4 b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(as_v8h(a), as_v8h(b), c, 0, 0, 0); }

// How a wave's 64 weight rows meet the tile's matrix rows.  Small tiles (16 rows): v_mfma_f32_16x16x32_f16, four sets of 16 weight rows, a quarter
// of a block per lane.  Others (up to 64 rows): v_mfma_f32_32x32x16_f16, two sets of 32, half a block per lane.
template <bool SMALL> struct TileShape {
    static constexpr int kRows = SMALL ? 16 : kTileRows;
    static constexpr int kSets = SMALL ? 4 : 2, kCols = SMALL ? 16 : 32, kParts = SMALL ? 4 : 2, kSteps = 32 / kParts, kRegs = SMALL ? 4 : 16;
    using Acc = std::conditional_t<SMALL, v4f, v16f>;
};
// Activations pass through a ring of three chunks of 16 KB: two blocks of 16 rows, or half a block of up to 64.
constexpr int kChunk = 16384, kRing = 3;
// until at most N of the wave's memory operations are outstanding, then the other waves (no LDS access moves past either)
template <int N> __device__ __forceinline__ void wait_and_meet() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory"); }
__device__ __forceinline__ int ring_after(int at) { return at == kRing - 1 ? 0 : at + 1; }

// A workgroup goes through its units (a tile of routes and as many weight rows as its waves own) without a break: while it is at the last blocks
// of one, the weights, the activations and the first codebook reads of the next are on their way, so that between two units there is only the
// epilogue.  One barrier per chunk of activations.
template <typename FMT, bool SMALL, int TERMS, bool GATE_UP>
__global__ __launch_bounds__(64 * kWaves, 2) void moe_tile_kernel(
    TileArgs a, const int4* __restrict__ tiles, const int32_t* __restrict__ n_tiles, const int64_t* __restrict__ route_tokens) {
    using S = TileShape<SMALL>;
    using Acc = typename S::Acc;
    extern __shared__ __align__(1024) unsigned char smem[];
    constexpr int kRows = S::kRows, kActOff = FMT::kTableBytes + kWaves * wave_slot(SMALL);
    constexpr int kRowBytes = SMALL ? 512 : 256, kPieces = kRowBytes / 16;           // of one row in a chunk (small tiles: of either block)
    constexpr int kDma = kChunk / 1024 / kWaves;                                     // direct-to-LDS instructions of a wave per chunk, 1 KB each
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane % S::kCols, part = lane / S::kCols;
    const int kp = a.bpr * 256, row_bytes = a.bpr * FMT::kBlockBytes, chunks = SMALL ? (a.bpr + 1) / 2 : 2 * a.bpr, grid = gridDim.x;

    const int tile_count = __builtin_amdgcn_readfirstlane(n_tiles[0]);
    // Waves of a workgroup that compute: as few as one round of the machine needs, as they share its LDS and SIMDs (32 experts of 3072 -> 1536 with 6 routes, gate / up:
    // 192 units of eight waves 41.9 us, 256 of six 38.0; 8 experts, in twos as before, 25)
    int width = kWaves, col_groups = (a.wave_cols + kWaves - 1) / kWaves;
    if constexpr (SMALL) {
#pragma unroll
        for (int w = kWaves - 1; w >= 1; --w) {
            const int groups = (a.wave_cols + w - 1) / w;
            if (tile_count * groups <= grid) width = w, col_groups = groups;
        }
    }
    width = __builtin_amdgcn_readfirstlane(width), col_groups = __builtin_amdgcn_readfirstlane(col_groups);
    const int units = tile_count * col_groups;
    // The units of a last round that would keep a few compute units busy for a whole round are dealt out by waves: `parts` workgroups
    // take kWaves / parts waves' columns each (a unit's waves share the LDS and the SIMDs of one compute unit otherwise).  2048 routes over 256
    // experts are 1536 units and a few for experts of more than 16 routes, whose round would take as long as each of the six before it.
    // (Those experts as tiles of 32 rows instead: IQ1_M 130 -> 126 us, but the registers of IQ2_XXS overflow, 272 -> 343.)
    const int whole_units = SMALL ? units - units % grid : units, left = units - whole_units;
    int parts = 1;
    if constexpr (SMALL) {
        for (int p = 2; p <= kWaves; ++p)
            if (kWaves % p == 0 && left * p <= grid && width == kWaves) parts = p;
    }
    const int total = whole_units + left * parts;
    if (static_cast<int>(blockIdx.x) >= total) return;

    struct Unit { int expert, first, routes, wave0, mine; };       // wave0: the first of its waves among the tile's; !mine: the wave only moves its share of the activations
    auto unit_at = [&](int at) {
        const bool split = at >= whole_units;
        const int unit = split ? whole_units + (at - whole_units) / parts : at, part_of = split ? (at - whole_units) % parts : 0;
        const int4 t = tiles[unit / col_groups];
        const auto scalar = [](int value) { return __builtin_amdgcn_readfirstlane(value); };       // (the same for all lanes, and so is what follows from it)
        return Unit{scalar(t.x), scalar(t.y), scalar(t.z), scalar(unit % col_groups * width), scalar(wave < width && (!split || wave / (kWaves / parts) == part_of))};
    };
    int at = blockIdx.x;
    Unit u = unit_at(at);

    // ---- weights, a block of the wave's rows at a time --------------------------------------------------------------------
    // A block's bytes are fetched with four neighbouring lanes on one weight row (set s, half k: rows 16 k .. 16 k + 15 of the set's 32),
    // then turned in the wave's own LDS slot: asked for by the lanes that decode them, every instruction would touch 32 rows' lines
    // (the fetches then cost 100 of 383 us at 256 experts and 2048 routes).
    const bool word_rows = (row_bytes & 3) == 0 && ((reinterpret_cast<uintptr_t>(a.w0) | (GATE_UP ? reinterpret_cast<uintptr_t>(a.w1) : 0)) & 3) == 0;
    const int piece = lane & 3;
    const uint8_t *base0, *base1;
    int c0, c1, expert, block;                      // first weight row of either set, expert and block that the bases stand at
    auto to_block = [&]() {             // (scalar arithmetic)
        const size_t from = static_cast<size_t>(__builtin_amdgcn_readfirstlane(expert)) * a.n * row_bytes + __builtin_amdgcn_readfirstlane(block) * FMT::kBlockBytes;
        base0 = a.w0 + from;
        base1 = (GATE_UP ? a.w1 : a.w0) + from;
    };
    auto to_unit = [&](const Unit& v) {
        expert = v.expert;
        c0 = (v.wave0 + wave) * (GATE_UP ? kWaveCols : 2 * kWaveCols);
        c1 = GATE_UP ? c0 : c0 + kWaveCols;
        block = 0;
    };
    typename FMT::Piece fetched[2][2];
    auto words = [&]() { return word_rows && (block & 1) == 0; };
    auto fetch = [&](int s, int k) {                // (24-bit product: rows and bytes of a row lie below 2^24, an expert's matrix below 2^32)
        const uint32_t row = min(__builtin_amdgcn_readfirstlane(s ? c1 : c0) + 16 * k + (lane >> 2), a.n - 1);
        FMT::load_piece(fetched[s][k], s ? base1 : base0, __umul24(row, row_bytes), piece, words());
    };
    auto fetch_all = [&]() {
#pragma unroll
        for (int g = 0; g < 4; ++g) fetch(g >> 1, g & 1);
    };
    // to the block after the one that was fetched last (behind a unit's last: the first of unit `following`, or what was fetched before where there is none)
    auto advance = [&](int following) {
        if (block + 1 < a.bpr) ++block;
        else if (following < total) to_unit(unit_at(following));
        to_block();
    };
    unsigned char* slot = smem + FMT::kTableBytes + wave * wave_slot(SMALL);
    const uint32_t slot_in = (lane >> 2) * 64u + ((piece ^ ((lane >> 4) & 3)) << 4), slot_swz = ((r >> 2) & 3) << 4;
    typename FMT::Raw raw[S::kSets];
    uint32_t turned_d[2];                           // block scales of the bytes in `raw`: of sets 2 s and 2 s + 1 as two halves (small tiles), or of set s
    auto turn = [&]() {                             // (one wave's LDS operations take effect in order: the slot serves one half after the other)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                *reinterpret_cast<uint4*>(slot + (SMALL ? 0 : 1024 * k) + slot_in) = FMT::codes(fetched[s][k], piece, words());
                if constexpr (SMALL) FMT::template pick<4>(raw[2 * s + k], slot + r * 64, slot_swz, part);
            }
            if constexpr (!SMALL) FMT::template pick<2>(raw[s], slot + r * 64, slot_swz, part);
            if constexpr (FMT::kScaleApart) {       // from the first of a row's four lanes to the lanes that decode the row
                const uint32_t both = __builtin_amdgcn_perm(FMT::scale(fetched[s][1], words()), FMT::scale(fetched[s][0], words()), 0x05040100u);
                turned_d[s] = __builtin_amdgcn_ds_bpermute(16 * (r & 15), both);
                if constexpr (!SMALL) turned_d[s] >>= r & 16;
            }
        }
    };

    // ---- activations -----------------------------------------------------------------------------------------------------------
    // Instruction q of a chunk fills 1 KB: rows of kRowBytes each, 16-byte piece p of row r at position p ^ (r % kPieces).  A chunk of up to 64 rows
    // holds eight neighbouring pieces of either half of the block.  Rows that the tile does not have are left as they are: theirs are the
    // products that nobody stores.
    uint32_t xoff[kDma];
    int x_rows;                                     // of the tile whose activations are on their way
    auto to_rows = [&](const Unit& v, int lane_token) {
        x_rows = v.routes * TERMS;
#pragma unroll
        for (int i = 0; i < kDma; ++i) {
            const int q = wave + kWaves * i, row = (q * (1024 / kRowBytes)) % kRows + lane / kPieces, at_piece = (lane ^ row) & (kPieces - 1);
            const uint32_t src = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(4 * min(row / TERMS, v.routes - 1), lane_token)) * (GATE_UP ? TERMS : 1) + (GATE_UP ? row % TERMS : 0);
            xoff[i] = src * (2u * kp) + (SMALL ? 16u * at_piece : 16u * (at_piece & 7) + 256u * (at_piece >> 3));
        }
    };
    auto dma = [&](int chunk, int to) {             // chunk of the tile into place `to` of the ring
        const unsigned char* src = reinterpret_cast<const unsigned char*>(a.rows) + (SMALL ? 1024 * chunk : 512 * (chunk >> 1) + 128 * (chunk & 1));
#pragma unroll
        for (int i = 0; i < kDma; ++i) {
            const int q = wave + kWaves * i, second = SMALL && q >= 8;
            if ((q * (1024 / kRowBytes)) % kRows < x_rows && (!SMALL || 2 * chunk + second < a.bpr))
                lds_dma16_at(src + 512 * second, xoff[i], __builtin_amdgcn_readfirstlane(kActOff + to * kChunk + q * 1024));
        }
    };
    // the row that lane l's route of the tile has among the activations (its token, or itself), and the epilogue's factors of that route
    auto token_of = [&](const Unit& v) {
        const int route = v.first + min(lane, v.routes - 1);
        return GATE_UP ? static_cast<int>(route_tokens[route]) : route;
    };

    int ring = 0, lane_token = token_of(u);
    const int ahead = chunks > 1 ? 2 : 1;           // chunks on their way
    to_unit(u);
    to_block();
    fetch_all();
    FMT::stage_tables(smem, tid);                   // (while the first loads are on their way; visible behind the first barrier)
    to_rows(u, lane_token);
    for (int c = 0; c < ahead; ++c) dma(c, c);
    const uint32_t copy = FMT::table_lane(lane);
    const uint32_t abase = static_cast<uint32_t>(r) * kRowBytes | (static_cast<uint32_t>((r ^ 8 * part) & (kPieces - 1)) << 4);
    typename FMT::Look look[S::kSets];              // codebook reads run one entry ahead, activation reads too
    uint4 bw[S::kSets];
    turn();
    wait_vm<0>();
    advance(at + grid);
    fetch_all();
    __syncthreads();                                // the first chunks and the tables are there (the second blocks are still on their way)
#pragma unroll
    for (int s = 0; s < S::kSets; ++s) {
        FMT::template look<0>(look[s], raw[s], copy);
        bw[s] = FMT::finish(look[s]);
        FMT::template look<1>(look[s], raw[s], copy);
    }

    for (;;) {
        const int next_at = at + grid;
        const bool has_next = next_at < total;
        const Unit v = has_next ? unit_at(next_at) : u;
        const int col0 = (u.wave0 + wave) * (GATE_UP ? kWaveCols : 2 * kWaveCols), col1 = GATE_UP ? col0 : col0 + kWaveCols;
        int next_token = 0;
        float lane_unscale = 0.0f, lane_weight = 0.0f;
        // Gate of chunk `chunk`: all that is outstanding was asked for about a chunk ago, the chunk after this one among it.  Behind the barrier every
        // wave has left the chunk before this one, whose place the next to load takes.
        auto gate = [&](int chunk, auto newer) {    // (newer: loads behind those that are waited for)
            wait_and_meet<decltype(newer)::value>();
            const int load = chunk + ahead, to = ahead == 2 ? ring_after(ring_after(ring)) : ring_after(ring);
            if (load < chunks) {
                dma(load, to);
            } else if (has_next) {
                if (load == chunks) to_rows(v, next_token);
                dma(load - chunks, to);
            }
            ring = ring_after(ring);
        };
        auto blocks = [&](auto kMt) {
            constexpr int kM = kMt, kAv = kM == 1 ? 2 : 1;      // (64 rows: registers for one step's activations)
            constexpr int kTurn = S::kSteps - 3;                // step at whose end the next block's bytes are turned and those of the one after it asked for
            Acc acc[kM][S::kSets];
#pragma unroll
            for (int m = 0; m < kM; ++m)
#pragma unroll
                for (int s = 0; s < S::kSets; ++s) acc[m][s] = Acc{};
            const Acc zero = {};
            uint32_t now = kActOff + ring * kChunk + abase;     // LDS address of the lane's rows in the chunk being read
            uint4 av[kAv][kM];
#pragma unroll
            for (int m = 0; m < kM; ++m) av[0][m] = lds_read16(now + m * 32 * kRowBytes);
#pragma unroll 1
            for (int b = 0; b < a.bpr; ++b) {
                Acc c[kM][S::kSets];
                float d[S::kSets];
#pragma unroll
                for (int s = 0; s < S::kSets; ++s)
                    d[s] = FMT::kScaleApart ? 0.125f * f16_bits_to_float((SMALL ? turned_d[s >> 1] >> (16 * (s & 1)) : turned_d[s & 1]) & 0xffffu) : FMT::block_scale(raw[s]);
                // step i: matrix instructions of entry i, the second half of the decode of entry i + 1, LDS reads for later entries
                static_for<0, S::kSteps>([&](auto I) {
                    constexpr int i = I;
                    if constexpr (i == 0) {
                        if (b == 0) next_token = token_of(v);
                    }
                    if constexpr (!SMALL && i == kTurn - 8) gate(2 * b, std::integral_constant<int, 4 * FMT::kLoads>{});
                    // where the activations of step i + 1 lie
                    constexpr int n = (i + 1) % S::kSteps, kStep = (SMALL ? n : n & 7) << 4;
                    if constexpr (i + 1 == S::kSteps || (!SMALL && i == 7)) {
                        if (SMALL && !(b & 1) && b + 1 < a.bpr) now += 8192;
                        else now = kActOff + ring * kChunk + abase;
                    }
                    const uint32_t from = now ^ kStep;
                    if constexpr (kAv == 2) {
#pragma unroll
                        for (int m = 0; m < kM; ++m) av[(i + 1) % kAv][m] = lds_read16(from + m * 32 * kRowBytes);
                    }
                    static_for<0, kM * S::kSets>([&](auto U) {
                        constexpr int m = U / S::kSets, s = U % S::kSets;
                        c[m][s] = mfma(av[i % kAv][m], bw[s], i == 0 ? zero : c[m][s]);
                        if constexpr (kAv == 1 && s == S::kSets - 1) av[0][m] = lds_read16(from + m * 32 * kRowBytes);
                        if constexpr (m == kM - 1) {
                            bw[s] = FMT::finish(look[s]);
                            FMT::template look<(i + 2) % S::kSteps>(look[s], raw[s], copy);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    if constexpr (i == kTurn) {     // (the last entries of `raw` have been looked up)
                        if (!SMALL || (b & 1) || b + 1 == a.bpr) gate(SMALL ? b >> 1 : 2 * b + 1, std::integral_constant<int, 0>{});
                        turn();
                        advance(a.bpr > 1 ? next_at : next_at + grid);
                        if (b + 1 == a.bpr) {
                            lane_unscale = a.unscale ? a.unscale[lane_token] : 1.0f;
                            if constexpr (GATE_UP) lane_weight = a.route_weights[u.first + min(lane, u.routes - 1)];
                        }
                        fetch_all();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
#pragma unroll
                for (int s = 0; s < S::kSets; ++s)
#pragma unroll
                    for (int m = 0; m < kM; ++m)
#pragma unroll
                        for (int e = 0; e < S::kRegs; ++e) acc[m][s][e] += d[s] * c[m][s][e];
            }
            float* factors = reinterpret_cast<float*>(slot);      // (the wave's own, free until its next turn)
            factors[lane] = lane_unscale;
            if constexpr (GATE_UP) factors[kTileRows + lane] = lane_weight;
            // Stores go through buffers that end with the tile's last route: what lies beyond is dropped, so every lane stores without a branch.
            const auto out = __builtin_amdgcn_make_buffer_rsrc(a.out + static_cast<size_t>(u.first) * a.out_pitch, 0, u.routes * a.out_pitch * 4, 0x00020000);
            // lane: column r of each set; matrix rows 4 part + e of 16, or 8 (e / 4) + 4 part + e % 4 of each 32: four neighbouring rows at a time
            uint32_t at_col[S::kSets];
#pragma unroll
            for (int s = 0; s < S::kSets; ++s) {
                int col = (!GATE_UP && s >= S::kSets / 2 ? col1 : col0) + (s % (S::kSets / 2)) * S::kCols + r;
                asm volatile("" : "+v"(col));
                at_col[s] = col < (GATE_UP ? a.out_pitch : a.n) ? 4u * col : 0x80000000u;
            }
            const uint32_t pitch = 4u * a.out_pitch;
            // (kept from being worked out ahead of the loop over the units: some thirty row offsets and columns in scratch memory, each of whose reloads
            // waits for the loads of the next unit: 8 - 11 us per unit)
            uint32_t first_row = part * (4 / TERMS);
            asm volatile("" : "+v"(first_row));
            const float* row_factors = factors + first_row;
            const uint32_t row_start = __umul24(first_row, pitch);
#pragma unroll
            for (int m = 0; m < kM; ++m)
#pragma unroll
                for (int e = 0; e < S::kRegs; e += 4) {
                    const int row = (SMALL ? 0 : 32 * m + 2 * e) / TERMS;      // beyond the lane's first (8 (e / 4) = 2 e)
#pragma unroll
                    for (int s = 0; s < (GATE_UP ? S::kSets / 2 : S::kSets); ++s) {
                        float value[4 / TERMS];
#pragma unroll
                        for (int q = 0; q < 4 / TERMS; ++q) {
                            auto total_of = [&](int set) { return (acc[m][set][e + TERMS * q] + (TERMS == 2 ? acc[m][set][e + TERMS * q + TERMS - 1] : 0.0f)) * row_factors[row + q]; };
                            value[q] = total_of(s);
                            if constexpr (GATE_UP) {
                                float g = value[q], up = total_of(s + S::kSets / 2);
                                if (a.limit > 0.0f) {
                                    up = fminf(fmaxf(up, -a.limit), a.limit);
                                    g = fminf(g, a.limit);
                                }
                                // (a division: v_rcp_f32, 3 % of the launch faster, is a unit in the last place off and flushes what 1 + exp(-g) beyond 2^126 gives)
                                value[q] = col0 + s * S::kCols + r < a.n ? g / (1.0f + expf(-g)) * up * row_factors[kTileRows + row + q] : 0.0f;   // (padding columns: zeros)
                            }
                        }
#pragma unroll
                        for (int q = 0; q < 4 / TERMS; ++q) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(value[q]), out, row_start + at_col[s] + (row + q) * pitch, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        if constexpr (SMALL) {
            if (!u.mine) {                          // the barriers of the waves that compute (a unit that is dealt out is a workgroup's last)
                for (int c = 0; c < chunks; ++c) gate(c, std::integral_constant<int, 0>{});
                return;
            }
            blocks(std::integral_constant<int, 1>{});
        } else if (u.routes * TERMS > kTileRows / 2) {
            blocks(std::integral_constant<int, 2>{});
        } else {
            blocks(std::integral_constant<int, 1>{});
        }
        if (!has_next) break;
        at = next_at;
        u = v;
        lane_token = next_token;
        if (ahead == 1) {                           // (one chunk per unit: it is not waited for by the gate before it)
            wait_and_meet<0>();
        }
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

// hidden rows of the down projection: h16[route][k] = h[route][k] * s, s the power of two of rows_scale for the route's largest
// magnitude; unscale[route] = 1 / s.  One workgroup per route; every thread keeps its pieces of four values, so a row of up to 1024 * HELD is read once.
template <int HELD>
__global__ __launch_bounds__(256) void rows_hidden_half_kernel(const float* __restrict__ h, int h_kpad, _Float16* __restrict__ h16, float* __restrict__ unscale) {
    __shared__ float part[4];
    const int route = blockIdx.x, tid = threadIdx.x, pieces = h_kpad / 4;
    const float4* src = reinterpret_cast<const float4*>(h + static_cast<size_t>(route) * h_kpad);
    float4 v[HELD];
    float am = 0.0f;
    auto take = [&](const float4& x) { am = fmaxf(fmaxf(fmaxf(am, fabsf(x.x)), fmaxf(fabsf(x.y), fabsf(x.z))), fabsf(x.w)); };
#pragma unroll
    for (int j = 0; j < HELD; ++j) v[j] = src[tid + 256 * j < pieces ? tid + 256 * j : 0];
#pragma unroll
    for (int j = 0; j < HELD; ++j) take(v[j]);
    for (int k = tid + 256 * HELD; k < pieces; k += 256) take(src[k]);
    am = group_max<64>(am);
    if ((tid & 63) == 0) part[tid >> 6] = am;
    __syncthreads();
    const float s = rows_scale(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
    uint2* dst = reinterpret_cast<uint2*>(h16 + static_cast<size_t>(route) * h_kpad);
    auto put = [&](int k, const float4& x) {
        union { _Float16 h[4]; uint2 u; } c;
        c.h[0] = static_cast<_Float16>(x.x * s); c.h[1] = static_cast<_Float16>(x.y * s);
        c.h[2] = static_cast<_Float16>(x.z * s); c.h[3] = static_cast<_Float16>(x.w * s);
        dst[k] = c.u;
    };
#pragma unroll
    for (int j = 0; j < HELD; ++j)
        if (tid + 256 * j < pieces) put(tid + 256 * j, v[j]);
    for (int k = tid + 256 * HELD; k < pieces; k += 256) put(k, src[k]);
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

struct TileList { const int4* tiles; const int32_t* count; const int64_t* route_tokens; };     // {expert, first route, routes, 0}

template <typename FMT, bool SMALL, int TERMS, bool GATE_UP>
int launch_tiles_rows(TileArgs a, const TileList& list, int most_tiles, hipStream_t stream) {
    static SmemGrant granted;
    constexpr size_t smem = FMT::kTableBytes + kWaves * wave_slot(SMALL) + kRing * kChunk;
    static_assert(smem <= 160 * 1024, "tables, slots and ring fit the LDS");
    auto kern = moe_tile_kernel<FMT, SMALL, TERMS, GATE_UP>;
    if (!grant_dynamic_smem(reinterpret_cast<const void*>(kern), smem, granted)) return PLLM_ERR_UNSUPPORTED;
    static const bool starts_at_0 = [&]() {
        hipFuncAttributes f;
        return hipFuncGetAttributes(&f, reinterpret_cast<const void*>(kern)) == hipSuccess && f.sharedSizeBytes == 0;
    }();
    if (!starts_at_0) return PLLM_ERR_UNSUPPORTED;
    const int wave_width = GATE_UP ? kWaveCols : 2 * kWaveCols;
    a.wave_cols = ((GATE_UP ? a.out_pitch : a.n) + wave_width - 1) / wave_width;
    // (tiles of 16 rows: one workgroup per compute unit whatever the number of units, since the kernel deals out units by waves.  Gate / up and down with
    // everything around them, us, one workgroup per unit / per compute unit: 8 experts of 3072 -> 1536 with 16 routes 123 / 85, 16 with 96 126 /
    // 89, 32 with 64 126 / 104, 64 of 2048 -> 768 with 128 103 / 93; 64 of 2048 -> 1280 and larger sets alike)
    const long long units = static_cast<long long>(most_tiles) * ((a.wave_cols + kWaves - 1) / kWaves);
    const int grid = SMALL ? compute_units() : static_cast<int>(std::min<long long>(units, compute_units()));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * kWaves), smem, stream, a, list.tiles, list.count, list.route_tokens);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}
template <typename FMT, int TERMS, bool GATE_UP>
int launch_tiles(const TileArgs& a, const TileList& list, int most_tiles, bool small, hipStream_t stream) {
    return small ? launch_tiles_rows<FMT, true, TERMS, GATE_UP>(a, list, most_tiles, stream) : launch_tiles_rows<FMT, false, TERMS, GATE_UP>(a, list, most_tiles, stream);
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
    // activation rows are addressed with 32-bit byte offsets, and so are the rows of one expert's matrices and those of a tile's outputs
    if (dim >= (1 << 20) || inter >= (1 << 20)) return false;
    const unsigned long long kx = (static_cast<unsigned long long>(dim) + 255) / 256 * 256, kh = (static_cast<unsigned long long>(inter) + 255) / 256 * 256;
    const unsigned long long x_bytes = 4ull * tokens * kx, h_bytes = 2ull * routes * kh, w_bytes = std::max(kx * inter, kh * dim);
    return x_bytes < (1ull << 32) && h_bytes < (1ull << 32) && w_bytes < (1ull << 32);
}

size_t moe_rows_x_bytes(int64_t tokens, int64_t dim) {
    const size_t kpad = static_cast<size_t>((dim + 255) / 256) * 256;
    return align256(static_cast<size_t>(tokens) * 2 * kpad * sizeof(_Float16)) + align256(static_cast<size_t>(tokens) * sizeof(float));
}

// hidden rows of the routes: float32 values [routes][h_kpad], half-precision rows, 1 / scale
struct RowsHidden { float* values; _Float16* half_rows; float* unscale; size_t bytes; };

static RowsHidden rows_hidden(void* ws, int64_t routes, int64_t inter) {
    const size_t kpad = static_cast<size_t>((inter + 255) / 256) * 256, r = static_cast<size_t>(routes);
    unsigned char* p = static_cast<unsigned char*>(ws);
    RowsHidden h;
    h.values = reinterpret_cast<float*>(p);        p += align256(r * kpad * sizeof(float));
    h.half_rows = reinterpret_cast<_Float16*>(p);  p += align256(r * kpad * sizeof(_Float16));
    h.unscale = reinterpret_cast<float*>(p);       p += align256(r * sizeof(float));
    h.bytes = static_cast<size_t>(p - static_cast<unsigned char*>(ws));
    return h;
}

size_t moe_rows_h_bytes(int64_t routes, int64_t inter) { return rows_hidden(nullptr, routes, inter).bytes; }

size_t moe_tiles_list_bytes(int64_t routes) { return align256(static_cast<size_t>(routes) * sizeof(int4)) + 256; }

namespace {
// matrix rows per expert on average up to which tiles of 16 rows are taken (us for gate / up + down, 16- / 64-row tiles, 256 experts of 3072 ->
// 1536: 8 rows on average 402 / 474, 12 rows 434 / 485, 14 rows 486 / 490, 16 rows 554 / 496, as half of the experts then need two of the small tiles).
// Other sets go up at the line, so theirs lies further on: the whole call at 13 / 14 rows, bf16, 16 experts of 4096 -> 1536 69 / 91 us, 64 of 3072 -> 1536 132 / 151, 128 of
// 2048 -> 768 102 / 113; with float32 rows (6.4 / 8 routes) 16 of 4096 -> 1536 67 / 86, 128 of 2048 -> 768 94 / 103
constexpr int kSmallTileRows = 13;
bool small_tiles(int terms, int routes, int n_experts) { return static_cast<long long>(routes) * terms <= static_cast<long long>(kSmallTileRows) * n_experts; }
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
    // fp16 rows of whole blocks go in as the caller holds them: the same bits, for subnormal values too (rows_tiles.h says why), and the launch that scales
    // rows saved (5.1 us at 1024 tokens of 3072, 3.7 at 256)
    const bool held = x_dtype == PLLM_F16 && dim == kpad && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    int st = held ? PLLM_OK : half_rows_stage(x, x_dtype, tokens, dim, kpad, x_rows, unscale, stream);
    if (st != PLLM_OK) return st;
    const TileList list = {static_cast<const int4*>(list_ws), moe_tile_list_count(list_ws, routes), route_tokens};
    TileArgs a{};
    a.rows = held ? static_cast<const _Float16*>(x) : x_rows;
    a.unscale = held ? nullptr : unscale;
    a.route_weights = route_weights;
    a.w0 = w1;
    a.w1 = w3;
    a.out = hid.values;
    a.limit = limit;
    a.bpr = bpr;
    a.n = inter;
    a.out_pitch = h_kpad;
    const bool small = small_tiles(terms, routes, n_experts);
    const int per_tile = (small ? 16 : kTileRows) / terms, tiles = moe_tile_list_most(routes, n_experts, per_tile);
    st = moe_tile_list(seg, n_experts, per_tile, routes, list_ws, stream);
    if (st != PLLM_OK) return st;
    st = terms == 2 ? launch_tiles<TileIQ2XXS, 2, true>(a, list, tiles, small, stream) : launch_tiles<TileIQ2XXS, 1, true>(a, list, tiles, small, stream);
    if (st != PLLM_OK) return st;
    hipLaunchKernelGGL(rows_hidden_half_kernel<2>, dim3(routes), dim3(256), 0, stream, hid.values, h_kpad, hid.half_rows, hid.unscale);
    return hipGetLastError() == hipSuccess ? PLLM_OK : PLLM_ERR_LAUNCH;
}

// partial [routes][dim] = W2_e times the half-precision hidden rows of every route
int moe_tiles_w2(void* h_rows_ws, void* list_ws, int x_dtype, int inter, const int32_t* seg, const uint8_t* w2, float* partial, int dim, int n_experts,
                 int routes, hipStream_t stream) {
    const RowsHidden hid = rows_hidden(h_rows_ws, routes, inter);
    const TileList list = {static_cast<const int4*>(list_ws), moe_tile_list_count(list_ws, routes), nullptr};
    TileArgs a{};
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
    return launch_tiles<TileIQ1M, 1, false>(a, list, moe_tile_list_most(routes, n_experts, per_tile), small, stream);
}

}  // namespace pllm
