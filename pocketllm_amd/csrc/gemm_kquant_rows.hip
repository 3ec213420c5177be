// y[T, N] = x[T, K] . dequant(W)[N, K]^T over raw Q6_K, IQ4_XS and Q2_K super-blocks for the row counts between decode and prompts, on f16 MFMA.
//
// The group's whole-number scale goes either on the group's sums, in float32 (IQ4_XS, and Q6_K up to 32 matrix rows), or on the codes:
// a code times that scale is exact in half precision once the scale's lowest bit goes into an operand of its own
// (Q2_K, where both are small, uses that second operand for the minima), and so are bf16 / fp16 activations scaled by a power of two per
// row (fp16 rows of whole super-blocks go in as the caller holds them, float32 rows as two half-precision terms = two matrix rows): a block's sums come out of the matrix cores in float32 without any
// operand rounding, and its float scale goes on once.  Against float64: 1e-7; the tile kernel, which rounds the decoded weight to a half, 2e-4.
//
// A workgroup owns 32 matrix rows (16 in LDS where the call has no more) and 128 weight rows (four waves) or 64 and 256 (eight waves), over a slice of K; a step is one super-block
// of every weight row.  A wave's 32 blocks come to registers two steps ahead, neighbouring lanes on neighbouring 16-byte pieces of a row, and
// go from there into the wave's own LDS slot, which it reads in the order of the matrix operand: lane (n, h) = row n, eight codes 16 G + 8 h ..
// of 16-column group G.  (Rows of a slot are an odd number of 16-byte pieces apart, so 32 rows read at one place meet no bank more often than the
// width of the read asks for.)  Activation rows come to LDS by direct-to-LDS loads, 256 columns at a time, double-buffered, 16-byte piece p of
// row r at position p ^ (r % 32).  One barrier per step.
//
// Bound: decode and scaling in the waves (vector ALU 38 % with 1.6 waves per SIMD, LDS 22 %; Q6_K 5120x17408 at 7 rows, this kernel alone: 21.3 us; where it took
// 24.2 it took 21.9 without its weight loads, and the weight loads alone 15.5, which is what HBM gives).  The tile kernel of prompts
// (gemm_tile.h) would take these calls too, with every weight rounded to a half.  us, bf16 rows, that one / this one:
//   Q6_K    5120x17408  8 rows 43.7 / 30.9, 64 rows 47.0 / 45.7     17408x5120  8 rows 41.1 / 30.3     5120x5120  16 rows 22.7 / 17.6     2048x3072  16 rows 17.9 / 11.7
//   IQ4_XS  5120x17408 16 rows 34.5 / 26.5, 64 rows 38.4 / 37.5     17408x5120 16 rows 31.5 / 26.8     5120x5120  16 rows 19.6 / 16.5     2048x3072  16 rows 14.9 / 11.5
//   Q2_K    5120x17408  8 rows 28.2 / 25.7, 64 rows 32.7 / 36.7     17408x5120  8 rows 25.2 / 25.8     5120x5120  16 rows 16.9 / 16.0     2048x3072  16 rows 13.4 / 11.8
// The calls in which that one is faster by now stay here for their bits.
// (Blocks one step ahead instead of two, Q6_K 5120x17408 at 7 rows: 2.7 us more.  Its rows from between two words as they lie, without the shift: 24 rows
// 38.0 against 35.5, 5120x5120 32 rows 21.9 / 20.4.)
#include "rows_tiles.h"

namespace pllm {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t add_pair(uint32_t halves, float v) {
    const v2h b = {static_cast<_Float16>(v), static_cast<_Float16>(v)};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, halves) + b);
}
// eight unsigned code bytes -> eight halves code - BIAS (1024 + code on the bits, then one packed addition)
template <int BIAS> __device__ __forceinline__ uint4 code_halves(uint2 c) {
    return make_uint4(add_pair(__builtin_amdgcn_perm(0x64646464u, c.x, 0x04010400u), -1024.0f - BIAS), add_pair(__builtin_amdgcn_perm(0x64646464u, c.x, 0x04030402u), -1024.0f - BIAS),
                      add_pair(__builtin_amdgcn_perm(0x64646464u, c.y, 0x04010400u), -1024.0f - BIAS), add_pair(__builtin_amdgcn_perm(0x64646464u, c.y, 0x04030402u), -1024.0f - BIAS));
}

__device__ __forceinline__ uint4 times_pair(uint4 u, v2h s) {
    auto times = [&](uint32_t p) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, p) * s); };
    return make_uint4(times(u.x), times(u.y), times(u.z), times(u.w));
}
// codes times a whole-number scale as two exact operands: times the scale without its lowest bit (at most 2^12 and even), and the codes again
// where that bit is set
__device__ __forceinline__ void scaled_codes(uint4 u, int scale, uint4& first, uint4& second) {
    const _Float16 e = static_cast<_Float16>(static_cast<short>(scale & ~1));
    const uint32_t odd = static_cast<uint32_t>(-(scale & 1));
    first = times_pair(u, v2h{e, e});
    second = make_uint4(u.x & odd, u.y & odd, u.z & odd, u.w & odd);
}

// A format: kPieces 16-byte pieces of a block from kFirst on come to the slot (kStride bytes per row), its tail behind them.  head: what the whole block shares; d and e multiply the sums of the first and of the second operand.  raw<G>: the LDS
// reads of 16-column group G; operands<G>: the lane's eight columns of it.
struct RowsQ6K {
    static constexpr int kBlockBytes = 210, kFirst = 0, kPieces = 13, kStride = 208;
    static constexpr bool kHalfWords = true;                 // every other block of a row starts between two words
    struct Head { uint4 sc; float d, e; };
    struct Raw { uint2 ql, qh; };
    static __device__ __forceinline__ uint16_t load_tail(const uint8_t* blk) { return *reinterpret_cast<const uint16_t*>(blk + 208); }
    static __device__ __forceinline__ Head head(const unsigned char* row, uint32_t tail) {
        const float d = f16_bits_to_float(tail);
        return Head{*reinterpret_cast<const uint4*>(row + 192), d, d};
    }
    template <int G> static __device__ __forceinline__ Raw raw(const unsigned char* row, int h) {
        constexpr int half = G >> 3, j = (G & 7) >> 1, e = G & 1;
        return Raw{*reinterpret_cast<const uint2*>(row + 64 * half + 32 * (j & 1) + 16 * e + 8 * h), *reinterpret_cast<const uint2*>(row + 128 + 32 * half + 16 * e + 8 * h)};
    }
    template <int G> static __device__ __forceinline__ uint4 codes(const Raw& w) {
        constexpr int j = (G & 7) >> 1, nib = 4 * (j >> 1), up = 4 - 2 * j;              // (the two upper bits to bits 4 and 5 of their byte)
        auto word = [&](uint32_t ql, uint32_t qh) {
            const uint32_t high = up > 0 ? qh << (up > 0 ? up : 0) : qh >> (up < 0 ? -up : 0);
            return (((ql >> nib) & 0x0f0f0f0fu) | (high & 0xf0f0f0f0u)) & 0x3f3f3f3fu;
        };
        return code_halves<32>(make_uint2(word(w.ql.x, w.qh.x), word(w.ql.y, w.qh.y)));
    }
    // sets of groups that share their bytes, in the order they are taken: (half, e), j = 0 .. 3
    static constexpr int kSets = 4, kChain = 1;
    struct Set { uint2 ql[2], qh; };
    static constexpr int group(int t) { return 8 * (t >> 3) + 2 * (t & 3) + ((t >> 2) & 1); }
    template <int S> static __device__ __forceinline__ Set set(const unsigned char* row, int h) {
        constexpr int half = S >> 1, e = S & 1;
        return Set{{*reinterpret_cast<const uint2*>(row + 64 * half + 16 * e + 8 * h), *reinterpret_cast<const uint2*>(row + 64 * half + 32 + 16 * e + 8 * h)},
                   *reinterpret_cast<const uint2*>(row + 128 + 32 * half + 16 * e + 8 * h)};
    }
    template <int T> static __device__ __forceinline__ uint4 set_codes(const Set& w) { return codes<group(T)>(Raw{w.ql[T & 1], w.qh}); }
    template <int G> static __device__ __forceinline__ int group_scale(const Head& a) {
        const uint32_t sc = G < 4 ? a.sc.x : G < 8 ? a.sc.y : G < 12 ? a.sc.z : a.sc.w;
        return static_cast<int8_t>(sc >> (8 * (G & 3)));
    }
    template <int G> static __device__ __forceinline__ void operands(const Head& a, const Raw& w, uint4& first, uint4& second) {
        scaled_codes(codes<G>(w), group_scale<G>(a), first, second);
    }
};

struct RowsIQ4XS {
    static constexpr int kBlockBytes = 136, kFirst = 8, kPieces = 8, kStride = 144;
    static constexpr bool kHalfWords = false;
    struct Head { uint32_t lo, hi; float d, e; };            // scales_l, scales_h
    struct Raw { uint2 q; };
    static __device__ __forceinline__ uint2 load_tail(const uint8_t* blk) { return *reinterpret_cast<const uint2*>(blk); }
    static __device__ __forceinline__ Head head(const unsigned char*, uint2 tail) {
        const float d = f16_bits_to_float(tail.x & 0xffffu);
        return Head{tail.y, tail.x >> 16, d, d};
    }
    static __device__ __forceinline__ uint32_t values4(uint32_t codes) {                 // kvalues[code] + 128, four at a time: the lower nibbles of the bytes
        const uint32_t low3 = codes & 0x07070707u;
        const uint32_t lower = __builtin_amdgcn_perm(0x766A5D4Fu, 0x3F2D1801u, low3);   // 1 24 45 63 | 79 93 106 118
        const uint32_t upper = __builtin_amdgcn_perm(0xF1D9C5B5u, 0xA6998D81u, low3);   // 129 141 153 166 | 181 197 217 241
        return __builtin_amdgcn_perm(upper, lower, ((codes >> 1) & 0x04040404u) | 0x03020100u);
    }
    template <int G> static __device__ __forceinline__ Raw raw(const unsigned char* row, int h) { return Raw{*reinterpret_cast<const uint2*>(row + 16 * (G >> 1) + 8 * h)}; }
    template <int G> static __device__ __forceinline__ uint4 codes(const Raw& w) {
        constexpr int nib = 4 * (G & 1);                     // 32 weights of a scale: low nibbles the first 16, high nibbles the others
        return code_halves<128>(make_uint2(values4(w.q.x >> nib), values4(w.q.y >> nib)));
    }
    static constexpr int kSets = 8, kChain = 2;              // (a scale's 32 weights: the low and the high nibbles of the same bytes)
    using Set = Raw;
    static constexpr int group(int t) { return t; }
    template <int S> static __device__ __forceinline__ Set set(const unsigned char* row, int h) { return raw<2 * S>(row, h); }
    template <int T> static __device__ __forceinline__ uint4 set_codes(const Set& w) { return codes<T>(w); }
    template <int G> static __device__ __forceinline__ int group_scale(const Head& a) {
        constexpr int g = G >> 1;
        return static_cast<int>(((a.lo >> (4 * g)) & 15u) | (((a.hi >> (2 * g)) & 3u) << 4)) - 32;
    }
};

// (the second operand: sixteen times the group's minimum, so its sums are the minima times the activation sums)
struct RowsQ2K {
    static constexpr int kBlockBytes = 84, kFirst = 0, kPieces = 5, kStride = 80;
    static constexpr bool kHalfWords = false;
    struct Head { uint4 sc; float d, e; };
    struct Raw { uint2 q; };
    static __device__ __forceinline__ uint32_t load_tail(const uint8_t* blk) { return *reinterpret_cast<const uint32_t*>(blk + 80); }
    static __device__ __forceinline__ Head head(const unsigned char* row, uint32_t tail) {
        return Head{*reinterpret_cast<const uint4*>(row), f16_bits_to_float(tail & 0xffffu), -f16_bits_to_float(tail >> 16)};
    }
    static __device__ __forceinline__ v2h small_pair(uint32_t v) {                       // 0 .. 15 as two halves
        const v2h k = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-1024.0f)};
        return __builtin_bit_cast(v2h, v * 0x00010001u + 0x64006400u) + k;
    }
    template <int G> static __device__ __forceinline__ Raw raw(const unsigned char* row, int h) {
        return Raw{*reinterpret_cast<const uint2*>(row + 16 + 32 * (G >> 3) + 16 * (G & 1) + 8 * h)};
    }
    template <int G> static __device__ __forceinline__ void operands(const Head& a, const Raw& w, uint4& first, uint4& second) {
        constexpr int shift = 2 * ((G >> 1) & 3);
        const uint32_t word = G < 4 ? a.sc.x : G < 8 ? a.sc.y : G < 12 ? a.sc.z : a.sc.w, sc = (word >> (8 * (G & 3))) & 0xffu;
        first = times_pair(code_halves<0>(make_uint2((w.q.x >> shift) & 0x03030303u, (w.q.y >> shift) & 0x03030303u)), small_pair(sc & 15u));
        const uint32_t m = __builtin_bit_cast(uint32_t, small_pair(sc >> 4));
        second = make_uint4(m, m, m, m);
    }
};

__device__ __forceinline__ v16f rows_mfma(uint4 a, uint4 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// a wave's LDS: its pieces and the tails of its rows
template <typename FMT> constexpr int slot_bytes() { return kWaveCols * (FMT::kStride + static_cast<int>(sizeof(decltype(FMT::load_tail(nullptr))))); }

// SUMS > 0: calls of up to so many matrix rows whose group scales go on the groups' sums, in float32 (SUMS / 2 registers a lane; a matrix instruction
// has 32 rows, the sums of rows beyond are not looked at): one operand and one matrix instruction per group where codes times scale take two, and
// the bytes that several groups share are read once.  us, bf16 rows, scaled codes / scaled sums: Q6_K 5120x17408 8 rows 34.4 / 30.7, 16 rows 34.4 / 32.0, 32 rows
// 36.4 / 35.5; IQ4_XS 17408x5120 16 rows 31.0 / 26.7, 32 rows 32.1 / 29.4, 64 rows 40.2 / 37.7 (Q6_K at 64 rows would spill: 44.3 / 73.5).  Eight rows have a
// form of their own in Q6_K (17408x5120 31.3 / 30.2, 200064x3072 133.7 / 128.2).  Three workgroups per compute unit where registers allow it
// (IQ4_XS 17408x5120 16 rows 28.9 / 28.2 before the bytes were shared).
constexpr int matrix_rows(int mb, int sums) { return sums == 0 ? 32 * mb : sums <= 16 ? 16 : sums; }       // of a workgroup's LDS

template <typename FMT, int MB, int TERMS, int SUMS>
__global__ __launch_bounds__(64 * tile_waves(MB), (SUMS == 8 || SUMS == 16) && !FMT::kHalfWords ? 3 : 2) void kquant_rows_kernel(RowsArgs a) {
    extern __shared__ __align__(1024) unsigned char smem[];
    constexpr int kWaves = tile_waves(MB), kCols = kWaves * kWaveCols;
    constexpr int kRows = matrix_rows(MB, SUMS), kChunk = kRows * 512, kDma = kRows / 2 / kWaves;
    constexpr int kSums = SUMS / 2 / MB;                      // (SUMS: registers of a lane's sums that belong to rows of the call)
    constexpr int kTotal = kWaveCols * FMT::kPieces, kLoads = (kTotal + 63) / 64;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroups of one XCD (number modulo 8) take neighbouring tiles, those that share weights first
    const int total = a.row_tiles * a.col_tiles * a.slices, per = (total + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per || tile >= total) return;
    const auto scalar = [](int value) { return __builtin_amdgcn_readfirstlane(value); };       // (divisions leave them in vector registers)
    const int rt = scalar(tile % a.row_tiles), slice = scalar(tile / a.row_tiles % a.slices), ct = scalar(tile / (a.row_tiles * a.slices));
    const int b0 = slice * a.steps + min(slice, a.steps_more), b1 = b0 + a.steps + (slice < a.steps_more ? 1 : 0);
    const int t0 = rt * kRows, c0 = ct * kCols + wave * kWaveCols;

    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte_ptr)smem));
    unsigned char* slot = smem + 2 * kChunk + wave * slot_bytes<FMT>();
    const unsigned char* xb = reinterpret_cast<const unsigned char*>(a.rows) + static_cast<size_t>(t0) * 2 * a.kp;
    uint32_t xoff[kDma];
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
        const int row = 2 * (wave * kDma + i) + h;
        xoff[i] = static_cast<uint32_t>(min(row, a.m_rows - 1 - t0)) * (2u * a.kp) + 16u * (r ^ (row & 31));
    }
    auto dma = [&](int b, int buf) {
#pragma unroll
        for (int i = 0; i < kDma; ++i) lds_dma16_at(xb + 512 * static_cast<size_t>(b), xoff[i], lds0 + buf * kChunk + (wave * kDma + i) * 1024);
    };
    const size_t row_bytes = static_cast<size_t>(a.blocks) * FMT::kBlockBytes;
    const uint8_t* wtile = a.w + static_cast<size_t>(min(c0, a.n - 1)) * row_bytes;
    const int last_row = max(min(a.n - 1 - c0, kWaveCols - 1), 0);                // (rows past the end: the last one again, dropped at the store)
    uint32_t woff[kLoads], place[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int piece = min(64 * i + lane, kTotal - 1), row = piece / FMT::kPieces, p = piece - row * FMT::kPieces;
        woff[i] = static_cast<uint32_t>(min(row, last_row) * row_bytes) + FMT::kFirst + 16u * p;
        place[i] = row * FMT::kStride + 16 * p;
    }
    const uint32_t toff = static_cast<uint32_t>(min(r, last_row) * row_bytes);
    // blocks on their way: two steps ahead
    using Tail = decltype(FMT::load_tail(nullptr));
    struct Fetched { uint4 piece[kLoads]; std::conditional_t<FMT::kHalfWords, uint32_t, Tail> tail; };
    // Blocks that start between two words are fetched from two bytes earlier on, by whole words, and moved into place on their way to the slot; the
    // last two bytes come with the tail.  (A 16-byte load from between two words takes an access of the L1 per lane, not per four lanes.)
    const bool word_rows = FMT::kHalfWords && (row_bytes & 3) == 0 && (reinterpret_cast<uintptr_t>(a.w) & 3) == 0;
    auto moved = [&](int b) { return FMT::kHalfWords && word_rows && (b & 1); };
    Fetched set0, set1;
    Tail* tails = reinterpret_cast<Tail*>(slot + kWaveCols * FMT::kStride);      // [32] behind the pieces
    auto fetch = [&](int b, Fetched& f) {
        const uint8_t* base = wtile + static_cast<size_t>(b) * FMT::kBlockBytes;
        const uint8_t* from = base - (moved(b) ? 2 : 0);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) f.piece[i] = load16_a2(from + woff[i]);
        if constexpr (FMT::kHalfWords) {
            if (moved(b)) f.tail = *reinterpret_cast<const uint32_t*>(base + FMT::kStride - 2 + toff);
            else f.tail = FMT::load_tail(base + toff);
        } else {
            f.tail = FMT::load_tail(base + toff);
        }
    };
    auto put = [&](const Fetched& f, int b) {                        // (a wave's LDS operations take effect in order: what was read before is not touched)
        if constexpr (FMT::kHalfWords) {
            if (moved(b)) {
#pragma unroll
                for (int i = 0; i < kLoads; ++i) {
                    const uint4 v = f.piece[i];      // (the next lane's piece follows; behind the last lane's, the next load's first)
                    const uint32_t after = __builtin_amdgcn_update_dpp(__builtin_amdgcn_readfirstlane(f.piece[i + 1 < kLoads ? i + 1 : i].x), v.x, 0x130, 0xf, 0xf, false);
                    *reinterpret_cast<uint4*>(slot + place[i]) = make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, 16), __builtin_amdgcn_alignbit(v.z, v.y, 16),
                                                                           __builtin_amdgcn_alignbit(v.w, v.z, 16), __builtin_amdgcn_alignbit(after, v.w, 16));
                }
                *reinterpret_cast<uint16_t*>(slot + r * FMT::kStride + FMT::kStride - 2) = static_cast<uint16_t>(f.tail);
                tails[r] = static_cast<Tail>(f.tail >> 16);
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i) *reinterpret_cast<uint4*>(slot + place[i]) = f.piece[i];
        tails[r] = static_cast<Tail>(f.tail);        // (both halves of the wave: the same value)
    };

    v16f acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[m] = v16f{};
    const v16f zero = {};
    const int ar = r & (kRows < 32 ? 15 : 31);                 // (the instruction's rows 16 .. 31 are the first ones again)
    const uint32_t abase = static_cast<uint32_t>(ar) * 512u | (static_cast<uint32_t>(ar ^ h) << 4);
    const unsigned char* row = slot + r * FMT::kStride;
    dma(b0, 0);
    fetch(b0, set0);
    fetch(min(b0 + 1, b1 - 1), set1);
    put(set0, b0);
    wait_vm<kLoads + 1>();                           // (all but the second block)
    __syncthreads();
    // step of block b, held by the slot: block b + 1 is in `near`, block b + 2 goes to `far`
    auto step = [&](int b, int buf, Fetched& near, Fetched& far) {
        dma(min(b + 1, b1 - 1), buf ^ 1);
        fetch(min(b + 2, b1 - 1), far);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* at = smem + buf * kChunk;
        auto hd = FMT::head(row, tails[r]);
        asm("" : "+v"(hd.d), "+v"(hd.e));            // (float32 factors: as halves inside the multiply-adds they take twice the time)
        // piece of group G, half h: 2 G + h
        auto act_read = [&](int g, int m) { return *reinterpret_cast<const uint4*>(at + (abase ^ ((2 * g) << 4)) + m * 16384); };
        if constexpr (SUMS > 0) {
            // group t of the format's order: its matrix instruction, the scaling of the sums that are ready, the codes of group t + 1, the LDS reads of the
            // next set of groups and of the activations of group t + 2
            constexpr int kPer = 16 / FMT::kSets, kChain = FMT::kChain;          // kChain groups of one scale go through one chain of matrix instructions
            v16f c[2][MB];
            typename FMT::Set now = FMT::template set<0>(row, h), later;
            uint4 codes = FMT::template set_codes<0>(now), av[2][MB];
            float sums[MB][kSums], scale = 0.0f;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                av[0][m] = act_read(FMT::group(0), m);
                av[1][m] = act_read(FMT::group(1), m);
#pragma unroll
                for (int v = 0; v < kSums; ++v) sums[m][v] = 0.0f;
            }
            static_for<0, 16>([&](auto I) {
                constexpr int t = I, set = t / kPer, chain = t / kChain, next = t < 15 ? t + 1 : 15;
                uint4 next_codes;
                if constexpr (t % kPer == 0 && set + 1 < FMT::kSets) later = FMT::template set<(set + 1 < FMT::kSets ? set + 1 : set)>(row, h);
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    c[chain & 1][m] = rows_mfma(av[t & 1][m], codes, t % kChain == 0 ? zero : c[chain & 1][m]);
                    if constexpr (t < 14) av[t & 1][m] = act_read(FMT::group(t < 14 ? t + 2 : 15), m);
                    if constexpr (t < 15)
                        if (m == 0) next_codes = FMT::template set_codes<next>(next / kPer == set ? now : later);
                    if constexpr (t % kChain == kChain - 1 && chain > 0) {
#pragma unroll
                        for (int v = 0; v < kSums; ++v) sums[m][v] += scale * c[(chain & 1) ^ 1][m][v];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (t % kChain == kChain - 1) scale = static_cast<float>(FMT::template group_scale<FMT::group(t)>(hd));
                if constexpr (t < 15) codes = next_codes;
                if constexpr (next / kPer != set) now = later;
            });
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int v = 0; v < kSums; ++v) {
                    float sum = acc[m][v] + hd.d * (sums[m][v] + scale * c[1][m][v]);
                    asm volatile("" : "+v"(sum));    // (worked out here: put off behind the branch of `put`, the sums of all groups would stay in registers)
                    acc[m][v] = sum;
                }
        } else {
            // group G: its matrix instructions, the operands of group G + 1, the LDS reads of group G + 2
            v16f c0[MB], c1[MB];
            uint4 first, second, av[2][MB];
            FMT::template operands<0>(hd, FMT::template raw<0>(row, h), first, second);
            typename FMT::Raw ahead = FMT::template raw<1>(row, h);
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                av[0][m] = act_read(0, m);
                av[1][m] = act_read(1, m);
            }
            static_for<0, 16>([&](auto I) {
                constexpr int g = I;
                uint4 next_first, next_second;
                typename FMT::Raw further;
                if constexpr (g < 14) further = FMT::template raw<(g < 14 ? g + 2 : 15)>(row, h);
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    c0[m] = rows_mfma(av[g & 1][m], first, g == 0 ? zero : c0[m]);
                    c1[m] = rows_mfma(av[g & 1][m], second, g == 0 ? zero : c1[m]);
                    if constexpr (g < 14) av[g & 1][m] = act_read(g + 2, m);
                    if constexpr (g < 15)
                        if (m == 0) FMT::template operands<(g < 15 ? g + 1 : 15)>(hd, ahead, next_first, next_second);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (g < 15) { first = next_first; second = next_second; }
                if constexpr (g < 14) ahead = further;
            });
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][v] = __builtin_fmaf(hd.e, c1[m][v], __builtin_fmaf(hd.d, c0[m][v], acc[m][v]));
        }
        __builtin_amdgcn_sched_barrier(0);
        put(near, min(b + 1, b1 - 1));
        wait_vm<kLoads + 1>();
        __syncthreads();                             // the next step's rows are there, this one's have been read
    };
    for (int b = b0; b < b1; b += 2) {
        step(b, 0, set1, set0);
        if (b + 1 < b1) step(b + 1, 1, set0, set1);
    }
    wait_vm<0>();
    // lane: weight row r, matrix rows 8 (v / 4) + 4 h + v % 4
    if (a.partial) {
        float4* out = reinterpret_cast<float4*>(a.partial) + (((static_cast<size_t>(slice) * a.col_tiles + ct) * a.row_tiles + rt) * kWaves + wave) * (MB * 4 * 64) + lane;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                if (t0 + 32 * m + 8 * q4 + 4 * h < a.m_rows)      // (rows past the end are not read again)
                    out[(m * 4 + q4) * 64] = make_float4(acc[m][4 * q4], acc[m][4 * q4 + 1], acc[m][4 * q4 + 2], acc[m][4 * q4 + 3]);
        return;
    }
    const int col = c0 + r;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int v = 0; v < 16; v += TERMS) {
            const int out_row = (t0 + 32 * m + 8 * (v >> 2) + 4 * h + (v & 3)) / TERMS;
            float s = acc[m][v];
            if constexpr (TERMS == 2) s += acc[m][v + 1];
            if (out_row * TERMS < a.m_rows && col < a.n) store_any(a.y, a.y_dtype, static_cast<size_t>(out_row) * a.n + col, s * row_factor(a, out_row));
        }
}

constexpr RowsCost kCost = {3.0, 1.6, 3.0};

template <typename FMT, int MB, int TERMS, int SUMS>
int launch_rows(const RowsArgs& a, hipStream_t stream) {
    static SmemGrant granted;
    constexpr int kWaves = tile_waves(MB);
    const size_t smem = 2 * matrix_rows(MB, SUMS) * 512 + kWaves * slot_bytes<FMT>();
    auto kern = kquant_rows_kernel<FMT, MB, TERMS, SUMS>;
    if (!grant_dynamic_smem(reinterpret_cast<const void*>(kern), smem, granted)) return PLLM_ERR_UNSUPPORTED;
    const int total = a.row_tiles * a.col_tiles * a.slices;
    hipLaunchKernelGGL(kern, dim3((total + 7) / 8 * 8), dim3(64 * kWaves), smem, stream, a);
    if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    if (a.partial) {
        const size_t per_slice = static_cast<size_t>(a.col_tiles) * a.row_tiles * kWaves * MB * 4 * 64;
        hipLaunchKernelGGL((rows_reduce_kernel<MB, TERMS>), dim3(static_cast<unsigned>((per_slice + 255) / 256)), dim3(256), 0, stream, a);
        if (hipGetLastError() != hipSuccess) return PLLM_ERR_LAUNCH;
    }
    return PLLM_OK;
}

template <typename FMT>
int launch_format(const RowsArgs& a, int mb, int terms, hipStream_t stream) {
    constexpr bool kQ6 = std::is_same_v<FMT, RowsQ6K>, kQ2 = std::is_same_v<FMT, RowsQ2K>;
    if constexpr (kQ6)
        if (terms == 1 && a.m_rows <= 8) return launch_rows<FMT, 1, 1, 8>(a, stream);      // (float32 rows are ten matrix rows or more here, IQ4_XS rows nine)
    if constexpr (!kQ2) {
        if (a.m_rows <= 16) return terms == 2 ? launch_rows<FMT, 1, 2, 16>(a, stream) : launch_rows<FMT, 1, 1, 16>(a, stream);
        if (mb == 1) return terms == 2 ? launch_rows<FMT, 1, 2, 32>(a, stream) : launch_rows<FMT, 1, 1, 32>(a, stream);
    } else {
        if (mb == 1) return terms == 2 ? launch_rows<FMT, 1, 2, 0>(a, stream) : launch_rows<FMT, 1, 1, 0>(a, stream);
    }
    constexpr int kSums = kQ6 || kQ2 ? 0 : 64;
    return terms == 2 ? launch_rows<FMT, 2, 2, kSums>(a, stream) : launch_rows<FMT, 2, 1, kSums>(a, stream);
}

}  // namespace

// Up to 64 matrix rows, on matrices of up to 32M weights up to 128 (above, the weights are decoded again per 64 rows; us, bf16 rows, this one / the
// tile kernel, Q6_K: 17408x5120 64 rows 44.6 / 47.2, 100 rows 93.5 / 54.4; 5120x5120 64 rows 25.2 / 26.2, 100 rows 31.9 / 30.7, 128 rows 33.1 / 31.5, 200 rows
// 48.7 / 39.3; the lines were drawn against an earlier tile kernel, and calls within them keep weights that are not rounded).
// (2-byte loads; Q2_K tails and IQ4_XS headers at 4 and 8 bytes; 32-bit offsets inside 32 weight rows and inside 64 activation rows)
bool gemm_kquant_rows_supports(int type_id, int rows, int x_dtype, int n, int bpr, const uint8_t* w) {
    if (type_id != PLLM_TYPE_Q6_K && type_id != PLLM_TYPE_Q2_K && type_id != PLLM_TYPE_IQ4_XS) return false;
    const uintptr_t align = type_id == PLLM_TYPE_Q6_K ? 1u : type_id == PLLM_TYPE_Q2_K ? 3u : 7u;
    const int most = static_cast<long long>(n) * bpr * 256 <= (32ll << 20) ? 128 : 64;
    return rows >= 1 && rows <= (x_dtype == PLLM_F32 ? most / 2 : most) && n >= 1 && (reinterpret_cast<uintptr_t>(w) & align) == 0 &&
           static_cast<long long>(bpr) * 210 * 32 < (1ll << 31) && rows_offsets_fit(bpr);
}

// (the query knows no activation type: room for float32 rows, which are two matrix rows each)
size_t gemm_kquant_rows_workspace_bytes(int type_id, int rows, int n, int bpr) {
    const size_t one = gemm_kquant_rows_supports(type_id, rows, PLLM_F16, n, bpr, nullptr) ? rows_workspace(rows, 1, n, bpr, kCost).bytes : 0;
    const size_t two = gemm_kquant_rows_supports(type_id, rows, PLLM_F32, n, bpr, nullptr) ? rows_workspace(rows, 2, n, bpr, kCost).bytes : 0;
    return std::max(one, two);
}

int gemm_kquant_rows(const void* x, int x_dtype, const uint8_t* w, int type_id, void* y, int y_dtype, int rows, int k, int n, int bpr, void* workspace,
                     size_t workspace_bytes, hipStream_t stream) {
    const int terms = x_dtype == PLLM_F32 ? 2 : 1;
    const RowsWorkspace ws = rows_workspace(rows, terms, n, bpr, kCost);
    if (!workspace || workspace_bytes < ws.bytes) return PLLM_ERR_WORKSPACE;
    unsigned char* base = static_cast<unsigned char*>(workspace);
    const RowsPlan p = plan_rows(rows * terms, n, bpr, kCost);
    RowsArgs a{};
    a.rows = reinterpret_cast<const _Float16*>(base);
    a.unscale = reinterpret_cast<const float*>(base + ws.unscale);
    a.w = w;
    a.y = y;
    a.partial = p.slices > 1 ? reinterpret_cast<float*>(base + ws.partial) : nullptr;
    a.y_dtype = y_dtype;
    a.m_rows = rows * terms;
    a.n = n;
    a.blocks = bpr;
    a.kp = bpr * 256;
    a.row_tiles = p.row_tiles;
    a.col_tiles = p.col_tiles;
    a.slices = p.slices;
    a.steps = bpr / p.slices;
    a.steps_more = bpr % p.slices;
    // (the staging of the tile kernel puts its scales where these lie, for one term)
    if (rows_as_held(x, x_dtype, k, a.kp)) {
        a.rows = static_cast<const _Float16*>(x);
        a.unscale = nullptr;
    } else {
        const int st = terms == 1 ? gemm_f16_stage_rows(x, x_dtype, nullptr, rows, k, bpr, base, stream)
                                  : half_rows_stage(x, x_dtype, rows, k, a.kp, base, reinterpret_cast<float*>(base + ws.unscale), stream);
        if (st != PLLM_OK) return st;
    }
    switch (type_id) {
        case PLLM_TYPE_Q6_K: return launch_format<RowsQ6K>(a, p.mb, terms, stream);
        case PLLM_TYPE_Q2_K: return launch_format<RowsQ2K>(a, p.mb, terms, stream);
        case PLLM_TYPE_IQ4_XS: return launch_format<RowsIQ4XS>(a, p.mb, terms, stream);
        default: return PLLM_ERR_UNSUPPORTED;
    }
}

}  // namespace pllm
