// Block formats of the prompt tile kernel (gemm_tile.h): how a wave gets from raw blocks to half-precision operands of
// v_mfma_f32_32x32x16_f16, in registers.
//
// Lane (l, hs) = (lane % 32, lane / 32) owns weight row l of a 32-row block.  A super-block is four pairs p of 64 weights, a pair two
// half steps e of 32; of a half step the lane decodes the 16 weights [32 (2 p + e) + 16 hs, + 16), eight per matrix instruction, as
// eight dwords ("pairs" g = 0 .. 7 of two weights).  A format provides
//   Head / load_head          what a whole block needs (scales), fetched one block ahead;  Expanded / expand: the same, unpacked
//   Part / load_part          the codes of kPairs consecutive pairs (kPairs = 1: a part is a pair, 2: half a block)
//   hold(Part)                a use of the registers, so that the wait for them stands where it is called
//   Scale / scale             the factors of a half step's 16 weights
//   Look / look               codebook entries of eight weights, read from LDS ahead of their use (kLooks; others: nothing)
//   pair                      two weights: the value in float32 exactly as the block decoders state it, rounded once to half precision
//   kTableBytes / stage_table the codebook in LDS
#pragma once

#include "block_dot4.h"
#include "pllm_internal.h"

namespace pllm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr int kTileThreads = 256;

// two float32 values, each rounded to nearest half precision, in one instruction.  (Stated as two conversions the compiler folds the
// multiplication in front of each into v_fma_mixlo / mixhi_f16, which write half a register and take 8.8 cycles where every other
// vector instruction here takes 5: 17.6 cycles per pair of weights against 15.)
__device__ __forceinline__ uint32_t pack_halves(float lo, float hi) {
    uint32_t o;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(o) : "v"(lo), "v"(hi));
    return o;
}
struct Affine { float scale, minus; };                    // scale times 2^24
// Codes in bytes 2 g', 2 g' + 1 of a word (g' = HI) -> half(scale * code - minus).  A code byte in the low bits of a half is the
// subnormal code * 2^-24, which the mixed-precision multiply takes as it is: the product with scale * 2^24 has the bits of
// scale * code, and no conversion of the code is needed.
template <int HI>
__device__ __forceinline__ uint32_t affine_pair(uint32_t codes, const Affine& s) {
    const half2v v = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0u, codes, HI ? 0x0c030c02u : 0x0c010c00u));
    return pack_halves(__builtin_fmaf(static_cast<float>(v.x), s.scale, -s.minus), __builtin_fmaf(static_cast<float>(v.y), s.scale, -s.minus));
}
// two halves with their sign bits flipped by `flip`, times a float32 scale
__device__ __forceinline__ uint32_t scaled_pair(uint32_t bits, uint32_t flip, float scale) {
    const half2v v = __builtin_bit_cast(half2v, bits ^ flip);
    return pack_halves(static_cast<float>(v.x) * scale, static_cast<float>(v.y) * scale);
}
// Codes as the load instruction returned them, in one piece.  (As four members the compiler carried them around the loop in other registers than
// they were loaded to, and the copies at the end of every super-block waited for all loads on their way: FP8 17408x5120 at 512 rows 115 -> 108
// us, Q6_K 16384x5120 at 1024 rows 187 -> 182, Q5_K 5120x17408 at 1999 rows 369 -> 363.)
typedef uint32_t words4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ words4 words_of(const uint4& v) { return __builtin_bit_cast(words4, v); }
__device__ __forceinline__ uint32_t word_of(const words4& v, int j) { return v[j]; }
__device__ __forceinline__ void hold_registers(words4& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ uint32_t word_of(const uint4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }
__device__ __forceinline__ void hold_registers(uint32_t& v) { asm volatile("" : "+v"(v)); }
constexpr float kTwo24 = 16777216.0f;

struct __attribute__((packed, aligned(2))) UnalignedWord { uint32_t v; };
__device__ __forceinline__ uint32_t word_at(const uint8_t* p) { return reinterpret_cast<const UnalignedWord*>(p)->v; }

struct NoLook {};
struct NoTable {
    static constexpr int kTableBytes = 0;
    static constexpr bool kLooks = false;
    typedef NoLook Look;
    static __device__ __forceinline__ void stage_table(unsigned char*) {}
};

// Six-bit scales and minima of Q4_K / Q5_K: byte j of s0 (m0) belongs to group j, of s1 (m1) to group 4 + j.
struct K4Expanded { uint32_t s0, s1, m0, m1; float d, dmin; };
__device__ __forceinline__ void k4_expand(const uint4& hdr, K4Expanded& k) {
    k.s0 = hdr.y & 0x3f3f3f3fu;
    k.m0 = hdr.z & 0x3f3f3f3fu;
    k.s1 = (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u);
    k.m1 = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
    k.d = f16_bits_to_float(hdr.x & 0xffffu) * kTwo24;
    k.dmin = f16_bits_to_float(hdr.x >> 16);
}
__device__ __forceinline__ Affine k4_scale(const K4Expanded& k, int p, int e) {
    const int at = 8 * (2 * (p & 1) + e);
    return {k.d * static_cast<float>(((p < 2 ? k.s0 : k.s1) >> at) & 0xffu), k.dmin * static_cast<float>(((p < 2 ? k.m0 : k.m1) >> at) & 0xffu)};
}

struct TQ4K : NoTable {
    static constexpr int kBlockBytes = 144, kPairs = 1;
    struct Head { uint4 hdr; };
    typedef K4Expanded Expanded;
    typedef Affine Scale;
    struct Part { words4 q; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.hdr = *reinterpret_cast<const uint4*>(blk); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { k4_expand(r.hdr, x); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        r.q = *reinterpret_cast<const words4*>(blk + 16 + 32 * p + 16 * hs);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int e, int) { return k4_scale(x, p, e); }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part& r, const Look&, const Scale& s, int, int e, int) {
        return affine_pair<G & 1>((word_of(r.q, G >> 1) >> (4 * e)) & 0x0f0f0f0fu, s);
    }
};

struct TQ5K : NoTable {
    static constexpr int kBlockBytes = 176, kPairs = 1;
    struct Head { uint4 hdr, qh; };
    struct Expanded { K4Expanded k; uint4 qh; };
    typedef Affine Scale;
    struct Part { words4 q; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int hs, const float*, int) {
        r.hdr = *reinterpret_cast<const uint4*>(blk);
        r.qh = *reinterpret_cast<const uint4*>(blk + 16 + 16 * hs);
    }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { k4_expand(r.hdr, x.k); x.qh = r.qh; }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        r.q = *reinterpret_cast<const words4*>(blk + 48 + 32 * p + 16 * hs);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int e, int) { return k4_scale(x.k, p, e); }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded& x, const Part& r, const Look&, const Scale& s, int p, int e, int) {
        const int bit = 2 * p + e;                         // the group's bit of the high-bit bytes
        const uint32_t h = word_of(x.qh, G >> 1), top = bit <= 4 ? h << (4 - bit) : h >> (bit - 4);
        return affine_pair<G & 1>(((word_of(r.q, G >> 1) >> (4 * e)) & 0x0f0f0f0fu) | (top & 0x10101010u), s);
    }
};

// Q2_K: 84 B = scales(16) qs(64) d(2) dmin(2).  Half step c = 2 p + e: byte qs[32 (c / 4) + l] >> 2 (c % 4), so pairs 0, 1 and 2, 3 share
// their bytes; the lane's 16 weights are group 2 c + hs with scale byte scales[2 c + hs] (low nibble scale, high nibble min).
struct TQ2K : NoTable {
    static constexpr int kBlockBytes = 84, kPairs = 2;
    struct Head { uint4 sc; uint32_t dd; };
    struct Expanded { uint4 sc; float d, dmin; };
    typedef Affine Scale;
    struct Part { words4 q; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(blk);           // blocks are 4-byte aligned
        r.sc = make_uint4(w[0], w[1], w[2], w[3]);
        r.dd = w[20];
    }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) {
        x.sc = r.sc;
        x.d = f16_bits_to_float(r.dd & 0xffffu) * kTwo24;
        x.dmin = f16_bits_to_float(r.dd >> 16);
    }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(blk) + 4 + 8 * (p >> 1) + 4 * hs;
        r.q = words4{q[0], q[1], q[2], q[3]};
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int e, int hs) {
        const int c = 2 * p + e;                           // group 2 c + hs: byte 2 (c % 2) + hs of word c / 2
        const uint32_t sb = word_of(x.sc, c >> 1) >> (16 * (c & 1) + 8 * hs);
        return {x.d * static_cast<float>(sb & 15u), x.dmin * static_cast<float>((sb >> 4) & 15u)};
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part& r, const Look&, const Scale& s, int p, int e, int) {
        return affine_pair<G & 1>((word_of(r.q, G >> 1) >> (2 * ((2 * p + e) & 3))) & 0x03030303u, s);
    }
};

// Q6_K: 210 B = ql(128) qh(64) scales int8(16) d(2); weight 128 half + 32 j + l takes nibble j / 2 of ql[64 half + 32 (j % 2) + l], bit
// pair j of qh[32 half + l] and scale 8 half + 2 j + l / 16; w = d * scale * (q - 32).  Here half = p / 2, j = 2 (p % 2) + e, l = 16 hs + ...
// Blocks are only 2-byte aligned.
struct TQ6K : NoTable {
    static constexpr int kBlockBytes = 210, kPairs = 2;
    struct Head { uint32_t d; };
    struct Expanded { float d; };
    typedef Affine Scale;
    struct Part { words4 qa, qb, qh; uint32_t s0, s1; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.d = *reinterpret_cast<const uint16_t*>(blk + 208); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x.d = f16_bits_to_float(r.d); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        const int half = p >> 1;
        r.qa = words_of(load16_a2(blk + 64 * half + 16 * hs));
        r.qb = words_of(load16_a2(blk + 64 * half + 32 + 16 * hs));
        r.qh = words_of(load16_a2(blk + 128 + 32 * half + 16 * hs));
        r.s0 = word_at(blk + 192 + 8 * half);
        r.s1 = word_at(blk + 196 + 8 * half);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.qa); hold_registers(r.qb); hold_registers(r.qh); hold_registers(r.s0); hold_registers(r.s1); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part& r, int p, int e, int hs) {
        const float s = x.d * static_cast<float>(static_cast<int8_t>(((p & 1) ? r.s1 : r.s0) >> (16 * e + 8 * hs)));
        return {s * kTwo24, 32.0f * s};
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part& r, const Look&, const Scale& s, int p, int e, int) {
        const uint32_t lo = (word_of(e ? r.qb : r.qa, G >> 1) >> (4 * (p & 1))) & 0x0f0f0f0fu;
        const int j = 2 * (p & 1) + e;                     // bit pair j to bits 4, 5
        const uint32_t h = word_of(r.qh, G >> 1), top = j <= 2 ? h << (4 - 2 * j) : h >> 2;
        return affine_pair<G & 1>(lo | (top & 0x30303030u), s);
    }
};

// IQ4_XS: 136 B = d(2) scales_h(2) scales_l(4) qs(128); group g = 2 p + e of 32 weights: bytes qs[16 g, +16), low nibbles = its first
// 16 weights (hs = 0), high nibbles the others; w = d * (ls - 32) * kvalues[code].  The 16-entry table sits in four constants, biased
// by 128 so that the codes stay unsigned bytes; three byte permutes pick four values.
struct TIQ4XS : NoTable {
    static constexpr int kBlockBytes = 136, kPairs = 1;
    struct Head { uint2 hdr; };
    struct Expanded { uint2 hdr; float d; };
    typedef Affine Scale;
    struct Part { words4 q0, q1; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.hdr = *reinterpret_cast<const uint2*>(blk); }   // 8-byte aligned
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x.hdr = r.hdr; x.d = f16_bits_to_float(r.hdr.x & 0xffffu); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int) {
        r.q0 = words_of(load16_a2(blk + 8 + 32 * p));
        r.q1 = words_of(load16_a2(blk + 24 + 32 * p));
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q0); hold_registers(r.q1); }
    static __device__ __forceinline__ uint32_t biased4(uint32_t codes) {     // kvalues[code] + 128, four at a time
        const uint32_t low3 = codes & 0x07070707u;
        const uint32_t lower = __builtin_amdgcn_perm(0x766A5D4Fu, 0x3F2D1801u, low3);   // 1 24 45 63 | 79 93 106 118
        const uint32_t upper = __builtin_amdgcn_perm(0xF1D9C5B5u, 0xA6998D81u, low3);   // 129 141 153 166 | 181 197 217 241
        return __builtin_amdgcn_perm(upper, lower, ((codes >> 1) & 0x04040404u) | 0x03020100u);
    }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int e, int) {
        const int ls = static_cast<int>(((x.hdr.y >> (8 * p + 4 * e)) & 15u) | (((x.hdr.x >> (16 + 2 * (2 * p + e))) & 3u) << 4)) - 32;
        const float s = x.d * static_cast<float>(ls);
        return {s * kTwo24, 128.0f * s};
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part& r, const Look&, const Scale& s, int, int e, int hs) {
        return affine_pair<G & 1>(biased4((word_of(e ? r.q1 : r.q0, G >> 1) >> (4 * hs)) & 0x0f0f0f0fu), s);
    }
};

// FP8 E4M3 (OCP) codes, one byte per weight, rows of k bytes with k a multiple of 256; a "block" is 256 consecutive codes of a row.
// The float32 scale of the 128 x 128 block is folded into the weight: half(f32(code) * scale).
struct TFP8 : NoTable {
    static constexpr int kBlockBytes = 256, kPairs = 1;
    struct Head { float s0, s1; };
    typedef Head Expanded;
    typedef float Scale;
    struct Part { words4 q0, q1; };
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t*, int, const float* srow, int b) {
        r.s0 = srow[2 * b];
        r.s1 = srow[2 * b + 1];
    }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x = r; }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        r.q0 = *reinterpret_cast<const words4*>(blk + 64 * p + 16 * hs);
        r.q1 = *reinterpret_cast<const words4*>(blk + 64 * p + 32 + 16 * hs);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q0); hold_registers(r.q1); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int, int) { return p < 2 ? x.s0 : x.s1; }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part& r, const Look&, const Scale& s, int, int e, int) {
        typedef float v2f __attribute__((ext_vector_type(2)));
        const v2f v = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word_of(e ? r.q1 : r.q0, G >> 1)), (G & 1) != 0);
        return pack_halves(v.x * s, v.y * s);
    }
};

// Sign patterns of the IQ2 / IQ3 formats: seven bits plus their parity, as eight halves that hold the sign bit or nothing.  (Tables are staged
// by entries of 16 bytes: value by value a workgroup spent 1.5 us on them.)
__device__ __forceinline__ void stage_signs(unsigned char* lds) {
    for (int i = threadIdx.x; i < 128; i += kTileThreads) {
        const uint32_t s8 = static_cast<uint32_t>(i) | ((__popc(static_cast<uint32_t>(i)) & 1u) << 7);
        auto two = [&](int at) { return (((s8 >> at) & 1u) << 15) | (((s8 >> (at + 1)) & 1u) << 31); };
        reinterpret_cast<uint4*>(lds)[i] = make_uint4(two(0), two(2), two(4), two(6));
    }
}
// four magnitudes in bytes -> four halves
__device__ __forceinline__ uint2 halves_of_bytes(uint32_t v) {
    auto half_bits = [](uint32_t b) { return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(b & 0xffu)))); };
    return make_uint2(half_bits(v) | (half_bits(v >> 8) << 16), half_bits(v >> 16) | (half_bits(v >> 24) << 16));
}
template <int ENTRIES>
__device__ __forceinline__ void stage_grid8(unsigned char* lds, const uint64_t* grid) {
    for (int i = threadIdx.x; i < ENTRIES; i += kTileThreads) {
        const uint64_t g = grid[i];
        const uint2 lo = halves_of_bytes(static_cast<uint32_t>(g)), hi = halves_of_bytes(static_cast<uint32_t>(g >> 32));
        reinterpret_cast<uint4*>(lds)[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
}
struct GridLook { uint4 m, f; };                           // magnitudes and sign bits of eight weights, as halves

// IQ2_XXS: 66 B = d(2) + 8 sub-blocks of 8 B (four grid ids, then a u32: four 7-bit sign indices and a 4-bit scale); the lane takes grid
// entries 2 hs and 2 hs + 1 of its sub-block.  w = d (2 s + 1) / 8 * magnitude, negated where the sign pattern says so.  LDS: the
// 256 x 8 magnitudes (8, 25 and 43 are exact) and the 128 x 8 sign bits.
struct TIQ2XXS {
    static constexpr int kBlockBytes = 66, kPairs = 1, kTableBytes = 4096 + 2048;
    static constexpr bool kLooks = true;
    struct Head { uint32_t d; };
    struct Expanded { float d; };
    typedef float Scale;
    typedef GridLook Look;
    struct Part { words4 q; };
    static __device__ __forceinline__ void stage_table(unsigned char* lds) {
        stage_grid8<256>(lds, PLLM_IQ2XXS_GRID);
        stage_signs(lds + 4096);
    }
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.d = *reinterpret_cast<const uint16_t*>(blk); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x.d = 0.125f * f16_bits_to_float(r.d); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int) { r.q = words_of(load16_a2(blk + 2 + 16 * p)); }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part& r, int, int e, int) {
        return x.d * static_cast<float>(2 * ((e ? r.q.w : r.q.y) >> 28) + 1);
    }
    static __device__ __forceinline__ void look(Look& k, const Part& r, int, int e, int hs, int u, const unsigned char* table) {
        const uint32_t ids = e ? r.q.z : r.q.x, aux = e ? r.q.w : r.q.y;
        k.m = *reinterpret_cast<const uint4*>(table + 16 * ((ids >> (16 * hs + 8 * u)) & 0xffu));
        k.f = *reinterpret_cast<const uint4*>(table + 4096 + 16 * ((aux >> (14 * hs + 7 * u)) & 127u));
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part&, const Look& k, const Scale& s, int, int, int) {
        return scaled_pair(word_of(k.m, G & 3), word_of(k.f, G & 3), s);
    }
};

// IQ2_XS: 74 B = d(2) qs u16[32] scales(8).  Entry (8 weights) = 9-bit grid id + 7-bit sign index; two 4-bit scales per 32
// weights (low nibble: first 16).  The lane's 16 weights are entries 8 p + 4 e + 2 hs and the next one.  LDS tables as for
// IQ2_XXS with 512 grid entries.
struct TIQ2XS {
    static constexpr int kBlockBytes = 74, kPairs = 1, kTableBytes = 8192 + 2048;
    static constexpr bool kLooks = true;
    struct Head { uint32_t d; };
    struct Expanded { float d; };
    typedef float Scale;
    typedef GridLook Look;
    struct Part { uint32_t q0, q1, sc; };
    static __device__ __forceinline__ void stage_table(unsigned char* lds) {
        stage_grid8<512>(lds, PLLM_IQ2XS_GRID);
        stage_signs(lds + 8192);
    }
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.d = *reinterpret_cast<const uint16_t*>(blk); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x.d = 0.125f * f16_bits_to_float(r.d); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        r.q0 = word_at(blk + 2 + 16 * p + 4 * hs);
        r.q1 = word_at(blk + 10 + 16 * p + 4 * hs);
        r.sc = *reinterpret_cast<const uint16_t*>(blk + 66 + 2 * p);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.q0); hold_registers(r.q1); hold_registers(r.sc); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part& r, int, int e, int hs) {
        return x.d * static_cast<float>(2 * ((r.sc >> (8 * e + 4 * hs)) & 15u) + 1);
    }
    static __device__ __forceinline__ void look(Look& k, const Part& r, int, int e, int, int u, const unsigned char* table) {
        const uint32_t q16 = ((e ? r.q1 : r.q0) >> (16 * u)) & 0xffffu;
        k.m = *reinterpret_cast<const uint4*>(table + 16 * (q16 & 511u));
        k.f = *reinterpret_cast<const uint4*>(table + 8192 + 16 * (q16 >> 9));
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part&, const Look& k, const Scale& s, int, int, int) {
        return scaled_pair(word_of(k.m, G & 3), word_of(k.f, G & 3), s);
    }
};

// IQ3_XXS: 98 B = d(2) grid ids(64) aux u32[8].  An id gives four weights; aux of a 32-weight sub-block = four 7-bit sign indices
// (one per 8 weights) and a 4-bit scale.  The lane's 16 weights are ids 8 (2 p + e) + 4 hs .. + 3 with sign indices 2 hs, 2 hs + 1.
// LDS tables: 256 x 4 magnitudes as halves, then the 128 x 8 sign bits.
struct TIQ3XXS {
    static constexpr int kBlockBytes = 98, kPairs = 1, kTableBytes = 2048 + 2048;
    static constexpr bool kLooks = true;
    struct Head { uint32_t d; };
    struct Expanded { float d; };
    typedef float Scale;
    typedef GridLook Look;
    struct Part { uint32_t i0, i1, a0, a1; };
    static __device__ __forceinline__ void stage_table(unsigned char* lds) {
        for (int i = threadIdx.x; i < 256; i += kTileThreads) reinterpret_cast<uint2*>(lds)[i] = halves_of_bytes(PLLM_IQ3XXS_GRID[i]);
        stage_signs(lds + 2048);
    }
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.d = *reinterpret_cast<const uint16_t*>(blk); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) { x.d = 0.25f * f16_bits_to_float(r.d); }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int hs) {
        r.i0 = word_at(blk + 2 + 16 * p + 4 * hs);
        r.i1 = word_at(blk + 10 + 16 * p + 4 * hs);
        r.a0 = word_at(blk + 66 + 8 * p);
        r.a1 = word_at(blk + 70 + 8 * p);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.i0); hold_registers(r.i1); hold_registers(r.a0); hold_registers(r.a1); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part& r, int, int e, int) {
        return x.d * static_cast<float>(2 * ((e ? r.a1 : r.a0) >> 28) + 1);
    }
    static __device__ __forceinline__ void look(Look& k, const Part& r, int, int e, int hs, int u, const unsigned char* table) {
        const uint32_t ids = (e ? r.i1 : r.i0) >> (16 * u), aux = e ? r.a1 : r.a0;
        const uint2 lo = *reinterpret_cast<const uint2*>(table + 8 * (ids & 0xffu)), hi = *reinterpret_cast<const uint2*>(table + 8 * ((ids >> 8) & 0xffu));
        k.m = make_uint4(lo.x, lo.y, hi.x, hi.y);
        k.f = *reinterpret_cast<const uint4*>(table + 2048 + 16 * ((aux >> (14 * hs + 7 * u)) & 127u));
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part&, const Look& k, const Scale& s, int, int, int) {
        return scaled_pair(word_of(k.m, G & 3), word_of(k.f, G & 3), s);
    }
};

// IQ1_M: 56 B = qs(32) qh(16) scales(8).  One codebook index per 8 weights (qs byte plus the low three bits of its qh nibble; bit 3 of
// the nibble picks delta = -+0.125); sixteen 3-bit scales, one per 16 weights, in the low 12 bits of four u16 words whose top nibbles
// spell the fp16 block scale.  The lane's 16 weights are entries 8 p + 4 e + 2 hs and the next one, scale group 4 p + 2 e + hs.
// LDS: the 2048 codebook entries as bytes 8 c + 8, c in -1, 0, 1; a lookup adds 2 to each where the delta is positive, so that
// w = d (2 s + 1) (c + delta) = d (2 s + 1) / 8 * (byte - 9) with a byte that is never negative.
struct TIQ1M {
    static constexpr int kBlockBytes = 56, kPairs = 1, kTableBytes = 2048 * 8;
    static constexpr bool kLooks = true;
    struct Head { uint2 sc; };
    struct Expanded { uint2 sc; float d; };
    typedef Affine Scale;
    struct Look { uint2 c; };
    struct Part { uint2 qs; uint32_t qh; };
    static __device__ __forceinline__ void stage_table(unsigned char* lds) {
        uint2* t = reinterpret_cast<uint2*>(lds);
        for (int i = threadIdx.x; i < 2048; i += kTileThreads) {
            const uint32_t v = PLLM_IQ1_GRID_PACKED[i];    // element k in bits [2k, 2k+1], c + 1
            auto four = [](uint32_t b) { return ((b & 3u) | ((b & 0xcu) << 6) | ((b & 0x30u) << 12) | ((b & 0xc0u) << 18)) << 3; };
            t[i] = make_uint2(four(v), four(v >> 8));
        }
    }
    static __device__ __forceinline__ void load_head(Head& r, const uint8_t* blk, int, const float*, int) { r.sc = *reinterpret_cast<const uint2*>(blk + 48); }
    static __device__ __forceinline__ void expand(const Head& r, Expanded& x) {
        x.sc = r.sc;
        const uint32_t bits = ((r.sc.x >> 12) & 0xfu) | ((r.sc.x >> 24) & 0xf0u) | ((r.sc.y >> 4) & 0xf00u) | ((r.sc.y >> 16) & 0xf000u);
        x.d = 0.125f * f16_bits_to_float(bits);
    }
    static __device__ __forceinline__ void load_part(Part& r, const uint8_t* blk, int p, int) {
        r.qs = *reinterpret_cast<const uint2*>(blk + 8 * p);                  // blocks are 8-byte aligned
        r.qh = *reinterpret_cast<const uint32_t*>(blk + 32 + 4 * p);
    }
    static __device__ __forceinline__ void hold(Part& r) { hold_registers(r.qs.x); hold_registers(r.qs.y); hold_registers(r.qh); }
    static __device__ __forceinline__ Scale scale(const Expanded& x, const Part&, int p, int e, int hs) {
        const uint32_t word = (p < 2 ? x.sc.x : x.sc.y) >> (16 * (p & 1) + 6 * e + 3 * hs);      // group 4 p + 2 e + hs
        const float s = x.d * static_cast<float>(2 * (word & 7u) + 1);
        return {s * kTwo24, 9.0f * s};
    }
    static __device__ __forceinline__ void look(Look& k, const Part& r, int, int e, int hs, int u, const unsigned char* table) {
        const uint32_t qb = ((e ? r.qs.y : r.qs.x) >> (16 * hs + 8 * u)) & 0xffu, nib = r.qh >> (16 * e + 8 * hs + 4 * u);
        const uint2 c = *reinterpret_cast<const uint2*>(table + 8 * (qb | ((nib & 7u) << 8)));
        const uint32_t delta = (nib & 8u) ? 0u : 0x02020202u;
        k.c = make_uint2(c.x + delta, c.y + delta);
    }
    template <int G>
    static __device__ __forceinline__ uint32_t pair(const Expanded&, const Part&, const Look& k, const Scale& s, int, int, int) {
        return affine_pair<G & 1>((G & 2) ? k.c.y : k.c.x, s);
    }
};

}  // namespace pllm
