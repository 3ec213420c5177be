// y[T, N] = x[T, K] . dequant(W)[N, K]^T over raw Q8_0 blocks (fp16 scale + 32 int8 codes), several activation rows, on f16 MFMA.
//
// Codes are exact in half precision and so are bf16 / fp16 activations scaled by a power of two per row (fp16 rows of whole steps go in as the caller holds them, float32 rows as two
// half-precision terms = two matrix rows): a block's sum of products comes out of the matrix cores in float32 without any operand
// rounding, and the block scale goes on as it joins the total.
//
// A workgroup owns 64 matrix rows and 256 weight rows (eight waves), or 32 and 128 (four waves), over a slice of K.  Every wave owns 32
// of the weight rows: their blocks come 256 columns (eight blocks) ahead into the wave's own LDS slot, by direct-to-LDS loads of whole
// 16-byte pieces where rows are whole steps on aligned bases (with registers in between 29.2 us where these take 22.4: a 16-byte load
// at a 2-byte boundary costs the memory path more), are read from there in the order of the matrix operand (lane (n, h) = row n,
// codes 16 h .. 16 h + 15 of a block) and unpacked in registers: bytes biased by 128 into the mantissa of 1024, minus 1152.
// v_mfma_f32_32x32x16_f16, two per block and 32 rows, then one fused multiply-add per sum.  Activation rows come to LDS by
// direct-to-LDS loads, 256 columns at a time, double-buffered, 16-byte piece p of row r at position p ^ (r % 32).  Slices along K fill
// the machine where there are few tiles; their sums leave in lane order and a second kernel adds them in slice order.
//
// Bound, up to 32 rows: weights from memory (17408x5120 at 4 rows 25.6 us = 3.7 TB/s; 32 rows and fewer run four waves per workgroup,
// two workgroups per compute unit); above: the vector ALU, which unpacks the weights again per 64 matrix rows and scales every block's sums,
// and the turns between it and the other units (4096x4096 at 203 rows: 7200 cycles a step, 1150 of them to take the codes from the slot, where the matrix
// cores need 2050).  Codes are taken in whole 16-byte pieces, which 32 rows read without bank conflicts (as the compiler's single words, 16 banks for all:
// 1400 cycles), and scaled with float32 factors: 17408x5120 at 203 rows 132.7 -> 126.9 us, 512 rows 237.6 -> 225.0.  4096x4096 at 203 rows takes 28 - 30 us (row staging 3.7, this kernel 21.9, sums of the slices 5.1) against 970 us on the kernels that
// run once per row.
#include "rows_tiles.h"

namespace pllm {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kOctet = 256;                          // columns per step: eight blocks
constexpr int kSlotCodes = kWaveCols * kOctet, kSlotBytes = kSlotCodes + kWaveCols * 8 * 4;      // a wave's codes and block scales of a step

constexpr RowsCost kCost = {3.0, 2.4, 3.4};
// eight int8 codes -> eight halves
__device__ __forceinline__ v8h unpack8(uint32_t lo, uint32_t hi) {
    const v2h bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
    auto pair = [&](uint32_t w, uint32_t sel) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, w, sel)) + bias); };
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    return __builtin_bit_cast(v8h, make_uint4(pair(lo, 0x04010400u), pair(lo, 0x04030402u), pair(hi, 0x04010400u), pair(hi, 0x04030402u)));
}

template <int MB, int TERMS, bool ALIGNED>
__global__ __launch_bounds__(64 * tile_waves(MB), 2) void q8_rows_kernel(RowsArgs a) {
    extern __shared__ __align__(1024) unsigned char smem[];
    constexpr int kWaves = tile_waves(MB), kCols = kWaves * kWaveCols;
    constexpr int kRows = 32 * MB, kChunk = kRows * 512, kDma = kRows / 2 / kWaves;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroups of one XCD (number modulo 8) take neighbouring tiles, those that share weights first
    const int total = a.row_tiles * a.col_tiles * a.slices, per = (total + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per || tile >= total) return;
    const int rt = tile % a.row_tiles, slice = tile / a.row_tiles % a.slices, ct = tile / (a.row_tiles * a.slices);
    // (the first steps_more slices take one step more)
    const int o0 = slice * a.steps + min(slice, a.steps_more), o1 = o0 + a.steps + (slice < a.steps_more ? 1 : 0);
    const int t0 = rt * kRows, c0 = ct * kCols + wave * kWaveCols;

    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte_ptr)smem));
    unsigned char* slot = smem + 2 * kChunk + wave * kSlotBytes;
    float* slot_d = reinterpret_cast<float*>(slot + kSlotCodes);
    const unsigned char* xb = reinterpret_cast<const unsigned char*>(a.rows) + static_cast<size_t>(t0) * 2 * a.kp;
    uint32_t xoff[kDma];
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
        const int row = 2 * (wave * kDma + i) + h;
        xoff[i] = static_cast<uint32_t>(min(row, a.m_rows - 1 - t0)) * (2u * a.kp) + 16u * (r ^ (row & 31));
    }
    auto dma = [&](int o, int buf) {
#pragma unroll
        for (int i = 0; i < kDma; ++i) lds_dma16_at(xb + 512 * static_cast<size_t>(o), xoff[i], lds0 + buf * kChunk + (wave * kDma + i) * 1024);
    };
    const size_t row_bytes = static_cast<size_t>(a.blocks) * 34;
    const uint8_t* wtile = a.w + static_cast<size_t>(min(c0, a.n - 1)) * row_bytes;
    const int last_row = max(min(a.n - 1 - c0, kWaveCols - 1), 0);                // (rows past the end: the last one again, dropped at the store)
    uint4 codes[8];                                  // of the lane's row and half, blocks 0 .. 7 of the step
    float scales[8];
    // ALIGNED (whole steps, 16-byte aligned rows): the 272 bytes of a row's step go to the slot by direct-to-LDS loads, 17 pieces per row
    // end to end, and from there to the registers when the step begins; the next step's follow at once.
    constexpr int kMoves = (kWaveCols * 17 + 63) / 64;
    uint32_t woff[kMoves];
    // otherwise: instruction i brings the codes of rows 4 i + lane / 16, block (lane % 16) / 2 and half lane % 2 of it, or the scales
    // of rows 8 i + lane / 8, block lane % 8, which turn in the slot (blocks past the row's end: its last one again, against zero activations)
    uint32_t wrow[8], drow[4];
    uint4 fetched[8];
    uint32_t fetched_d[4];
    if constexpr (ALIGNED) {
#pragma unroll
        for (int i = 0; i < kMoves; ++i) {
            const int piece = min(64 * i + lane, kWaveCols * 17 - 1), row = piece / 17;
            woff[i] = static_cast<uint32_t>(min(row, last_row) * row_bytes) + 16u * (piece - 17 * row);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) wrow[i] = static_cast<uint32_t>(min(4 * i + (lane >> 4), last_row) * row_bytes) + 2 + 16 * (lane & 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) drow[i] = static_cast<uint32_t>(min(8 * i + (lane >> 3), last_row) * row_bytes);
    }
    auto fetch = [&](int o) {
        if constexpr (ALIGNED) {
            const uint32_t base = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(lds0 + 2 * kChunk + wave * kSlotBytes)));
#pragma unroll
            for (int i = 0; i < kMoves; ++i)
                if (i + 1 < kMoves || 64 * i + lane < kWaveCols * 17) lds_dma16_at(wtile + 272 * static_cast<size_t>(o), woff[i], base + 1024 * i);
        } else {
            const uint32_t cb = 34u * min(8 * o + ((lane >> 1) & 7), a.blocks - 1), db = 34u * min(8 * o + (lane & 7), a.blocks - 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) fetched[i] = load16_a2(wtile + (wrow[i] + cb));
#pragma unroll
            for (int i = 0; i < 4; ++i) fetched_d[i] = *reinterpret_cast<const uint16_t*>(wtile + (drow[i] + db));
        }
    };
    auto take = [&]() {                              // the step's codes and scales from the slot to the registers
        if constexpr (ALIGNED) {
            // block g's codes of half h lie 2 g + 2 bytes into piece 2 g + h and go on in the next one
            const uint4* row = reinterpret_cast<const uint4*>(slot + r * 272 + 16 * h);
            uint4 piece[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) piece[i] = row[i];
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(piece[i].x), "+v"(piece[i].y), "+v"(piece[i].z), "+v"(piece[i].w));      // (whole pieces: 32 rows' single words share 16 banks)
            static_for<0, 8>([&](auto G) {
                constexpr int g = G, q = (g + 1) / 2;
                const uint4 p0 = piece[2 * g], p1 = piece[2 * g + 1];
                const uint32_t w[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
                if constexpr (g & 1) {
                    codes[g] = make_uint4(w[q], w[q + 1], w[q + 2], w[q + 3]);
                } else {
                    codes[g] = make_uint4(__builtin_amdgcn_alignbit(w[q + 1], w[q], 16), __builtin_amdgcn_alignbit(w[q + 2], w[q + 1], 16), __builtin_amdgcn_alignbit(w[q + 3], w[q + 2], 16),
                                          __builtin_amdgcn_alignbit(w[q + 4], w[q + 3], 16));
                }
                scales[g] = f16_bits_to_float(*reinterpret_cast<const uint16_t*>(slot + r * 272 + 34 * g));
                asm("" : "+v"(scales[g]));           // (a float32 factor: as a half inside the multiply-adds it takes twice the time)
            });
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = 4 * i + (lane >> 4);
                *reinterpret_cast<uint4*>(slot + row * 256 + (((lane & 15) ^ (row & 15)) << 4)) = fetched[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) slot_d[(lane & 7) * kWaveCols + 8 * i + (lane >> 3)] = f16_bits_to_float(fetched_d[i]);
            const uint32_t cbase = static_cast<uint32_t>(r) * 256u | (static_cast<uint32_t>((r & 15) ^ h) << 4);
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                codes[g] = *reinterpret_cast<const uint4*>(slot + (cbase ^ (2 * g << 4)));
                scales[g] = slot_d[g * kWaveCols + r];
            }
        }
    };

    v16f acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[m] = v16f{};
    const v16f zero = {};
    const uint32_t abase = static_cast<uint32_t>(r) * 512u | (static_cast<uint32_t>(r ^ (2 * h)) << 4);
    fetch(o0);
    dma(o0, 0);
    wait_vm<0>();
    __syncthreads();
    for (int o = o0; o < o1; ++o) {
        const int nxt = min(o + 1, o1 - 1), buf = (o - o0) & 1;
        take();
        if constexpr (ALIGNED) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the slot has been read: it may be filled again)
        __builtin_amdgcn_sched_barrier(0);
        fetch(nxt);
        dma(nxt, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* at = smem + buf * kChunk;
        // piece of block g, instruction k, half h: 4 g + 2 h + k
        auto act_read = [&](int g, int k, int m) { return __builtin_bit_cast(v8h, *reinterpret_cast<const uint4*>(at + (abase ^ ((4 * g + k) << 4)) + m * 16384)); };
        v8h b0 = unpack8(codes[0].x, codes[0].y), b1 = unpack8(codes[0].z, codes[0].w), av[MB][2];
#pragma unroll
        for (int m = 0; m < MB; ++m) { av[m][0] = act_read(0, 0, m); av[m][1] = act_read(0, 1, m); }
        v16f c[2][MB];
        // block g: its matrix instructions, the scaling of block g - 1, the unpacking of block g + 1
        static_for<0, 8>([&](auto G) {
            constexpr int g = G;
            v8h n0, n1;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                c[g & 1][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[m][0], b0, zero, 0, 0, 0);
                if constexpr (g > 0) {
#pragma unroll
                    for (int v = 0; v < 8; ++v) acc[m][v] += scales[g - 1] * c[(g & 1) ^ 1][m][v];
                }
                if constexpr (g < 7) {
                    av[m][0] = act_read(g + 1, 0, m);
                    if (m == 0) n0 = unpack8(codes[g + 1].x, codes[g + 1].y);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                c[g & 1][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[m][1], b1, c[g & 1][m], 0, 0, 0);
                if constexpr (g > 0) {
#pragma unroll
                    for (int v = 8; v < 16; ++v) acc[m][v] += scales[g - 1] * c[(g & 1) ^ 1][m][v];
                }
                if constexpr (g < 7) {
                    av[m][1] = act_read(g + 1, 1, m);
                    if (m == 0) n1 = unpack8(codes[g + 1].z, codes[g + 1].w);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            b0 = n0;
            b1 = n1;
        });
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[m][v] += scales[7] * c[1][m][v];
        wait_vm<0>();
        __syncthreads();                             // the next step's rows are there, this one's have been read
    }
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
            const int row = (t0 + 32 * m + 8 * (v >> 2) + 4 * h + (v & 3)) / TERMS;
            float s = acc[m][v];
            if constexpr (TERMS == 2) s += acc[m][v + 1];
            if (row * TERMS < a.m_rows && col < a.n) store_any(a.y, a.y_dtype, static_cast<size_t>(row) * a.n + col, s * row_factor(a, row));
        }
}

template <int MB, int TERMS, bool ALIGNED>
int launch_q8_aligned(const RowsArgs& a, hipStream_t stream) {
    static SmemGrant granted;
    constexpr int kWaves = tile_waves(MB);
    const size_t smem = 2 * 32 * MB * 512 + kWaves * kSlotBytes;
    auto kern = q8_rows_kernel<MB, TERMS, ALIGNED>;
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

template <int MB, int TERMS>
int launch_q8(const RowsArgs& a, hipStream_t stream) {
    const bool aligned = a.blocks % 8 == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15u) == 0;
    return aligned ? launch_q8_aligned<MB, TERMS, true>(a, stream) : launch_q8_aligned<MB, TERMS, false>(a, stream);
}

}  // namespace

// From how many activation rows on this is faster than the kernels that run once per row (us, those kernels / this one, bf16 rows):
// 17408x5120 2 rows 38.3 / 37.0, 3 rows 52.6 / 37.3, 203 rows 3040 / 128; 4096x4096 2 rows 17.3 / 21.5, 3 rows 22.1 / 21.7; 3001x1984
// 4 rows 19.2 / 19.7, 8 rows 20.3 / 19.8; 1024x3072 8 rows 16.9 / 19.9, 12 rows 20.6 / 19.9.  Rows of an odd number of blocks have
// only a kernel of byte loads otherwise.
bool gemm_q8_0_supports(int rows, int n, int nb, const uint8_t* w) {
    const long long weights = static_cast<long long>(n) * nb * 32;
    const int least = (nb & 1) ? 2 : (weights >= (16ll << 20) ? 3 : (weights >= (4ll << 20) ? 8 : 12));
    // (2-byte loads, 32-bit offsets inside 32 weight rows and inside 64 activation rows)
    return rows >= least && (reinterpret_cast<uintptr_t>(w) & 1u) == 0 && static_cast<long long>(nb) * 34 * 32 < (1ll << 31) && rows_offsets_fit((nb + 7) / 8);
}

// (the query knows no activation type: room for float32 rows, which are two matrix rows each)
size_t gemm_q8_0_workspace_bytes(int rows, int n, int nb) { return std::max(rows_workspace(rows, 1, n, (nb + 7) / 8, kCost).bytes, rows_workspace(rows, 2, n, (nb + 7) / 8, kCost).bytes); }

int gemm_q8_0(const void* x, int x_dtype, const uint8_t* w, void* y, int y_dtype, int rows, int k, int n, int nb, void* workspace, size_t workspace_bytes,
              hipStream_t stream) {
    const int terms = x_dtype == PLLM_F32 ? 2 : 1, octets = (nb + 7) / 8;
    const RowsWorkspace ws = rows_workspace(rows, terms, n, octets, kCost);
    if (!workspace || workspace_bytes < ws.bytes) return PLLM_ERR_WORKSPACE;
    unsigned char* base = static_cast<unsigned char*>(workspace);
    const RowsPlan p = plan_rows(rows * terms, n, octets, kCost);
    RowsArgs a{};
    a.rows = reinterpret_cast<const _Float16*>(base);
    a.unscale = reinterpret_cast<const float*>(base + ws.unscale);
    a.w = w;
    a.y = y;
    a.partial = p.slices > 1 ? reinterpret_cast<float*>(base + ws.partial) : nullptr;
    a.y_dtype = y_dtype;
    a.m_rows = rows * terms;
    a.n = n;
    a.blocks = nb;
    a.kp = octets * kOctet;
    a.row_tiles = p.row_tiles;
    a.col_tiles = p.col_tiles;
    a.slices = p.slices;
    a.steps = octets / p.slices;
    a.steps_more = octets % p.slices;
    if (rows_as_held(x, x_dtype, k, a.kp)) {
        a.rows = static_cast<const _Float16*>(x);
        a.unscale = nullptr;
    } else {
        const int st = half_rows_stage(x, x_dtype, rows, k, a.kp, base, reinterpret_cast<float*>(base + ws.unscale), stream);
        if (st != PLLM_OK) return st;
    }
    if (p.mb == 1) return terms == 2 ? launch_q8<1, 2>(a, stream) : launch_q8<1, 1>(a, stream);
    return terms == 2 ? launch_q8<2, 2>(a, stream) : launch_q8<2, 1>(a, stream);
}

}  // namespace pllm
