// gemm_f32_split.hpp -- fp32 GEMM of K >= 256 (K % 32 == 0) on the bf16 matrix unit (gfx950).
//
//   Y[M, N] = X[M, K] * W, W as [K, N] or [N, K]; any M, N, stride and (4-byte) alignment; batched by strides.
//
// The fp32 matrix instruction does 64 flop a cycle, the bf16 one 1024.  Every fp32 number is the sum of three bf16 numbers (8 bits of
// significand each; hi, mid, lo), so a product is nine bf16 products, of which the ninth, of two lo parts, is below 2^-35 of it and left out: 128
// flop a cycle.  The products of two hi parts have a sum of their own, which rounds once in 32 k instead of 32 times; what the other seven
// round is 2^-8 of that; the two meet at the end of a slice of K.  (All in one sum, and without the products of mid and lo, rows of
// few nonzeros lost: one nonzero 2.5e-8 -> 3.5e-8.)  Error against 64-bit sums, relative in the 2-norm, before (gemm_f32.hpp) -> now, N(0, 1)
// operands: K = 256 1.5e-7 -> 6.8e-8, 1024 2.9e-7 -> 8.5e-8, 4096 5.7e-7 -> 1.4e-7; uniform in 0 .. 1 K = 1024 1.17e-7 -> 5.1e-8; rows of one
// nonzero 2.53e-8 in both, of eight 5.15e-8 -> 5.25e-8, of 32 6.9e-8 -> 6.1e-8.
// The parts are those of 2^23 times a number: a multiple of 2^-126, as every fp32 number is one of 2^-149, so that no part is below the smallest
// normal bf16 and the split is exact however small an element is beside the others.  The sums are 2^46 times the result and are scaled back
// at the end.  An output that is not finite then (infinities and NaN, magnitudes from 2^105, sums from 2^82) is computed again on the fp32
// unit, in the same slices; the other outputs of its tile stay as they are.
//
// Every tile sums in the same order, so an output depends on its row and its column alone: not on the tile, the batch around the row or the
// feature range around the column, whatever these hold.
// K goes in eight slices of whole chunks of 32, in a slice chunk by chunk the eight products, the slices one after the other.
//   * gemm_f32_split: (16 MI) x (16 NJ) tiles, a slice for each of 8 waves, no wave waits for another until the end.  A wave brings a chunk of
//     its slice to LDS of its own with direct-to-LDS loads (whole rows; straight to registers, as unaligned operands go, they
//     come in pieces of 16 bytes a lane, 800 x 4096 x 1024 85 instead of 65 us), takes it apart in registers and multiplies while
//     the next one lands.
//   * gemm_f32_split128: 128 x 128 tiles, the slices in turn; 8 waves share the operands, which are taken apart once on their way to LDS.
// What bounds the small tiles is taking operands apart (a lane spends 36 to 52 vector operations on its eight k of a row) and the traffic of the
// operands, the large ones the matrix unit with vector operations and LDS (192 KiB a chunk) beside it (1.0 PFLOP/s of bf16).
// Before (fp32 unit) -> now, us, [in, out]: 64 x 256 x 1024 5.2 -> 4.8, 800 x 1024 x 1024 22.5 -> 18.0, 800 x 4096 x 1024 81 -> 58, 800 x 1024 x
// 4096 73 -> 56, 4096 x 1024 x 4096 306 -> 228, 4096 x 4096 x 4096 1150 -> 960 ([out, in] 920: 150 TFLOP/s); up to 8 rows pay 0.4 at K = 1024 and 0.5
// at 4096 (8 x 1024 x 1024 4.4 -> 4.8), [out, in] weights gain there (8 x 1024 x 4096 14.1 -> 10.2).  The choice looks at K alone, so that a row
// has the same bits in every call; those rows are the price, and some unaligned operands with few tiles (800 x 1024 x 1024 22.7 -> 20.2, but
// 64 x 1024 x 1024 5.6 -> 6.4, 200 x 1024 x 256 4.7 -> 5.6).  Outputs summed again double the time of their tiles: 800 x 1024 x 1024 18 -> 39
// with an infinity in one row or in all, 4096 x 4096 x 4096 900 -> 990 and 2080 (another card).
#pragma once
#include "gemm_f32.hpp"

namespace lg {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

constexpr int FS_WAVES = 8, FS_THREADS = 64 * FS_WAVES, FS_K = 32;  // k of a chunk
constexpr float FS_SCALE = 0x1p23f, FS_UNSCALE = 0x1p-46f;

// -1 as bf16 in one half of a register
__device__ __forceinline__ unsigned minus_one(int shift) {
    unsigned v;
    asm("s_mov_b32 %0, %1" : "=s"(v) : "i"(0xbf80u << shift));
    return v;
}

// 2^23 v[0..7] = hi + mid + lo, each rounded to bf16 from what the one before leaves: exact for every finite v below 2^105.
// DOT: the rest is a two-term dot product with (-1, 0) or (0, -1), one instruction instead of two.  Tiles up to 32 x 32, whose time is the
// splitting, gain 2-9 % by it (8 x 1024 x 4096 11.5 -> 10.7 us); the 128 x 128 one loses 18-20 %, 64 x 64 1 %.
struct Split { bf16x8_t hi, mid, lo; };
template <bool DOT>
__device__ __forceinline__ Split split8(const float (&v)[8]) {
    union { bf16x8_t b; bf16x2_t p[4]; } h, m, l;
    const bf16x2_t first = __builtin_bit_cast(bf16x2_t, minus_one(0)), second = __builtin_bit_cast(bf16x2_t, minus_one(16));
    auto rest = [&](float2_t a, bf16x2_t part) {
        const unsigned bits = __builtin_bit_cast(unsigned, part);
        if (DOT) return float2_t{__builtin_amdgcn_fdot2_f32_bf16(part, first, a[0], false), __builtin_amdgcn_fdot2_f32_bf16(part, second, a[1], false)};
        return float2_t{a[0] - __builtin_bit_cast(float, bits << 16), a[1] - __builtin_bit_cast(float, bits & 0xffff0000u)};
    };
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const float2_t a = {v[2 * p] * FS_SCALE, v[2 * p + 1] * FS_SCALE};
        h.p[p] = __builtin_convertvector(a, bf16x2_t);
        const float2_t r = rest(a, h.p[p]);
        m.p[p] = __builtin_convertvector(r, bf16x2_t);
        l.p[p] = __builtin_convertvector(rest(r, m.p[p]), bf16x2_t);
    }
    return Split{h.b, m.b, l.b};
}

// the r-th of the eight k of a chunk that a lane multiplies, from 4 lk on: four in either half of the chunk, so that four lanes read 64 bytes of a row
__device__ __forceinline__ int split_k(int r) { return r < 4 ? r : r + 12; }

// The products of a chunk, small ones first; those of two hi parts have a sum of their own, so that its one rounding in a chunk is all that
// large products pay.  The weights are the A operand: acc[i][j][v] = token 16 i + l16, feature 4 lk + v of tile column j
template <int MI, int NJ, int JG>
__device__ __forceinline__ void split_multiply(float4_t (&acc)[MI][NJ], float4_t (&low)[MI][NJ], const Split (&xs)[MI], const Split (&ws)[JG], int j0) {
    auto product = [&](float4_t (&sum)[MI][NJ], auto wpart, auto xpart) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < JG; ++j) sum[i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wpart(ws[j]), xpart(xs[i]), sum[i][j0 + j], 0, 0, 0);
    };
    auto hi = [](const Split& s) { return s.hi; };
    auto mid = [](const Split& s) { return s.mid; };
    auto lo = [](const Split& s) { return s.lo; };
    product(low, lo, mid);
    product(low, mid, lo);
    product(low, lo, hi);
    product(low, hi, lo);
    product(low, mid, mid);
    product(low, mid, hi);
    product(low, hi, mid);
    product(acc, hi, hi);
}
// the same products in the fp32 unit, for outputs that the scaled sums do not reach
template <int MI, int NJ>
__device__ __forceinline__ void plain_multiply(float4_t (&acc)[MI][NJ], const float (&x)[MI][8], const float (&w)[NJ][8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][r], x[i][r], acc[i][j], 0, 0, 0);
}
__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= __FLT_MAX__; }

template <int WL, int MI, int NJ, bool STAGED>
__global__ __launch_bounds__(FS_THREADS, 2) void gemm_f32_split(GemmArgsF32 g, int tiles_m, int tiles_n) {
    constexpr int TM = 16 * MI, TN = 16 * NJ, PITCH = TN + 4;
    constexpr int X_CHUNK = TM * FS_K, W_CHUNK = TN * FS_K, CHUNK = X_CHUNK + W_CHUNK;  // floats
    extern __shared__ __attribute__((aligned(16))) float lds[];  // STAGED: a chunk of both operands for each wave; then the waves' sums
    float* const sums = lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lk = lane >> 4;

    // Workgroup ids are dealt to the 8 XCDs in turn: every XCD takes a contiguous run of tiles, rows fastest.
    int tm, tn, z;
    {
        const int total = gridDim.x, q = total >> 3, r = total & 7;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        const int id = xcd * q + min(xcd, r) + slot;
        const int strip = id / tiles_m;
        tm = id - strip * tiles_m;
        z = strip / tiles_n;
        tn = strip - z * tiles_n;
    }
    const int m0 = tm * TM, nlo = tn * TN;
    // [K, N] weights are loaded a whole tile wide: the last tile column is moved back so that it ends with the matrix (N >= TN then); the
    // features it shares with its neighbour are not stored.  (One feature tile, a feature at a time, may begin anywhere.)
    const int n0 = WL == W_KN && (NJ > 1 || STAGED) ? min(nlo, g.N - TN) : nlo;
    const float* const X = g.X + (int64_t)z * g.strideX;
    const float* const W = g.W + (int64_t)z * g.strideW;
    float* const Y = g.Y + (int64_t)z * g.strideY;

    const float* xp[MI];
    const float* wp[WL == W_NK ? NJ : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i) xp[i] = X + (int64_t)min(m0 + i * 16 + l16, g.M - 1) * g.ldx + 4 * lk;
    if (WL == W_NK) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) wp[j] = W + (int64_t)min(n0 + j * 16 + l16, g.N - 1) * g.ldw + 4 * lk;
    } else {
        wp[0] = W + (int64_t)(4 * lk) * g.ldw + (NJ == 1 ? min(n0 + l16, g.N - 1) : n0 + NJ * l16);
    }
    typedef typename FloatU<NJ>::type wvec_t;
    struct Chunk { float x[MI][8], w[NJ][8]; };
    auto load = [&](Chunk& c, int64_t k0) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4u_t v = *reinterpret_cast<const float4u_t*>(xp[i] + k0 + 16 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r) c.x[i][4 * h + r] = v[r];
            }
        if constexpr (WL == W_NK) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4u_t v = *reinterpret_cast<const float4u_t*>(wp[j] + k0 + 16 * h);
#pragma unroll
                    for (int r = 0; r < 4; ++r) c.w[j][4 * h + r] = v[r];
                }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const wvec_t v = *reinterpret_cast<const wvec_t*>(wp[0] + (k0 + split_k(r)) * g.ldw);
                if constexpr (NJ == 1) c.w[0][r] = v;
                else
#pragma unroll
                    for (int j = 0; j < NJ; ++j) c.w[j][r] = v[j];
            }
        }
    };
    float4_t acc[MI][NJ], low[MI][NJ];
    auto clear = [](float4_t (&sum)[MI][NJ]) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) sum[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    };
    clear(acc);
    clear(low);
    // all of X is taken apart, W a few tile columns at a time: registers
    constexpr int JG = MI == 4 || NJ == 1 ? 1 : 2;
    constexpr bool DOT = MI * NJ <= 4;
    Split xs[MI];
    auto multiply = [&](const float (&w)[NJ][8]) {
#pragma unroll
        for (int j = 0; j < NJ; j += JG) {
            Split ws[JG];
#pragma unroll
            for (int u = 0; u < JG; ++u) ws[u] = split8<DOT>(w[j + u]);
            split_multiply<MI, NJ, JG>(acc, low, xs, ws, j);
        }
    };

    const int chunks = g.K / FS_K, part = (chunks + FS_WAVES - 1) / FS_WAVES;
    const int first = wave * part, mine = min(chunks - first, part);  // this wave's chunks: first, first + 1, ...
    if constexpr (STAGED) {
        float* const xl = lds + wave * CHUNK;
        float* const wl = xl + X_CHUNK;
        constexpr int WPIECES = WL == W_NK ? 2 * NJ : 1, PIECE_K = 16 / NJ;  // [K, N] weights: a piece is PIECE_K rows, the pieces are alike
        unsigned xo[2 * MI], wo[WPIECES];  // element offsets in the 1 KiB pieces
#pragma unroll
        for (int i = 0; i < 2 * MI; ++i) {
            const int row = i * 8 + (lane >> 3);
            xo[i] = (unsigned)min(row, g.M - 1 - m0) * (unsigned)g.ldx + swz_a(row, lane & 7) * 4;
        }
#pragma unroll
        for (int i = 0; i < WPIECES; ++i) {
            if (WL == W_NK) {
                const int row = i * 8 + (lane >> 3);
                wo[i] = (unsigned)min(row, g.N - 1 - n0) * (unsigned)g.ldw + swz_a(row, lane & 7) * 4;
            } else {
                wo[i] = (unsigned)(lane / (4 * NJ)) * (unsigned)g.ldw + lane % (4 * NJ) * 4;
            }
        }
        const float* const xb = X + (int64_t)m0 * g.ldx;
        const float* const wb = WL == W_NK ? W + (int64_t)n0 * g.ldw : W + n0;
        auto fetch = [&](int t) {
            const float* const xk = xb + (int64_t)t * FS_K;
            const float* const wk = wb + (int64_t)t * FS_K * (WL == W_NK ? 1 : g.ldw);
#pragma unroll
            for (int i = 0; i < 2 * MI; ++i) load_lds16(reinterpret_cast<const half_t*>(xk + xo[i]), reinterpret_cast<half_t*>(xl + i * 256));
#pragma unroll
            for (int i = 0; i < 2 * NJ; ++i) {
                const float* const p = WL == W_NK ? wk + wo[WL == W_NK ? i : 0] : wk + (int64_t)(i * PIECE_K) * g.ldw + wo[0];
                load_lds16(reinterpret_cast<const half_t*>(p), reinterpret_cast<half_t*>(wl + i * 256));
            }
        };
        auto read8 = [&](float (&v)[8], const float* base) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4_t q = *reinterpret_cast<const float4_t*>(base + l16 * FS_K + swz_a(l16, 4 * h + lk) * 4);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[4 * h + r] = q[r];
            }
        };
        if (mine > 0) fetch(first);
        for (int t = 0; t < mine; ++t) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                float v[8];
                read8(v, xl + i * 16 * FS_K);
                xs[i] = split8<DOT>(v);
            }
            float w[NJ][8];
            if constexpr (WL == W_NK) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) read8(w[j], wl + j * 16 * FS_K);
            } else {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    typedef float rowvec_t __attribute__((ext_vector_type(NJ > 1 ? NJ : 2)));
                    const float* const p = wl + (4 * lk + split_k(r)) * TN + NJ * l16;
                    if constexpr (NJ == 1) w[0][r] = *p;
                    else {
                        const rowvec_t q = *reinterpret_cast<const rowvec_t*>(p);
#pragma unroll
                        for (int j = 0; j < NJ; ++j) w[j][r] = q[j];
                    }
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // everything has been read: the next chunk may land
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1 < mine) fetch(first + t + 1);
            multiply(w);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if constexpr (MI == 4) {
        // its sums leave no registers for a chunk on its way: the other wave of the SIMD multiplies meanwhile (800 x 1024 x 1024 20.2 us, in tiles of
        // 32 x 64 30.7)
        for (int t = 0; t < mine; ++t) {
            Chunk c;
            load(c, (int64_t)(first + t) * FS_K);
#pragma unroll
            for (int i = 0; i < MI; ++i) xs[i] = split8<DOT>(c.x[i]);
            multiply(c.w);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if (mine > 0) {
        Chunk c;
        load(c, (int64_t)first * FS_K);
        for (int t = 0; t < mine; ++t) {
#pragma unroll
            for (int i = 0; i < MI; ++i) xs[i] = split8<DOT>(c.x[i]);
            float w[NJ][8];
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 8; ++r) w[j][r] = c.w[j][r];
            load(c, (int64_t)(first + min(t + 1, mine - 1)) * FS_K);
            __builtin_amdgcn_sched_barrier(0);
            multiply(w);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] += low[i][j];

    // ---- the eight sums of an output meet, 16 token rows at a time; if one is not finite, those outputs are summed in the fp32 unit -----
    unsigned bad = 0;  // of this thread's outputs, 4 of each 16 rows
    for (bool again = false;; again = true) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            float* const mybuf = sums + (wave * 16 + l16) * PITCH;
            if (STAGED || i > 0 || again) __syncthreads();
            if constexpr (WL == W_NK || NJ == 1) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) *reinterpret_cast<float4_t*>(mybuf + j * 16 + 4 * lk) = acc[i][j];
            } else {
                typedef float rowvec_t __attribute__((ext_vector_type(NJ)));
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    rowvec_t o;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) o[j] = acc[i][j][v];
                    *reinterpret_cast<rowvec_t*>(mybuf + NJ * (4 * lk + v)) = o;
                }
            }
            __syncthreads();
            const int row = tid / (TN / 4), col = tid % (TN / 4) * 4;
            const int m = m0 + i * 16 + row, n = n0 + col;
            if (row < 16 && m < g.M && n < g.N) {
                float4_t v = *reinterpret_cast<const float4_t*>(&sums[row * PITCH + col]);
#pragma unroll
                for (int s = 1; s < FS_WAVES; ++s) v += *reinterpret_cast<const float4_t*>(&sums[(s * 16 + row) * PITCH + col]);
                float* const p = Y + (int64_t)m * g.ldy + n;
                if (!again) {
                    v *= FS_UNSCALE;
#pragma unroll
                    for (int r = 0; r < 4; ++r) bad |= (finite(v[r]) ? 0u : 1u) << (4 * i + r);
                }
                if (n >= nlo && n + 3 < g.N && !again) {
                    *reinterpret_cast<float4u_t*>(p) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n + r >= nlo && n + r < g.N && (!again || (bad >> (4 * i + r) & 1))) p[r] = v[r];
                }
            }
        }
        if (again || !__syncthreads_or(bad != 0)) break;
        clear(acc);
        for (int t = 0; t < mine; ++t) {
            Chunk c;
            load(c, (int64_t)(first + t) * FS_K);
            plain_multiply<MI, NJ>(acc, c.x, c.w);
        }
    }
}

template <int WL, int MI, int NJ, bool STAGED>
static void launch_f32_split_tile(const GemmArgsF32& g, int batch, hipStream_t stream) {
    const int tiles_m = (g.M + 16 * MI - 1) / (16 * MI), tiles_n = (g.N + 16 * NJ - 1) / (16 * NJ);
    constexpr size_t chunks = STAGED ? (size_t)FS_WAVES * 16 * (MI + NJ) * FS_K * sizeof(float) : 0, sums = (size_t)FS_WAVES * 16 * (16 * NJ + 4) * sizeof(float);
    constexpr size_t smem = chunks > sums ? chunks : sums;
    static_assert(smem <= 160 * 1024, "a compute unit has 160 KiB of LDS");
    static const hipError_t attr_rc = hipFuncSetAttribute((const void*)gemm_f32_split<WL, MI, NJ, STAGED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    (void)attr_rc;
    hipLaunchKernelGGL((gemm_f32_split<WL, MI, NJ, STAGED>), dim3((unsigned)(tiles_m * tiles_n * batch)), dim3(FS_THREADS), smem, stream, g, tiles_m, tiles_n);
}

// ---- 128 x 128 tiles ----------------------------------------------------------------------------------------------------------
constexpr int FT_BLOCK = 4 * 320;           // bytes of one part of a block of 16 rows x 32 k: four groups of k, 16 rows of 16 bytes each, and 64 bytes apart
constexpr int FT_PART = 8 * FT_BLOCK;       // of one part of a 128-row operand
constexpr int FT_CHUNK = 6 * FT_PART;       // both operands: X hi, mid, lo, W hi, mid, lo
constexpr int FT_MI = 4, FT_NJ = 2;         // a wave's 64 x 32 outputs

template <int WL>
__global__ __launch_bounds__(FS_THREADS, 2) void gemm_f32_split128(GemmArgsF32 g, int tiles_m, int tiles_n) {
    extern __shared__ __attribute__((aligned(16))) char lds128[];  // two chunks
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int l16 = lane & 15, lk = lane >> 4;
    int tm, tn, z;
    {
        const int total = gridDim.x, q = total >> 3, r = total & 7;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        const int id = xcd * q + min(xcd, r) + slot;
        const int strip = id / tiles_m;
        tm = id - strip * tiles_m;
        z = strip / tiles_n;
        tn = strip - z * tiles_n;
    }
    const int m0 = tm * 128, n0 = tn * 128;
    const float* const X = g.X + (int64_t)z * g.strideX;
    const float* const W = g.W + (int64_t)z * g.strideW;
    float* const Y = g.Y + (int64_t)z * g.strideY;

    // A thread brings eight k of one row of X and of one feature of W into LDS: [N, K] rows four threads to a row, [K, N] weights one feature
    // a lane.  Rows beyond the matrix are read from its last one and never stored.
    const int xkb = lane & 3, wkb = WL == W_NK ? xkb : wave & 3;
    const int xrow = 16 * wave + (lane >> 2), wrow = WL == W_NK ? xrow : (wave >> 2) * 64 + lane;
    const float* const xp = X + (int64_t)min(m0 + xrow, g.M - 1) * g.ldx + 4 * xkb;
    const unsigned wfeature = min(n0 + wrow, g.N - 1);
    const float* const wp = WL == W_NK ? W + (int64_t)wfeature * g.ldw + 4 * wkb : W + (int64_t)(4 * wkb) * g.ldw;
    char* const xdst = lds128 + (xrow >> 4) * FT_BLOCK + xkb * 320 + (xrow & 15) * 16;
    char* const wdst = lds128 + 3 * FT_PART + (wrow >> 4) * FT_BLOCK + wkb * 320 + (wrow & 15) * 16;

    const int chunks = g.K / FS_K, part = (chunks + FS_WAVES - 1) / FS_WAVES;
    struct Raw { float x[8], w[8]; };
    auto gload = [&](Raw& raw, int c) {  // a whole chunk
        const int64_t k0 = (int64_t)c * FS_K;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4u_t v = *reinterpret_cast<const float4u_t*>(xp + k0 + 16 * h);
#pragma unroll
            for (int r = 0; r < 4; ++r) raw.x[4 * h + r] = v[r];
            if (WL == W_NK) {
                const float4u_t w = *reinterpret_cast<const float4u_t*>(wp + k0 + 16 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r) raw.w[4 * h + r] = w[r];
            }
        }
        if (WL == W_KN) {
#pragma unroll
            for (int r = 0; r < 8; ++r) raw.w[r] = (wp + (k0 + split_k(r)) * g.ldw)[wfeature];
        }
    };
    auto stage = [&](const Raw& raw, int buf) {
        const Split x = split8<false>(raw.x), w = split8<false>(raw.w);
        char* const xd = xdst + buf * FT_CHUNK;
        char* const wd = wdst + buf * FT_CHUNK;
        *reinterpret_cast<bf16x8_t*>(xd) = x.hi;
        *reinterpret_cast<bf16x8_t*>(xd + FT_PART) = x.mid;
        *reinterpret_cast<bf16x8_t*>(xd + 2 * FT_PART) = x.lo;
        *reinterpret_cast<bf16x8_t*>(wd) = w.hi;
        *reinterpret_cast<bf16x8_t*>(wd + FT_PART) = w.mid;
        *reinterpret_cast<bf16x8_t*>(wd + 2 * FT_PART) = w.lo;
    };
    struct Frags { Split x[FT_MI], w[FT_NJ]; };
    auto fetch = [&](Frags& f, int buf) {
        const char* const xb = lds128 + buf * FT_CHUNK + (wm * FT_MI) * FT_BLOCK + lk * 320 + l16 * 16;
        const char* const wb = lds128 + buf * FT_CHUNK + 3 * FT_PART + (wn * FT_NJ) * FT_BLOCK + lk * 320 + l16 * 16;
        auto part_of = [](const char* b, int p) { return *reinterpret_cast<const bf16x8_t*>(b + p * FT_PART); };
#pragma unroll
        for (int j = 0; j < FT_NJ; ++j) f.w[j] = Split{part_of(wb + j * FT_BLOCK, 0), part_of(wb + j * FT_BLOCK, 1), part_of(wb + j * FT_BLOCK, 2)};
#pragma unroll
        for (int i = 0; i < FT_MI; ++i) f.x[i] = Split{part_of(xb + i * FT_BLOCK, 0), part_of(xb + i * FT_BLOCK, 1), part_of(xb + i * FT_BLOCK, 2)};
    };
    float4_t acc[FT_MI][FT_NJ], low[FT_MI][FT_NJ], total[FT_MI][FT_NJ];
#pragma unroll
    for (int i = 0; i < FT_MI; ++i)
#pragma unroll
        for (int j = 0; j < FT_NJ; ++j) {
            acc[i][j] = low[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
            total[i][j] = float4_t{-0.f, -0.f, -0.f, -0.f};  // x + -0 is x
        }
    int left = part;  // chunks before the slice ends
    auto end_chunk = [&](bool last) {
        if (--left > 0 && !last) return;
        left = part;
#pragma unroll
        for (int i = 0; i < FT_MI; ++i)
#pragma unroll
            for (int j = 0; j < FT_NJ; ++j) {
                total[i][j] += acc[i][j] + low[i][j];
                acc[i][j] = low[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
    };

    // While chunk c is multiplied, c + 1 is split on its way to LDS and c + 2 comes from memory.
    Frags f;
    Raw raw;
    gload(raw, 0);
    stage(raw, 0);
    if (chunks > 1) gload(raw, 1);
    __syncthreads();
    int c = 0;
    for (; c + 2 < chunks; ++c) {
        __builtin_amdgcn_sched_barrier(0);
        fetch(f, c & 1);
        stage(raw, (c + 1) & 1);
        gload(raw, c + 2);
        split_multiply<FT_MI, FT_NJ, FT_NJ>(acc, low, f.x, f.w, 0);
        // the reads first, then three vector operations of the split under every matrix instruction
        __builtin_amdgcn_sched_group_barrier(0x100, 3 * (FT_MI + FT_NJ), 0);
#pragma unroll
        for (int m = 0; m < 8 * FT_MI * FT_NJ; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        end_chunk(false);
        __syncthreads();
    }
    for (; c < chunks; ++c) {
        fetch(f, c & 1);
        if (c + 1 < chunks) stage(raw, (c + 1) & 1);
        split_multiply<FT_MI, FT_NJ, FT_NJ>(acc, low, f.x, f.w, 0);
        end_chunk(c == chunks - 1);
        __syncthreads();
    }
    unsigned bad = 0;  // the outputs of this lane that are not finite, which the fp32 unit sums again
    for (bool again = false;; again = true) {
#pragma unroll
        for (int i = 0; i < FT_MI; ++i) {
            const int m = m0 + wm * 64 + i * 16 + l16;
#pragma unroll
            for (int j = 0; j < FT_NJ; ++j) {
                const int n = n0 + wn * 32 + j * 16 + 4 * lk, bit = 4 * (i * FT_NJ + j);
                float* const p = Y + (int64_t)m * g.ldy + n;
                if (!again) {
                    total[i][j] *= FS_UNSCALE;
#pragma unroll
                    for (int r = 0; r < 4; ++r) bad |= (finite(total[i][j][r]) ? 0u : 1u) << (bit + r);
                }
                if (m >= g.M) continue;
                if (n + 3 < g.N && !again) {
                    *reinterpret_cast<float4u_t*>(p) = total[i][j];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n + r < g.N && (!again || (bad >> (bit + r) & 1))) p[r] = total[i][j][r];
                }
            }
        }
        if (again || !__any(bad != 0)) break;
#pragma unroll
        for (int i = 0; i < FT_MI; ++i)
#pragma unroll
            for (int j = 0; j < FT_NJ; ++j) total[i][j] = float4_t{-0.f, -0.f, -0.f, -0.f};
        for (c = 0; c < chunks; ++c) {  // acc and low are zero
            const int64_t k0 = (int64_t)c * FS_K + 4 * lk;
            float x[FT_MI][8], w[FT_NJ][8];
            auto row8 = [](float (&v)[8], const float* p) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4u_t q = *reinterpret_cast<const float4u_t*>(p + 16 * h);
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[4 * h + r] = q[r];
                }
            };
#pragma unroll
            for (int i = 0; i < FT_MI; ++i) row8(x[i], X + (int64_t)min(m0 + wm * 64 + i * 16 + l16, g.M - 1) * g.ldx + k0);
#pragma unroll
            for (int j = 0; j < FT_NJ; ++j) {
                const int64_t n = min(n0 + wn * 32 + j * 16 + l16, g.N - 1);
                if constexpr (WL == W_NK) row8(w[j], W + n * g.ldw + k0);
                else
#pragma unroll
                    for (int r = 0; r < 8; ++r) w[j][r] = W[(k0 + split_k(r)) * g.ldw + n];
            }
            plain_multiply<FT_MI, FT_NJ>(acc, x, w);
            end_chunk(c == chunks - 1);
        }
    }
}

template <int WL>
static void launch_f32_split128(const GemmArgsF32& g, int batch, hipStream_t stream) {
    const int tiles_m = (g.M + 127) / 128, tiles_n = (g.N + 127) / 128;
    static const hipError_t attr_rc = hipFuncSetAttribute((const void*)gemm_f32_split128<WL>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * FT_CHUNK);
    (void)attr_rc;
    hipLaunchKernelGGL((gemm_f32_split128<WL>), dim3((unsigned)(tiles_m * tiles_n * batch)), dim3(FS_THREADS), 2 * FT_CHUNK, stream, g, tiles_m, tiles_n);
}

}  // namespace lg
