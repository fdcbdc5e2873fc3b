// gemm_f32.hpp -- fp32 GEMM for few output tiles (gfx950): v_mfma_f32_16x16x4_f32, operands straight from global memory to registers.
// Of K below 256 or not in chunks of 32; the others are the bf16 unit's (gemm_f32_split.hpp).
//
//   Y[M, N] = X[M, K] * W, W as [K, N] or [N, K]; any shape, stride and (4-byte) alignment; batched by strides.
//
// An fp32 matrix instruction does 64 flop a cycle: a (16 MI) x (16 NJ) tile of outputs needs 16 (MI + NJ) operand bytes a cycle at
// most, which the caches deliver without LDS.  What bounds the path is how the work is dealt out -- the 128 x 128 tiles that this
// replaces left a layer of hidden 1024 and 800 tokens on 56 of 256 compute units and one of hidden 256 on two -- and, inside a
// workgroup, the latency of the loads.  So:
//   * the four waves of a workgroup own the same tile and take a quarter of K each, no wave waits for another until the end, and
//     even a 16 x 16 tile has four SIMDs at work;
//   * a wave keeps D chunks of both operands in flight in registers;
//   * a lane loads 4 consecutive k of one row as 16 bytes ([N, K] weights, X) and feeds one of them to each of four matrix
//     instructions -- any assignment of k to instruction slots will do if both operands agree; of [K, N] weights it loads NJ
//     consecutive features, one for each tile column, so tile column j holds features NJ c + j;
//   * the four sums of an output meet in LDS, added in wave order, and leave as whole rows.
// Every tile size, and the 128 x 128 kernel of gemm.hip, adds the same products in the same order: within a quarter of K by chunks of 16
// k, in a chunk by the slots of the matrix instruction, then the four quarters.  So a result does not depend on the tile, the batch
// around a row or the feature range around a column.
#pragma once
#include "gemm_common.hpp"

namespace lg {

struct GemmArgsF32 {
    int M, N, K;
    const float* X; int64_t ldx; int64_t strideX;
    const float* W; int64_t ldw; int64_t strideW;
    float* Y;       int64_t ldy; int64_t strideY;
};

// vectors at 4-byte alignment: global memory takes them at any dword address
template <int N> struct FloatU;
template <> struct FloatU<1> { typedef float type; };
template <> struct FloatU<2> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct FloatU<4> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
typedef FloatU<4>::type float4u_t;

constexpr int SF_WAVES = 4, SF_THREADS = 64 * SF_WAVES, SF_K = 16;  // k of a chunk
// chunks in a quarter of K; the last ones may hold fewer, or none
__host__ __device__ inline int f32_quarter(int K) { return ((K + SF_K - 1) / SF_K + SF_WAVES - 1) / SF_WAVES; }

template <int WL, int MI, int NJ, int D>
__global__ __launch_bounds__(SF_THREADS, 2) void gemm_f32_direct(GemmArgsF32 g, int tiles_m, int tiles_n) {
    constexpr int TM = 16 * MI, TN = 16 * NJ, PITCH = TN + 4, BUFS = MI > 1 ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float sums[BUFS][SF_WAVES][16 * PITCH];
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
    // [K, N] weights are loaded NJ features at a time: the last tile column is moved back so that it ends with the matrix (N >= TN
    // unless NJ is 1); the features it shares with its neighbour are not stored.
    const int n0 = WL == W_KN && NJ > 1 ? min(nlo, g.N - TN) : nlo;
    const float* const X = g.X + (int64_t)z * g.strideX;
    const float* const W = g.W + (int64_t)z * g.strideW;
    float* const Y = g.Y + (int64_t)z * g.strideY;

    // rows beyond the matrix are read from its last row and never stored
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

    typedef typename FloatU<WL == W_NK ? 4 : NJ>::type wvec_t;
    constexpr int WV = WL == W_NK ? NJ : 4;  // weight loads of a chunk
    struct Chunk { float4u_t x[MI]; wvec_t w[WV]; };
    auto load = [&](Chunk& c, int64_t k0) {
#pragma unroll
        for (int i = 0; i < MI; ++i) c.x[i] = *reinterpret_cast<const float4u_t*>(xp[i] + k0);
#pragma unroll
        for (int i = 0; i < WV; ++i) c.w[i] = *reinterpret_cast<const wvec_t*>(WL == W_NK ? wp[WL == W_NK ? i : 0] + k0 : wp[0] + (k0 + i) * g.ldw);
    };
    // the k that are left over after whole chunks: what lies beyond K counts as zero in both operands
    auto load_tail = [&](Chunk& c, int64_t k0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool in = k0 + 4 * lk + r < g.K;
#pragma unroll
            for (int i = 0; i < MI; ++i) c.x[i][r] = in ? xp[i][k0 + r] : 0.f;
            if constexpr (WL == W_NK) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) c.w[j][r] = in ? wp[j][k0 + r] : 0.f;
            } else {
                wvec_t v{};
                if (in) v = *reinterpret_cast<const wvec_t*>(wp[0] + (k0 + r) * g.ldw);
                c.w[r] = v;
            }
        }
    };
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    // the weights are the A operand: acc[i][j][v] = token 16 i + l16, feature 4 lk + v of tile column j
    auto multiply = [&](const Chunk& c) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    float w;
                    if constexpr (WL == W_NK) w = c.w[j][r];
                    else if constexpr (NJ == 1) w = c.w[r];
                    else w = c.w[r][j];
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, c.x[i][r], acc[i][j], 0, 0, 0);
                }
    };

    const int chunks = g.K / SF_K, quarter = f32_quarter(g.K);
    const int first = wave * quarter, mine = min(chunks - first, quarter);  // this wave's whole chunks: first, first + 1, ...
    if (mine > 0) {
        Chunk c[D];
        // the chunk index is clamped to the last one: loads past it are not used
        auto at = [&](int t) { return (int64_t)(first + min(t, mine - 1)) * SF_K; };
#pragma unroll
        for (int d = 0; d < D; ++d) load(c[d], at(d));
        for (int t = 0; t < mine; t += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (t + d < mine) multiply(c[d]);
                __builtin_amdgcn_sched_barrier(0);
                load(c[d], at(t + d + D));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if (g.K % SF_K != 0 && wave == chunks / quarter) {
        Chunk c;
        load_tail(c, (int64_t)chunks * SF_K);
        multiply(c);
    }

    // ---- the four sums of an output meet, 16 token rows at a time -----------------------------------------------------------
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        float* const mybuf = sums[i % BUFS][wave] + l16 * PITCH;
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
            float4_t v = *reinterpret_cast<const float4_t*>(&sums[i % BUFS][0][row * PITCH + col]);
#pragma unroll
            for (int s = 1; s < SF_WAVES; ++s) v += *reinterpret_cast<const float4_t*>(&sums[i % BUFS][s][row * PITCH + col]);
            float* const p = Y + (int64_t)m * g.ldy + n;
            if (n >= nlo && n + 3 < g.N) {
                *reinterpret_cast<float4u_t*>(p) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r >= nlo && n + r < g.N) p[r] = v[r];
            }
        }
    }
}

template <int WL, int MI, int NJ, int D>
static void launch_f32_direct_tile(const GemmArgsF32& g, int batch, hipStream_t stream) {
    const int tiles_m = (g.M + 16 * MI - 1) / (16 * MI), tiles_n = (g.N + 16 * NJ - 1) / (16 * NJ);
    hipLaunchKernelGGL((gemm_f32_direct<WL, MI, NJ, D>), dim3((unsigned)(tiles_m * tiles_n * batch)), dim3(SF_THREADS), 0, stream, g, tiles_m, tiles_n);
}

}  // namespace lg
