// gemm.hip -- hand-written GEMMs for gfx950: the cuBLAS calls of the reference's launch vector.
//
//   gemm_f16_generic   128x128x32 tiles, 4 waves (2x2), MFMA 16x16x32 f16 -> fp32, any shape / stride /
//                      alignment, both weight layouts, optional fused epilogue.  Correctness workhorse
//                      (edge tiles, decomposed sub-ranges, attention GEMMs, small models).
//   gemm_f32_mfma      128x128x16 tiles on v_mfma_f32_16x16x4_f32 for the fp32 instantiation (any shape, both layouts); problems
//                      of few such tiles go to gemm_f32.hip, those of K >= 256 in whole chunks of 32 to gemm_f32_split.hip;
//   gemm_f32_generic   64x64x16 VALU tiles, kept as a cross-check.
// Aligned problems are routed to the tile kernels of gemm_mid.hpp and the weight-streaming ones.
#include <stdlib.h>

#include "gemm_common.hpp"
#include "gemm_f32.hpp"

namespace lg {

int launch_gemm_skinny_f16(const GemmArgs& g, const GemmGroup& grp, const RowMap* rows, int wlayout, int batch, hipStream_t stream, bool* handled);
int launch_gemv_f16(const GemmArgs& g, const GemmGroup& grp, const RowMap* rows, int wlayout, int batch, hipStream_t stream, bool* handled);
int launch_gemm_skinny_sliced_f16(const GemmArgs& g, int wlayout, int batch, hipStream_t stream, bool* handled);
int launch_gemm_f32_split(const GemmArgsF32& g, int wlayout, int batch, bool aligned, hipStream_t stream, bool* handled);
int launch_gemm_f32_direct(const GemmArgsF32& g, int wlayout, int batch, bool aligned, hipStream_t stream, bool* handled);

// ---------------------------------------------------------------------------------------------------
// fp16 generic kernel
// ---------------------------------------------------------------------------------------------------
constexpr int GB_M = 128, GB_N = 128, GB_K = 32;
constexpr int GA_STRIDE = GB_K + 8;    // halves per row of the [rows][k] tiles (80 B: conflict-light b128 reads)
constexpr int GBKN_STRIDE = GB_N + 8;  // halves per row of the [k][n] tile

// 8 consecutive halves p[0..7], the first `valid` of them (the others 0).  Whole vectors are one 16-byte load at any alignment, which
// global memory takes: an element at a time where rows are not 16-byte aligned, the products of attention over 2 x 333 tokens (48 heads
// of 128) took 78 us (scores) and 89 us (values); now 19 and 17.  Vectors outside the matrix skip the elements as a whole: every tile
// has some (rows beyond M, features beyond N), and eight compares for each cost 130 rows x 1000 x 2048 80 us instead of 44.
__device__ __forceinline__ half8_t load8(const half_t* p, int valid) {
    half8_t r = {0, 0, 0, 0, 0, 0, 0, 0};
    if (valid >= 8) return *reinterpret_cast<const half8u_t*>(p);
    if (valid > 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < valid) r[i] = p[i];
    }
    return r;
}

template <int WL, int EPI>
__global__ __launch_bounds__(256) void gemm_f16_generic(GemmArgs g) {
    __shared__ __attribute__((aligned(16))) half_t As[GB_M * GA_STRIDE];
    __shared__ __attribute__((aligned(16))) half_t Bs[(WL == W_KN) ? GB_K * GBKN_STRIDE : GB_N * GA_STRIDE];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;  // 2x2 waves, 64x64 each
    const int m0 = blockIdx.y * GB_M, n0 = blockIdx.x * GB_N;
    const half_t* X = g.X + (int64_t)blockIdx.z * g.strideX;
    const half_t* W = g.W + (int64_t)blockIdx.z * g.strideW;
    half_t* Y = g.Y + (int64_t)blockIdx.z * g.strideY;

    float4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    half8_t ra[2], rb[2];
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int v = tid + 256 * i;
            {   // X tile: 128 rows x 4 k-vectors
                const int row = v >> 2, kv = v & 3;
                const int m = m0 + row, k = k0 + kv * 8;
                ra[i] = load8(X + (int64_t)m * g.ldx + k, (m < g.M) ? (g.K - k) : 0);
            }
            if (WL == W_TILED) {  // W tile: 8 fragment blocks (16 features x 32 k each), one lane's 16 bytes per thread
                const int blk = v >> 6, ln = v & 63;
                const int n = n0 + blk * 16;   // N % 16 == 0 and K % 32 == 0: a block is there as a whole or not at all
                rb[i] = load8(W + ((int64_t)(n >> 4) * (g.K >> 5) + (k0 >> 5)) * 512 + ln * 8, (n < g.N) ? 8 : 0);
            } else if (WL == W_NK) {  // W tile: 128 n-rows x 4 k-vectors
                const int row = v >> 2, kv = v & 3;
                const int n = n0 + row, k = k0 + kv * 8;
                rb[i] = load8(W + (int64_t)n * g.ldw + k, (n < g.N) ? (g.K - k) : 0);
            } else {           // W tile: 32 k-rows x 16 n-vectors
                const int row = v >> 4, nv = v & 15;
                const int k = k0 + row, n = n0 + nv * 8;
                rb[i] = load8(W + (int64_t)k * g.ldw + n, (k < g.K) ? (g.N - n) : 0);
            }
        }
    };
    auto lstore = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int v = tid + 256 * i;
            *reinterpret_cast<half8_t*>(&As[(v >> 2) * GA_STRIDE + (v & 3) * 8]) = ra[i];
            if (WL == W_TILED)
                *reinterpret_cast<half8_t*>(&Bs[v * 8]) = rb[i];   // block v / 64 keeps its register order
            else if (WL == W_NK)
                *reinterpret_cast<half8_t*>(&Bs[(v >> 2) * GA_STRIDE + (v & 3) * 8]) = rb[i];
            else
                *reinterpret_cast<half8_t*>(&Bs[(v >> 4) * GBKN_STRIDE + (v & 15) * 8]) = rb[i];
        }
    };

    const int l16 = lane & 15, lk = lane >> 4;  // row inside a 16-row MFMA tile, k-chunk (8 halves) index
    gload(0);
    for (int k0 = 0; k0 < g.K; k0 += GB_K) {
        __syncthreads();  // previous tile fully consumed
        lstore();
        __syncthreads();
        if (k0 + GB_K < g.K) gload(k0 + GB_K);

        half8_t a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[i] = *reinterpret_cast<const half8_t*>(&As[(wm * 64 + i * 16 + l16) * GA_STRIDE + lk * 8]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (WL == W_TILED) {
                b[j] = *reinterpret_cast<const half8_t*>(&Bs[((wn * 4 + j) * 64 + lane) * 8]);
            } else if (WL == W_NK) {
                b[j] = *reinterpret_cast<const half8_t*>(&Bs[(wn * 64 + j * 16 + l16) * GA_STRIDE + lk * 8]);
            } else {
                const int col = wn * 64 + j * 16 + 4 * (l16 & 3);
                const int krow = lk * 8 + (l16 >> 2);
                half4_t lo = lds_read_tr4(&Bs[krow * GBKN_STRIDE + col]);
                half4_t hi = lds_read_tr4(&Bs[(krow + 4) * GBKN_STRIDE + col]);
                b[j] = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
        }
        // operands swapped so that each lane owns 4 consecutive output columns (n) of one row (m):
        //   acc[i][j][r] = Y[m_tile(i) + lane%16][n_tile(j) + 4*(lane/16) + r]
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = mfma16(b[j], a[i], acc[i][j]);
    }

    const bool vec_ok = EPI != LG_EPI_BIAS_HEADS || g.epi.d % 4 == 0;  // four outputs of one head
    if (EPI == LG_EPI_BIAS_GEGLU) {
        // a wave's four 16-feature tiles are two (gate, up) pairs (N % 32 == 0, tiles start at multiples of 64)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; j += 2)
                epilogue_geglu4(g, Y, m0 + wm * 64 + i * 16 + l16, n0 + wn * 64 + j * 16 + 4 * lk, acc[i][j], acc[i][j + 1], vec_ok);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + wm * 64 + i * 16 + l16;
            const int n = n0 + wn * 64 + j * 16 + 4 * lk;
            switch (EPI) {
                case LG_EPI_NONE: epilogue_store4<LG_EPI_NONE>(g, Y, m, n, acc[i][j], vec_ok); break;
                case LG_EPI_BIAS: epilogue_store4<LG_EPI_BIAS>(g, Y, m, n, acc[i][j], vec_ok); break;
                case LG_EPI_BIAS_GELU: epilogue_store4<LG_EPI_BIAS_GELU>(g, Y, m, n, acc[i][j], vec_ok); break;
                default: epilogue_store4<LG_EPI_BIAS_HEADS>(g, Y, m, n, acc[i][j], vec_ok); break;
            }
        }
}

template <int WL>
static void launch_generic_epi(const GemmArgs& g, dim3 grid, hipStream_t stream) {
    switch (g.epi.kind) {
        case LG_EPI_NONE: hipLaunchKernelGGL((gemm_f16_generic<WL, LG_EPI_NONE>), grid, dim3(256), 0, stream, g); break;
        case LG_EPI_BIAS: hipLaunchKernelGGL((gemm_f16_generic<WL, LG_EPI_BIAS>), grid, dim3(256), 0, stream, g); break;
        case LG_EPI_BIAS_GELU: hipLaunchKernelGGL((gemm_f16_generic<WL, LG_EPI_BIAS_GELU>), grid, dim3(256), 0, stream, g); break;
        case LG_EPI_BIAS_GEGLU: hipLaunchKernelGGL((gemm_f16_generic<WL, LG_EPI_BIAS_GEGLU>), grid, dim3(256), 0, stream, g); break;
        default: hipLaunchKernelGGL((gemm_f16_generic<WL, LG_EPI_BIAS_HEADS>), grid, dim3(256), 0, stream, g); break;
    }
}

// The kernels that run a problem, or a group as one launch: the matrix-vector kernel (1-4 rows), the unsliced weight-streaming
// kernel (few rows and features enough to give every compute unit two waves) and the tiles fitted to the token count.
static int launch_one_problem(const GemmArgs& g, const GemmGroup& grp, const RowMap* rows, int wlayout, int batch, hipStream_t stream, bool* handled) {
    int rc = launch_gemv_f16(g, grp, rows, wlayout, batch, stream, handled);
    if (*handled) return rc;
    rc = launch_gemm_skinny_f16(g, grp, rows, wlayout, batch, stream, handled);
    if (*handled) return rc;
    return launch_gemm_tiles_f16(g, grp, rows, wlayout, batch, stream, handled);
}

static int gemm_f16_dispatch(GemmArgs g, int wlayout, int batch, hipStream_t stream) {
    if (g.M == 0 || g.N == 0 || batch == 0) return LG_OK;
    if (g.K == 0) { set_error("gemm: k == 0 is not supported"); return LG_ERR_INVALID; }
    bool handled = false;
    const GemmGroup one = single_group(g);
    int rc = launch_one_problem(g, one, nullptr, wlayout, batch, stream, &handled);
    if (handled) return rc;
    rc = launch_gemm_skinny_sliced_f16(g, wlayout, batch, stream, &handled);
    if (handled) return rc;
    dim3 grid((g.N + GB_N - 1) / GB_N, (g.M + GB_M - 1) / GB_M, batch);
    if (grid.y > 65535 || grid.z > 65535) { set_error("gemm: problem too large for the generic grid"); return LG_ERR_INVALID; }
    if (wlayout == W_TILED) launch_generic_epi<W_TILED>(g, grid, stream);
    else if (wlayout == W_NK) launch_generic_epi<W_NK>(g, grid, stream);
    else launch_generic_epi<W_KN>(g, grid, stream);
    return check_launch("gemm_f16");
}

// ---------------------------------------------------------------------------------------------------
// fp32 generic kernel (plumbing configuration): 64x64x16 tiles, 256 threads, 4x4 outputs per thread
// ---------------------------------------------------------------------------------------------------
template <int WL>
__global__ __launch_bounds__(256) void gemm_f32_generic(GemmArgsF32 g) {
    __shared__ float As[16][64 + 4];  // [k][m]
    __shared__ float Bs[16][64 + 4];  // [k][n]
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;  // 16x16 threads, 4x4 outputs each
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const float* X = g.X + (int64_t)blockIdx.z * g.strideX;
    const float* W = g.W + (int64_t)blockIdx.z * g.strideW;
    float* Y = g.Y + (int64_t)blockIdx.z * g.strideY;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < g.K; k0 += 16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + 256 * i;  // 1024 elements per tile
            {
                const int r = e >> 4, kk = e & 15;  // X: 64 rows x 16 k, k fastest
                const int m = m0 + r, k = k0 + kk;
                As[kk][r] = (m < g.M && k < g.K) ? X[(int64_t)m * g.ldx + k] : 0.f;
            }
            if (WL == W_NK) {
                const int r = e >> 4, kk = e & 15;
                const int n = n0 + r, k = k0 + kk;
                Bs[kk][r] = (n < g.N && k < g.K) ? W[(int64_t)n * g.ldw + k] : 0.f;
            } else {
                const int kk = e >> 6, c = e & 63;  // W: 16 k x 64 n, n fastest
                const int n = n0 + c, k = k0 + kk;
                Bs[kk][c] = (n < g.N && k < g.K) ? W[(int64_t)k * g.ldw + n] : 0.f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
            if (m < g.M && n < g.N) Y[(int64_t)m * g.ldy + n] = acc[i][j];
        }
}

// ---------------------------------------------------------------------------------------------------
// fp32 on the matrix cores: 128 x 128 x 16 tiles, 8 waves (2 x 4), v_mfma_f32_16x16x4_f32
// ---------------------------------------------------------------------------------------------------
// The reference instantiates every layer for float through cublasGemmEx(..., CUDA_R_32F, ...) (context.h:49-55,
// linear.h:47-49,99-101).  A wave owns 64 x 32 outputs = 4 x 2 MFMA tiles; operands are swapped as in the fp16 kernels (the weight
// tile is the A operand), so a lane ends up with 4 consecutive output features of one token row:
// acc[i][j][v] = Y[token 16 i + lane % 16][feature 16 j + 4 (lane / 16) + v].  An output is summed as in gemm_f32.hpp, quarter of K by
// quarter, with the same instruction and the same k in each of its slots, so that the bits of a row do not depend on which of
// the two kernels its call takes; that costs a second set of accumulators, and 8 waves instead of 4 leave room for it with four
// waves on a SIMD.  Rows of 16 k sit in LDS 20 floats apart: a lane's four k are one 16-byte read, and the 16 rows of such a read
// cover all banks once.  [K, N] weights stay k-major, 132 floats a row: the four k of a read are 16 banks apart.  Two buffers, one
// barrier for every 16 k.  Against one sum over the whole of K in 4 waves of half the registers, microseconds: 800 x 4096 x 1024
// 88 -> 81, 1600 x 4096 x 1024 148 -> 145, 4096 x 1024 x 1024 80 -> 83, 4096 x 4096 x 1024 263 -> 285 (120 TFLOP/s: two workgroups share
// a compute unit, not three), 64 times 512 x 512 x 64 29 -> 33; error against 64-bit sums half as large (K = 1024: 5.7e-7 -> 2.9e-7).
constexpr int SB_M = 128, SB_N = 128, SB_K = SF_K, SB_ROW = SB_K + 4, SB_PITCH = 128 + 4, SB_THREADS = 512;

template <int WL, bool ALIGNED>
__global__ __launch_bounds__(SB_THREADS, 4) void gemm_f32_mfma(GemmArgsF32 g) {
    constexpr int W_TILE = WL == W_NK ? SB_N * SB_ROW : SB_K * SB_PITCH;
    __shared__ __attribute__((aligned(16))) float Xs[2][SB_M * SB_ROW];
    __shared__ __attribute__((aligned(16))) float Ws[2][W_TILE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    const int m0 = blockIdx.y * SB_M, n0 = blockIdx.x * SB_N;
    const float* X = g.X + (int64_t)blockIdx.z * g.strideX;
    const float* W = g.W + (int64_t)blockIdx.z * g.strideW;
    float* Y = g.Y + (int64_t)blockIdx.z * g.strideY;

    // 4 consecutive floats p[0..3] with `valid` of them inside the matrix
    auto load4f = [](const float* p, int valid) {
        float4_t r = {0.f, 0.f, 0.f, 0.f};
        if (ALIGNED && valid >= 4) return *reinterpret_cast<const float4_t*>(p);
        if (valid > 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i < valid) r[i] = p[i];
        }
        return r;
    };
    float4_t rx, rw;
    const int row = tid >> 2, kq = (tid & 3) * 4;    // rows of 16 k: thread = (row, quarter of the k)
    const int kr = tid >> 5, ns = (tid & 31) * 4;    // [K, N] weights: 16 k-rows x 128 features; thread = (k, 4 consecutive features)
    auto gload = [&](int k0) {
        rx = load4f(X + (int64_t)(m0 + row) * g.ldx + k0 + kq, m0 + row < g.M ? g.K - k0 - kq : 0);
        if (WL == W_NK) rw = load4f(W + (int64_t)(n0 + row) * g.ldw + k0 + kq, n0 + row < g.N ? g.K - k0 - kq : 0);
        else rw = load4f(W + (int64_t)(k0 + kr) * g.ldw + n0 + ns, k0 + kr < g.K ? g.N - n0 - ns : 0);
    };
    auto lstore = [&](int buf) {
        *reinterpret_cast<float4_t*>(&Xs[buf][row * SB_ROW + kq]) = rx;
        *reinterpret_cast<float4_t*>(WL == W_NK ? &Ws[buf][row * SB_ROW + kq] : &Ws[buf][kr * SB_PITCH + ns]) = rw;
    };

    const int l16 = lane & 15, lk = lane >> 4;
    float4_t acc[4][2], total[4][2];
    const int chunks = (g.K + SB_K - 1) / SB_K, quarter = f32_quarter(g.K);
    int c = 0;
    auto chunk = [&](auto first, float4_t (&sum)[4][2]) {  // first of its quarter: the sums start from zero
        const int buf = c & 1;
        lstore(buf);
        __syncthreads();  // the other buffer is refilled after the next one: every wave is done with it by then
        if (++c < chunks) gload(c * SB_K);
        float4_t x[4], w[2];  // k 4 lk .. 4 lk + 3 of row 16 i + l16
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const float4_t*>(&Xs[buf][(wm * 64 + i * 16 + l16) * SB_ROW + 4 * lk]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (WL == W_NK) {
                w[j] = *reinterpret_cast<const float4_t*>(&Ws[buf][(wn * 32 + j * 16 + l16) * SB_ROW + 4 * lk]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) w[j][r] = Ws[buf][(4 * lk + r) * SB_PITCH + wn * 32 + j * 16 + l16];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float4_t before = decltype(first)::value && r == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : sum[i][j];
                    sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][r], x[i][r], before, 0, 0, 0);
                }
    };
    gload(0);
    chunk(std::true_type{}, total);
#pragma unroll 1
    while (c < quarter) chunk(std::false_type{}, total);
#pragma unroll 1
    for (int q = 1; q < SF_WAVES; ++q) {
        const int end = min(chunks, (q + 1) * quarter);
        if (c >= end) break;  // (a wave of gemm_f32.hpp without chunks adds zero)
        chunk(std::true_type{}, acc);
#pragma unroll 1
        while (c < end) chunk(std::false_type{}, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) total[i][j] += acc[i][j];
    }
    const bool vec_ok = ALIGNED && (g.ldy % 4 == 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + wm * 64 + i * 16 + l16;
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 32 + j * 16 + 4 * lk;
            float* p = Y + (int64_t)m * g.ldy + n;
            if (vec_ok && n + 3 < g.N) {
                *reinterpret_cast<float4_t*>(p) = total[i][j];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < g.N) p[r] = total[i][j][r];
            }
        }
    }
}

static int gemm_f32_dispatch(const GemmArgsF32& g, int wlayout, int batch, hipStream_t stream) {
    if (g.M == 0 || g.N == 0 || batch == 0) return LG_OK;
    if (g.K == 0) { set_error("gemm: k == 0 is not supported"); return LG_ERR_INVALID; }
    // LG_GEMM_F32_VALU=1 in the environment (read once) selects the vector-ALU tile kernel instead: a cross-check for tests
    static const bool valu = [] { const char* e = getenv("LG_GEMM_F32_VALU"); return e && atoi(e) != 0; }();
    if (!valu) {
        dim3 grid((g.N + SB_N - 1) / SB_N, (g.M + SB_M - 1) / SB_M, batch);
        if (grid.y > 65535 || grid.z > 65535) { set_error("gemm: problem too large for the grid"); return LG_ERR_INVALID; }
        const bool aligned = aligned16(g.X) && aligned16(g.W) && aligned16(g.Y) && (g.ldx % 4 == 0) && (g.ldw % 4 == 0) &&
                             (g.strideX % 4 == 0) && (g.strideW % 4 == 0) && (g.strideY % 4 == 0);
        bool handled = false;
        int rc = launch_gemm_f32_split(g, wlayout, batch, aligned, stream, &handled);
        if (handled) return rc;
        rc = launch_gemm_f32_direct(g, wlayout, batch, aligned, stream, &handled);
        if (handled) return rc;
        if (wlayout == W_NK) {
            if (aligned) hipLaunchKernelGGL((gemm_f32_mfma<W_NK, true>), grid, dim3(SB_THREADS), 0, stream, g);
            else hipLaunchKernelGGL((gemm_f32_mfma<W_NK, false>), grid, dim3(SB_THREADS), 0, stream, g);
        } else {
            if (aligned) hipLaunchKernelGGL((gemm_f32_mfma<W_KN, true>), grid, dim3(SB_THREADS), 0, stream, g);
            else hipLaunchKernelGGL((gemm_f32_mfma<W_KN, false>), grid, dim3(SB_THREADS), 0, stream, g);
        }
        return check_launch("gemm_f32");
    }
    dim3 grid((g.N + 63) / 64, (g.M + 63) / 64, batch);
    if (grid.y > 65535 || grid.z > 65535) { set_error("gemm: problem too large for the generic grid"); return LG_ERR_INVALID; }
    if (wlayout == W_NK) hipLaunchKernelGGL((gemm_f32_generic<W_NK>), grid, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((gemm_f32_generic<W_KN>), grid, dim3(256), 0, stream, g);
    return check_launch("gemm_f32");
}

// cuBLAS column-major arguments -> row-major problem; returns LG_OK or sets the error text
static int check_blas_args(const char* what, int transa, int transb, int m, int n, int k, const void* A, int lda,
                           const void* B, int ldb, const void* C, int ldc, int batch) {
    if (transb != 0 || (transa != 0 && transa != 1 && transa != LG_OP_TILED)) { set_error("%s: only (N,N), (T,N) and (tiled,N) are supported", what); return LG_ERR_INVALID; }
    if (m < 0 || n < 0 || k < 0 || batch < 0) { set_error("%s: negative dimension", what); return LG_ERR_INVALID; }
    if (m == 0 || n == 0 || batch == 0) return LG_OK;
    if (!A || !B || !C) { set_error("%s: null pointer", what); return LG_ERR_INVALID; }
    if (transa == LG_OP_TILED && (m % 16 != 0 || k % 32 != 0 || lda != k || batch > 1 || ((uintptr_t)A & 15u))) {
        set_error("%s: tiled weights need features %% 16 == 0, k %% 32 == 0, lda == k, a 16-byte aligned pointer and no batch (m=%d k=%d lda=%d)", what, m, k, lda);
        return LG_ERR_INVALID;
    }
    const int min_lda = transa ? k : m;
    if (lda < (min_lda > 1 ? min_lda : 1) || ldb < (k > 1 ? k : 1) || ldc < (m > 1 ? m : 1)) {
        set_error("%s: leading dimension too small (lda=%d ldb=%d ldc=%d for m=%d n=%d k=%d)", what, lda, ldb, ldc, m, n, k);
        return LG_ERR_INVALID;
    }
    return LG_OK;
}

}  // namespace lg

using namespace lg;

extern "C" {

int lg_gemm_strided_batched_f16(int transa, int transb, int m, int n, int k, const void* A, int lda, int64_t strideA,
                                const void* B, int ldb, int64_t strideB, void* C, int ldc, int64_t strideC, int batch,
                                void* stream) {
    int rc = check_blas_args("gemm_f16", transa, transb, m, n, k, A, lda, B, ldb, C, ldc, batch);
    if (rc) return rc;
    GemmArgs g;
    g.M = n; g.N = m; g.K = k;
    g.X = (const half_t*)B; g.ldx = ldb; g.strideX = strideB;
    g.W = (const half_t*)A; g.ldw = lda; g.strideW = strideA;
    g.Y = (half_t*)C; g.ldy = ldc; g.strideY = strideC;
    g.epi = Epilogue{LG_EPI_NONE, nullptr, 0, 0, 0, 0};
    return gemm_f16_dispatch(g, transa == LG_OP_TILED ? W_TILED : (transa ? W_NK : W_KN), batch, (hipStream_t)stream);
}

int lg_gemm_f16(int transa, int transb, int m, int n, int k, const void* A, int lda, const void* B, int ldb, void* C,
                int ldc, void* stream) {
    return lg_gemm_strided_batched_f16(transa, transb, m, n, k, A, lda, 0, B, ldb, 0, C, ldc, 0, 1, stream);
}

int lg_gemm_fused_f16(int transa, int m, int n, int k, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                      int epilogue, const void* bias, int epi_arg0, int epi_arg1, int epi_arg2, void* stream) {
    int rc = check_blas_args("gemm_fused_f16", transa, 0, m, n, k, A, lda, B, ldb, C,
                             epilogue == LG_EPI_BIAS_HEADS ? (m > 1 ? m : 1) : (epilogue == LG_EPI_BIAS_GEGLU ? (ldc < m / 2 ? 0 : m) : ldc), 1);
    if (rc) return rc;
    if (epilogue != LG_EPI_BIAS_GEGLU && (epilogue < LG_EPI_NONE || epilogue > LG_EPI_BIAS_HEADS)) { set_error("gemm_fused_f16: unknown epilogue %d", epilogue); return LG_ERR_INVALID; }
    if (epilogue != LG_EPI_NONE && !bias) { set_error("gemm_fused_f16: epilogue needs a bias"); return LG_ERR_INVALID; }
    if (epilogue == LG_EPI_BIAS_GEGLU && m % 32 != 0) { set_error("gemm_fused_f16: the GeGLU epilogue needs features %% 32 == 0 (gate and up interleaved in groups of 16)"); return LG_ERR_INVALID; }
    if (epilogue == LG_EPI_BIAS_HEADS) {
        const int seq = epi_arg0, d = epi_arg1;
        if (seq <= 0 || d <= 0 || m % d != 0 || n % seq != 0 || d % 4 != 0 || ldc < seq ||
            (epi_arg2 != 0 && epi_arg2 < m / d)) {
            set_error("gemm_fused_f16: heads epilogue needs seq | tokens, size_per_head | features, size_per_head %% 4 == 0, "
                      "ldc (rows per head slot) >= seq, heads_total >= features / size_per_head");
            return LG_ERR_INVALID;
        }
        if (epi_arg2 == 0) epi_arg2 = m / d;
    }
    GemmArgs g;
    g.M = n; g.N = m; g.K = k;
    g.X = (const half_t*)B; g.ldx = ldb; g.strideX = 0;
    g.W = (const half_t*)A; g.ldw = lda; g.strideW = 0;
    g.Y = (half_t*)C; g.ldy = ldc; g.strideY = 0;
    g.epi = Epilogue{epilogue, (const half_t*)bias, epi_arg0, epi_arg1, epi_arg2, 0};
    return gemm_f16_dispatch(g, transa == LG_OP_TILED ? W_TILED : (transa ? W_NK : W_KN), 1, (hipStream_t)stream);
}

// mode: -1 = choose the plan, 1 = one launch if the kernels allow it (a sub-group of a plan)
static int gemm_fused_grouped_f16_impl(int mode, int transa, int m, int n, int k, int count, const void* const* A, int lda, const void* B, int ldb,
                                       void* const* C, const int* ldc, int epilogue, const void* const* bias, int epi_arg0, int epi_arg1,
                                       int epi_arg2, void* stream) {
    if (count < 1 || count > LG_MAX_GROUP || !A || !C || !ldc || (epilogue != LG_EPI_NONE && !bias)) {
        set_error("gemm_fused_grouped_f16: count must be 1..%d and the pointer arrays non-null", LG_MAX_GROUP);
        return LG_ERR_INVALID;
    }
    // One launch for the group, member by member, or in pieces: whichever the kernels' own estimate says is the fastest.  All ways
    // give the same bits above 64 rows, and at any count with weights [in, out] (the number of K-slices does not depend on it); at
    // 5-64 rows with weights [out, in] the weight-streaming kernel may take a group and not its members, in another order of the sum.
    GemmGroup grp{};
    grp.count = count;
    bool one_launch = m > 0 && n > 0 && k > 0 && count > 1 && B != nullptr;
    for (int i = 0; i < count; ++i) {
        grp.W[i] = (const half_t*)A[i];
        grp.Y[i] = (half_t*)C[i];
        grp.bias[i] = epilogue != LG_EPI_NONE ? (const half_t*)bias[i] : nullptr;
        grp.ldy[i] = ldc[i];
        if (!A[i] || !C[i] || (epilogue != LG_EPI_NONE && !bias[i])) one_launch = false;  // the plain call reports it
    }
    const int wl = transa == LG_OP_TILED ? W_TILED : (transa ? W_NK : W_KN);
    // a member of the group as a problem of its own, with some of its features
    auto member = [&](int features) {
        GemmArgs g{};
        g.M = n; g.N = features; g.K = k;
        g.X = (const half_t*)B; g.ldx = ldb;
        g.W = grp.W[0]; g.ldw = lda;
        g.Y = grp.Y[0]; g.ldy = grp.ldy[0];
        g.epi = Epilogue{epilogue, grp.bias[0], epi_arg0, epi_arg1, epi_arg2, 0};
        return g;
    };
    const int cus = stream_info((hipStream_t)stream).cus;
    // Fragment blocks and few rows: member by member where the weight-streaming kernel takes a member but not the group, whose features
    // are too many for one wave a feature tile (three times 12288 x 12288, 11 rows: 142 us, as tiles 159; x 4096, 32 rows: 60 and 67).
    // At 48 rows, with more features or with rows of [out, in], the tiles are level or ahead (x 4096, 48 rows: 63 and 59; 16384 x 4096, 11
    // rows: 80 and 68; [out, in], 12288 x 4096, 11 rows: 71 and 64).
    if (mode < 0 && one_launch && wl == W_TILED && n <= 32 && m <= 12288)
        one_launch = !skinny_takes_group(member(m), 1, wl, cus) || skinny_takes_group(member(m), count, wl, cus);
    if (mode < 0 && one_launch && n > 64) {
        constexpr double kLaunch = 1.5;  // microseconds between two launches
        auto plan = [&](int members, int features) {
            GemmGroup sub = grp;
            sub.count = members;
            return plan_gemm_tiles_f16(member(features), sub, wl, 1, (hipStream_t)stream);
        };
        const TilePlan together = plan(count, m), apart = plan(1, m);
        const double cost_apart = count * (apart.cost + kLaunch);
        // (in pairs of slices three of a kind are one launch wherever the plan has them, which the estimate of four slices alone, on the low
        // side, would not choose: 80 rows, fragment blocks of three times 6144 x 12288, in a layer 105 us, apart 130)
        if (together.nsplit == 0 || (!together.pairs && apart.nsplit != 0 && cost_apart < together.cost)) one_launch = false;
        // A third way for groups that are many full rounds of workgroups plus a remainder (Q, K, V of 4096 rows x 6144 features: 72
        // columns of 256-wide tiles, 16 columns to a round of 256 workgroups, 8 left over): the members before the last as one
        // launch of whole rounds, the last member's leading features as whole rounds too, and its remaining features as one round
        // of narrower tiles -- instead of six rounds of 192-wide tiles (4.6-6.6 % faster, measured).  Pieces are addressed like any
        // feature sub-range.  Only where the order of a sum over k does not depend on the feature's place in its launch.
        int split_at = 0;   // feature at which the last member is cut (0: no such plan)
        const int tiles_m = (n + 255) / 256;
        const bool range_ok = epilogue == LG_EPI_NONE || epilogue == LG_EPI_BIAS || epilogue == LG_EPI_BIAS_GELU ||
                              (epilogue == LG_EPI_BIAS_HEADS && epi_arg1 > 0 && 256 % epi_arg1 == 0);
        if (range_ok && n >= kSequentialRows && apart.nsplit == 1 && m % 256 == 0 && cus % tiles_m == 0 && (transa != LG_OP_TILED || lda == k)) {
            const int cols = m / 256, per_round = cus / tiles_m, rem = (count * cols) % per_round;
            if (rem > 0 && rem < cols && ((count - 1) * cols) % per_round == 0 && (cols - rem) % per_round == 0) {
                const TilePlan lead = plan(count - 1, m), body = plan(1, (cols - rem) * 256), tail = plan(1, rem * 256);
                const double pieces = lead.cost + body.cost + tail.cost + 3 * kLaunch;
                if (lead.nsplit == 1 && body.nsplit == 1 && tail.nsplit == 1 && pieces < together.cost && pieces < cost_apart) split_at = (cols - rem) * 256;
            }
        }
        // LG_GEMM_GROUP=1|0 in the environment (read once) forces one launch / member by member: a measurement knob
        static const int forced = [] { const char* e = getenv("LG_GEMM_GROUP"); return e ? atoi(e) : -1; }();
        if (forced == 0) { one_launch = false; split_at = 0; }
        else if (forced == 1) { one_launch = true; split_at = 0; }
        if (split_at > 0) {
            int rc = count - 1 > 1 ? gemm_fused_grouped_f16_impl(1, transa, m, n, k, count - 1, A, lda, B, ldb, C, ldc, epilogue, bias, epi_arg0, epi_arg1,
                                                                 epilogue == LG_EPI_BIAS_HEADS && epi_arg2 == 0 ? m / epi_arg1 : epi_arg2, stream)
                                   : lg_gemm_fused_f16(transa, m, n, k, A[0], lda, B, ldb, C[0], ldc[0], epilogue, epilogue != LG_EPI_NONE ? bias[0] : nullptr,
                                                       epi_arg0, epi_arg1, epi_arg2, stream);
            if (rc) return rc;
            const int last = count - 1;
            const int heads_total = epilogue == LG_EPI_BIAS_HEADS ? (epi_arg2 ? epi_arg2 : m / epi_arg1) : epi_arg2;
            const int cut[3] = {0, split_at, m};
            for (int piece = 0; piece < 2; ++piece) {
                const int f0 = cut[piece], f1 = cut[piece + 1];
                // features [f0, f1) of the last member: rows f0.. of an [out, in] weight (row-major or in fragment blocks, where
                // feature tile t starts 16 t k elements in), columns f0.. of an [in, out] one; heads f0 / d .. of a
                // head-transposed destination, columns f0.. of a plain one
                const int64_t w_off = transa == 0 ? (int64_t)f0 : (int64_t)f0 * (transa == LG_OP_TILED ? k : lda);
                const int64_t c_off = epilogue == LG_EPI_BIAS_HEADS ? (int64_t)(f0 / epi_arg1) * ldc[last] * epi_arg1 : (int64_t)f0;
                rc = lg_gemm_fused_f16(transa, f1 - f0, n, k, (const half_t*)A[last] + w_off, lda, B, ldb, (half_t*)C[last] + c_off, ldc[last], epilogue,
                                       epilogue != LG_EPI_NONE ? (const void*)((const half_t*)bias[last] + f0) : nullptr, epi_arg0, epi_arg1, heads_total, stream);
                if (rc) return rc;
            }
            return LG_OK;
        }
    }
    if (one_launch) {
        // same argument checks as the plain entry, member by member, before anything is launched
        for (int i = 0; i < count; ++i) {
            int rc = check_blas_args("gemm_fused_grouped_f16", transa, 0, m, n, k, A[i], lda, B, ldb, C[i],
                                     epilogue == LG_EPI_BIAS_HEADS ? (m > 1 ? m : 1) : ldc[i], 1);
            if (rc) return rc;
        }
        if (epilogue < LG_EPI_NONE || epilogue > LG_EPI_BIAS_HEADS) { set_error("gemm_fused_grouped_f16: unknown epilogue %d", epilogue); return LG_ERR_INVALID; }
        int heads_total = epi_arg2;
        bool ok = true;
        if (epilogue == LG_EPI_BIAS_HEADS) {
            const int seq = epi_arg0, d = epi_arg1;
            ok = seq > 0 && d > 0 && m % d == 0 && n % seq == 0 && d % 4 == 0 && (epi_arg2 == 0 || epi_arg2 >= m / d);
            for (int i = 0; i < count && ok; ++i) ok = ldc[i] >= seq;
            if (ok && heads_total == 0) heads_total = m / d;
        }
        if (ok) {
            GemmArgs g;
            g.M = n; g.N = m; g.K = k;
            g.X = (const half_t*)B; g.ldx = ldb; g.strideX = 0;
            g.W = grp.W[0]; g.ldw = lda; g.strideW = 0;
            g.Y = grp.Y[0]; g.ldy = grp.ldy[0]; g.strideY = 0;
            g.epi = Epilogue{epilogue, grp.bias[0], epi_arg0, epi_arg1, heads_total, 0};
            bool handled = false;
            int rc = launch_one_problem(g, grp, nullptr, wl, 1, (hipStream_t)stream, &handled);
            if (handled) return rc;
        }
    }
    for (int i = 0; i < count; ++i) {
        int rc = lg_gemm_fused_f16(transa, m, n, k, A[i], lda, B, ldb, C[i], ldc[i], epilogue, epilogue != LG_EPI_NONE ? bias[i] : nullptr,
                                   epi_arg0, epi_arg1, epi_arg2, stream);
        if (rc) return rc;
    }
    return LG_OK;
}

int lg_gemm_fused_grouped_f16(int transa, int m, int n, int k, int count, const void* const* A, int lda, const void* B, int ldb,
                              void* const* C, const int* ldc, int epilogue, const void* const* bias, int epi_arg0, int epi_arg1,
                              int epi_arg2, void* stream) {
    return gemm_fused_grouped_f16_impl(-1, transa, m, n, k, count, A, lda, B, ldb, C, ldc, epilogue, bias, epi_arg0, epi_arg1, epi_arg2, stream);
}

int lg_gemm_fused_grouped_rows_f16(int transa, int m, int n, int k, int count, const void* const* A, int lda, const void* B, int ldb,
                                   void* const* C, const int* ldc, const void* const* bias, int size_per_head, int heads_total,
                                   const int* use_rows, const int* slot, const int* pos, void* stream) {
    const int d = size_per_head;
    if (count < 1 || count > LG_MAX_GROUP || !A || !C || !ldc || !bias || !use_rows) {
        set_error("gemm_fused_grouped_rows_f16: count must be 1..%d and the pointer arrays non-null", LG_MAX_GROUP);
        return LG_ERR_INVALID;
    }
    if (m < 0 || n < 0 || k < 0 || n > LG_ROWMAP_MAX) { set_error("gemm_fused_grouped_rows_f16: at most %d token rows (n = %d)", LG_ROWMAP_MAX, n); return LG_ERR_INVALID; }
    if (m == 0 || n == 0) return LG_OK;
    if (d <= 0 || m % d != 0 || d % 4 != 0 || heads_total < m / d) {
        set_error("gemm_fused_grouped_rows_f16: size_per_head must divide the features and be a multiple of 4, heads_total >= features / size_per_head");
        return LG_ERR_INVALID;
    }
    bool any_rows = false;
    for (int i = 0; i < count; ++i) any_rows = any_rows || use_rows[i] != 0;
    if (any_rows && (!slot || !pos)) { set_error("gemm_fused_grouped_rows_f16: null slot / pos array"); return LG_ERR_INVALID; }
    RowMap rm{};
    for (int r = 0; r < n && any_rows; ++r) {
        if (slot[r] < 0 || pos[r] < 0) { set_error("gemm_fused_grouped_rows_f16: token row %d: slot %d, pos %d", r, slot[r], pos[r]); return LG_ERR_INVALID; }
        rm.slot[r] = slot[r];
        rm.pos[r] = pos[r];
    }
    GemmGroup grp{};
    grp.count = count;
    for (int i = 0; i < count; ++i) {
        int rc = check_blas_args("gemm_fused_grouped_rows_f16", transa, 0, m, n, k, A[i], lda, B, ldb, C[i], m > 1 ? m : 1, 1);
        if (rc) return rc;
        if (!bias[i]) { set_error("gemm_fused_grouped_rows_f16: null bias"); return LG_ERR_INVALID; }
        if (ldc[i] < 1) { set_error("gemm_fused_grouped_rows_f16: ldc (rows per head slot) must be >= 1"); return LG_ERR_INVALID; }
        for (int r = 0; r < n && use_rows[i]; ++r)
            if (pos[r] >= ldc[i]) { set_error("gemm_fused_grouped_rows_f16: token row %d: pos %d outside the %d rows of a head slot", r, pos[r], ldc[i]); return LG_ERR_INVALID; }
        grp.W[i] = (const half_t*)A[i];
        grp.Y[i] = (half_t*)C[i];
        grp.bias[i] = (const half_t*)bias[i];
        grp.ldy[i] = ldc[i];
        grp.rows[i] = use_rows[i] ? 1 : 0;
    }
    {
        GemmArgs g;
        g.M = n; g.N = m; g.K = k;
        g.X = (const half_t*)B; g.ldx = ldb; g.strideX = 0;
        g.W = grp.W[0]; g.ldw = lda; g.strideW = 0;
        g.Y = grp.Y[0]; g.ldy = grp.ldy[0]; g.strideY = 0;
        g.epi = Epilogue{LG_EPI_BIAS_HEADS_ROWS, grp.bias[0], 1, d, heads_total, grp.rows[0]};
        bool handled = false;
        int rc = launch_one_problem(g, grp, &rm, transa == LG_OP_TILED ? W_TILED : (transa ? W_NK : W_KN), 1, (hipStream_t)stream, &handled);
        if (handled) return rc;
    }
    // anything the weight-streaming kernels do not take: plain calls, one per member -- and one per token row for a member
    // whose rows go to their own places
    for (int i = 0; i < count; ++i) {
        if (!use_rows[i]) {
            int rc = lg_gemm_fused_f16(transa, m, n, k, A[i], lda, B, ldb, C[i], ldc[i], LG_EPI_BIAS_HEADS, bias[i], 1, d, heads_total, stream);
            if (rc) return rc;
            continue;
        }
        for (int r = 0; r < n; ++r) {
            half_t* dst = (half_t*)C[i] + ((int64_t)slot[r] * heads_total * ldc[i] + pos[r]) * d;
            int rc = lg_gemm_fused_f16(transa, m, 1, k, A[i], lda, (const half_t*)B + (int64_t)r * ldb, ldb, dst, ldc[i], LG_EPI_BIAS_HEADS,
                                       bias[i], 1, d, heads_total, stream);
            if (rc) return rc;
        }
    }
    return LG_OK;
}

int lg_gemm_strided_batched_f32(int transa, int transb, int m, int n, int k, const float* A, int lda, int64_t strideA,
                                const float* B, int ldb, int64_t strideB, float* C, int ldc, int64_t strideC, int batch,
                                void* stream) {
    if (transa == LG_OP_TILED) { set_error("gemm_f32: tiled weights are an fp16 layout"); return LG_ERR_INVALID; }
    int rc = check_blas_args("gemm_f32", transa, transb, m, n, k, A, lda, B, ldb, C, ldc, batch);
    if (rc) return rc;
    GemmArgsF32 g;
    g.M = n; g.N = m; g.K = k;
    g.X = B; g.ldx = ldb; g.strideX = strideB;
    g.W = A; g.ldw = lda; g.strideW = strideA;
    g.Y = C; g.ldy = ldc; g.strideY = strideC;
    return gemm_f32_dispatch(g, transa ? W_NK : W_KN, batch, (hipStream_t)stream);
}

int lg_gemm_f32(int transa, int transb, int m, int n, int k, const float* A, int lda, const float* B, int ldb, float* C,
                int ldc, void* stream) {
    return lg_gemm_strided_batched_f32(transa, transb, m, n, k, A, lda, 0, B, ldb, 0, C, ldc, 0, 1, stream);
}

}  // extern "C"
