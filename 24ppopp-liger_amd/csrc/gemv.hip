// gemv.hip -- weight-streaming fp16 matrix-vector kernel for one to four token rows (batch-1 decode) on gfx950.
//
//   Y[M, N] = X[M, K] * W^T with W stored [N, K], M <= 4.
// Every weight byte is used for 2*M flops, so the kernel is nothing but an HBM stream of W with the arithmetic on the
// vector ALUs (v_dot2_f32_f16); what matters is how the stream is issued:
//   * one block per compute unit, which stays until the end; its waves (8 where that deals the features evenly) own a feature at a
//     time and walk its weight row from one end to the other, 4 KiB at a time, and then the row of the next feature: a wave is one
//     sequential stream, and a compute unit has 8 x 4 KiB on their way, which is all it can have;
//   * the loads are marked non-temporal where the weights are more than the caches keep;
//   * a feature's row is summed by one wave, so there are no K-slices, no fp32 partials and no second kernel: lanes accumulate in
//     fp32, one butterfly sum per output at the end, epilogue (bias / GELU / head-transposed store) applied in place.  The loads of
//     the next feature are on their way by then;
//   * the M token rows are staged once per block in LDS (M * K * 2 bytes); the first weight loads are issued before that.
// Blocks of 4 waves that each walked 4 rows side by side, as many as the features made, left HBM pages after every KiB and drained at
// every change of blocks: with weights cycled through memory, in microseconds,
// 16384 x 12288 68.3 -> 60.7 (6.63 TB/s), 12288 x 6144 27.0 -> 25.1, 4096 x 4096 9.8 -> 8.5, 1024 x 4096 6.4 -> 4.7; at 4 token rows 12288 x 16384
// 72.5 -> 63.8 (in gemm_skinny.hip before, as the rows did not fit the LDS share of one block of several), 4096 x 4096 13.5 -> 10.2.
// Each output is one fixed-order fp32 sum (four partial sums per lane over k in an order fixed by the feature, then a butterfly; with one per
// lane 0.17 % of the outputs at K = 12288 were not the fp16 nearest to the 64-bit sum, with four 0.10 %, at the same time),
// independent of the other token rows and of the other members of a group.
#include <limits.h>
#include <stdlib.h>

#include "gemm_common.hpp"

namespace lg {

constexpr int GV_U = 4;             // k-steps in flight
constexpr int GV_KSTEP = 512;       // halves per wave instruction (64 lanes x 8)
constexpr int GV_MAX_WAVES = 12;
constexpr int GV_MAX_LDS = 160 * 1024;   // bytes of staged X per block

__device__ __forceinline__ float dot8(half8_t w, half8_t x, float acc) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
        acc = __builtin_amdgcn_fdot2(half2_t{w[2 * p], w[2 * p + 1]}, half2_t{x[2 * p], x[2 * p + 1]}, acc, false);
    return acc;
}

// MR = staged token rows (1, 2 or 4; rows >= M are zero); the members' features follow each other
template <int MR, int EPI, bool NT>
__global__ __launch_bounds__(GV_MAX_WAVES * 64) void gemv_nk_kernel(GemmArgs g, GemmGroup members, RowMap rm) {
    extern __shared__ __attribute__((aligned(16))) half_t xs[];  // [MR][K]
    const int tid = threadIdx.x, lane = tid & 63, threads = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = g.K, features = g.N * members.count, step = gridDim.x * (threads >> 6);
    const int groups = K / (GV_KSTEP * GV_U);  // the launcher guarantees whole groups
    auto load = [](const half_t* p) {
        const half8_t* v = reinterpret_cast<const half8_t*>(p);
        return NT ? __builtin_nontemporal_load(v) : *v;
    };
    // the weight row of a feature (those beyond the last are read as the last and never stored), and the group its walk starts at: with
    // a power-of-two row pitch (K = 16384) rows walked in phase would hit the same memory channels at the same time
    auto row_of = [&](int f) {
        const int c = min(f, features - 1), member = c / g.N;
        return (members.count > 1 ? members.W[member] : g.W) + (int64_t)(c - member * g.N) * g.ldw + lane * 8;
    };
    auto start_of = [&](int f) { return f % g.N % groups; };

    int f = blockIdx.x * (threads >> 6) + wave;
    const half_t* row = row_of(f);
    int grp = start_of(f);
    half8_t wv[GV_U];  // the stream starts before X is staged
#pragma unroll
    for (int u = 0; u < GV_U; ++u) wv[u] = load(row + (int64_t)(grp * GV_U + u) * GV_KSTEP);

    for (int v = tid; v < MR * (K / 8); v += threads) {
        const int r = v / (K / 8), c = v % (K / 8);
        half8_t val = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
        if (r < g.M) val = *reinterpret_cast<const half8_t*>(g.X + (int64_t)r * g.ldx + c * 8);
        *reinterpret_cast<half8_t*>(&xs[r * K + c * 8]) = val;
    }
    __syncthreads();

    for (; f < features; f += step) {
        const int member = f / g.N, n = f - member * g.N;
        const half_t* bias = members.count > 1 ? members.bias[member] : g.epi.bias;
        const float b = EPI == LG_EPI_NONE ? 0.f : (float)bias[n];  // on its way before it is needed
        float acc[MR][GV_U];  // a sum for each piece of a group: shorter chains round less
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int u = 0; u < GV_U; ++u) acc[m][u] = 0.f;
        for (int it = 0; it < groups; ++it) {
            const int cur = grp;
            if (it + 1 < groups) {
                grp = grp + 1 == groups ? 0 : grp + 1;
            } else {
                row = row_of(f + step);
                grp = start_of(f + step);
            }
#pragma unroll
            for (int u = 0; u < GV_U; ++u) {
#pragma unroll
                for (int m = 0; m < MR; ++m)
                    acc[m][u] = dot8(wv[u], *reinterpret_cast<const half8_t*>(&xs[m * K + (cur * GV_U + u) * GV_KSTEP + lane * 8]), acc[m][u]);
                wv[u] = load(row + (int64_t)(grp * GV_U + u) * GV_KSTEP);
                asm volatile("" ::: "memory");  // the load stays where it is written: the others are on their way beside it
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float v = 0.f;
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            static_assert(GV_U == 4, "four partial sums");
            const float s = wave_sum((acc[m][0] + acc[m][1]) + (acc[m][2] + acc[m][3]));
            v = lane == m ? s : v;
        }
        if (lane >= g.M) continue;
        if (EPI != LG_EPI_NONE) v += b;
        if (EPI == LG_EPI_BIAS_GELU) v = gelu_tanh(v);
        half_t* const Y = members.count > 1 ? members.Y[member] : g.Y;
        const int64_t ldy = members.count > 1 ? members.ldy[member] : g.ldy;
        const int mapped = members.count > 1 ? members.rows[member] : g.epi.rows;
        Y[output_offset<EPI>(g.epi, ldy, mapped, lane, n, &rm)] = (half_t)v;
    }
}

int launch_gemv_f16(const GemmArgs& g, const GemmGroup& grp, const RowMap* rows, int wlayout, int batch, hipStream_t stream, bool* handled) {
    *handled = false;
    if (batch != 1 || wlayout != W_NK) return LG_OK;
    if (g.M <= 0 || g.M > 4 || g.N < 256 || (g.N % 4) || g.K < GV_KSTEP * GV_U || (g.K % (GV_KSTEP * GV_U))) return LG_OK;
    const int mr = g.M == 1 ? 1 : (g.M == 2 ? 2 : 4);
    const size_t smem = (size_t)mr * g.K * sizeof(half_t);
    if (smem > (size_t)GV_MAX_LDS) return LG_OK;
    if (!aligned16(g.X) || (g.ldx % 8) || (g.ldw % 8) || !group_aligned(g, grp)) return LG_OK;
    if (g.epi.kind == LG_EPI_BIAS_HEADS_ROWS && (!rows || g.M > LG_ROWMAP_MAX)) return LG_OK;
    if (g.epi.kind == LG_EPI_BIAS_GEGLU) return LG_OK;  // pairs features 16 apart: left to the tile kernels
    *handled = true;
    const RowMap rm = rows ? *rows : RowMap{};
    // waves of a block: as many as give no compute unit more features than the others, 8 if that is a tie
    const int cus = stream_info(stream).cus, features = g.N * grp.count;
    int waves = 1, most = INT_MAX;
    for (int w = 1; w <= GV_MAX_WAVES; ++w) {
        const int rounds = (features + cus * w - 1) / (cus * w), per_cu = rounds * w;
        if (per_cu < most || (per_cu == most && abs(w - 8) <= abs(waves - 8))) { most = per_cu; waves = w; }
    }
    // Weights of 64 MiB and more come from memory whatever was read before (a layer has several such), and the non-temporal hint is worth
    // 6-10 % there (12288 x 16384 67.3 -> 59.9 us; 12288 x 4096, 96 MiB, 19.3 -> 18.0, and 16.5 -> 17.3 where it is the only weight and
    // the memory-side cache holds it); below, what the caches still hold counts for more (4096 x 4096 8.5 -> 8.4, repeated 5.1 -> 7.4).
    const bool nt = (int64_t)features * g.K * (int64_t)sizeof(half_t) >= (int64_t)64 << 20;
    const dim3 grid((features + waves - 1) / waves < cus ? (features + waves - 1) / waves : cus), block(64 * waves);
#define LG_GV_NT(MR_, E_, NT_)                                                                                      \
    do {                                                                                                            \
        /* set once per instantiation; the initialisation of a function-local static is thread-safe */              \
        static const hipError_t attr_rc = hipFuncSetAttribute((const void*)gemv_nk_kernel<MR_, E_, NT_>, hipFuncAttributeMaxDynamicSharedMemorySize, GV_MAX_LDS); \
        (void)attr_rc;                                                                                              \
        hipLaunchKernelGGL((gemv_nk_kernel<MR_, E_, NT_>), grid, block, smem, stream, g, grp, rm);                  \
    } while (0)
#define LG_GV(MR_, E_)                       \
    do {                                     \
        if (nt) LG_GV_NT(MR_, E_, true);     \
        else LG_GV_NT(MR_, E_, false);       \
    } while (0)
#define LG_GV_MR(E_)                                 \
    switch (mr) {                                    \
        case 1: LG_GV(1, E_); break;                 \
        case 2: LG_GV(2, E_); break;                 \
        default: LG_GV(4, E_); break;                \
    }
    switch (g.epi.kind) {
        case LG_EPI_NONE: LG_GV_MR(LG_EPI_NONE); break;
        case LG_EPI_BIAS: LG_GV_MR(LG_EPI_BIAS); break;
        case LG_EPI_BIAS_GELU: LG_GV_MR(LG_EPI_BIAS_GELU); break;
        case LG_EPI_BIAS_HEADS_ROWS: LG_GV_MR(LG_EPI_BIAS_HEADS_ROWS); break;
        default: LG_GV_MR(LG_EPI_BIAS_HEADS); break;
    }
#undef LG_GV_MR
#undef LG_GV
#undef LG_GV_NT
    return check_launch("gemv_f16");
}

}  // namespace lg
