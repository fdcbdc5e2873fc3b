// gemm_mid.hpp -- fp16 GEMM whose tile is fitted to the token count (gfx950): everything from a few token rows to full prefill batches.
//
//   Y[M, N] = X[M, K] * W, any weight layout, fp32 accumulate, fused epilogue, groups; K % 64 == 0, N a multiple of the tile width.
//
// What bounds it depends on M.  Up to about 200 token rows it is the stream of weights from memory, above that the matrix pipes --
// provided that the tiles cover the token rows without much padding and that there is one workgroup for every compute unit.  So here:
//   * the tile is (32 MI) x (32 NJ), MI = 1 .. 8 and NJ = 3, 4, 6, 8, chosen per problem (gemm_mid.hip), and K may be sliced;
//   * a workgroup is 4 waves, one per SIMD, in a 2 x 2 grid: a wave multiplies (16 MI) x (16 NJ) outputs, which costs
//     (MI + NJ) / (MI NJ) LDS reads per matrix instruction -- half to two thirds of what 8 waves of half the size read.  The
//     accumulators are AGPRs and named as such in the instruction: left to itself the compiler moves them back and forth;
//   * both operands go global -> LDS with direct-to-LDS loads into rings of 2 to 6 k-tiles (as many as 160 KiB hold), one barrier
//     per k-tile; fragments are double-buffered in registers and read by hand-issued LDS reads between the matrix instructions;
//   * a compute unit has 32 KiB of loads on their way at most, and they come back in order: X, from the L2 in 0.1 us, waits behind W,
//     from memory in 0.5 us and more.  Taken in turns, 60 GB/s of both together reach a compute unit, and that bounded most
//     prompts (384 rows x 12288 x 16384: 174 us of loads alone, 98 with W from the L2).  So W goes out for two k-tiles at a time and
//     then X for two (loads alone 147 us); tiles whose rings are too short for that spread their loads over both k-steps at least;
//   * with one or two rows of tiles every weight byte is read about once, and the loads say so (non-temporal: 84 -> 73 us for a
//     16384 x 12288 weight at 72 rows);
//   * up to 256 rows the workgroups of different feature blocks start their loop over k at different k-tiles, which spreads what
//     they read at one time over the memory channels (mid_turn in gemm_mid.hip: up to 28 % of a GEMM).  Where it starts depends on
//     the feature alone, not on the tile: a member of a group has the same bits as a call of its own;
//   * K-slices meet in the kernel: the slice of a tile that arrives last adds the others' sums and applies the epilogue.  A second
//     kernel for that cost 5-10 us per GEMM.
// 16384 x 12288 weight (403 MB), fragment blocks, all loads of a k-tile under its second k-step -> now: 80 rows 71 -> 69 us, 128 rows
// 80 -> 76, 256 rows 112 -> 100, 384 rows 150 -> 132 (1.17 PFLOP/s), 666 rows 241 -> 222, 1000 rows 310 -> 290 (1.39).
#pragma once
#include "gemm_common.hpp"

namespace lg {

constexpr int MID_K = 64;
constexpr int MID_THREADS = 256;
constexpr int MID_MAX_SPINS = 1 << 21;

struct MidLaunch {  // what a launch of one of the instantiations needs besides the problem
    int nsplit, kt_per_split;
    int turn;  // k-tiles by which the workgroups of neighbouring feature blocks are apart in their loop over k (0: all start at the first)
    bool pairs;  // a workgroup computes two of four K-slices, one after the other
    StreamInfo si;
    hipStream_t stream;
};

// block position of a [64 k][32 NJ n] weight tile: which logical 32-byte block sits at position `pos` of row k, and where block `blk` sits.
// Power-of-two widths XOR.  The 192-wide tile has 12 blocks to a row and rotates: its rows are 96 dwords apart, so rows k and k + 2 (and k + 8,
// k + 10: the other half of the 32 lanes that one transposed read serves together) would share banks.
template <int NJ> __device__ __forceinline__ int mid_swz_kn(int k, int pos) {
    if (NJ == 6) { const int b = pos + ((k >> 1) & 1) + 2 * ((k >> 3) & 1); return b >= 12 ? b - 12 : b; }
    return swz_b(k, pos);
}
template <int NJ> __device__ __forceinline__ int mid_unswz_kn(int k, int blk) {
    if (NJ == 6) { const int p = blk - ((k >> 1) & 1) - 2 * ((k >> 3) & 1); return p < 0 ? p + 12 : p; }
    return swz_b(k, blk);
}

__device__ __forceinline__ void mfma16_acc(float4_t& c, half8_t a, half8_t b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

typedef int int4_t __attribute__((ext_vector_type(4)));

// When the loads of later k-tiles are issued: all of a k-tile's under its second k-step, half of them there and half under the next k-tile's
// first, or for two k-tiles at a time, W before X
enum { MID_BURST, MID_SPREAD, MID_PAIRS };
// cache policy of the K-slices' sums: written through to, and read from, the level that all XCDs share
constexpr int CACHE_DEVICE = 16;
// the tile that comes with two K-slices to a workgroup as well, for K-contiguous weights
constexpr int MID_PAIR_MI = 4, MID_PAIR_NJ = 6;
// most K-slices of a tile (their sums are held in registers 64 fragments at a time)
constexpr int mid_max_splits(int mi, int nj) { return mi * nj <= 16 ? 8 : 2; }

// PAIR: a workgroup takes two K-slices of equal length, one after the other, and adds their sums.  It starts at the k-tile at which a single
// slice of both would start, in the first or the second, so that the starts are spread as far apart.
template <int WL, int MI, int NJ, int XS, int WS, int ORDER, bool NT, bool PAIR>
__global__ __launch_bounds__(MID_THREADS, 1) void gemm_f16_mid(GemmArgs g, GemmGroup grp, RowMap rm, int tiles_m, int tiles_n, float* partial, unsigned* arrivals, int nsplit, int kt_per_split, int turn, int wide_store, int region) {
    constexpr int TM = 32 * MI, TN = 32 * NJ;
    constexpr int X_TILE = TM * MID_K, W_TILE = TN * MID_K;  // halves per ring slot
    extern __shared__ __attribute__((aligned(16))) half_t smem[];  // X ring (XS tiles), then W ring (WS tiles)
    half_t* const wring = smem + XS * X_TILE;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int l16 = lane & 15, lk = lane >> 4;

    // Workgroup ids are dealt to the 8 XCDs in turn; every XCD takes a contiguous run of (K-slice, tile column, tile row) with the
    // row fastest, so the workgroups that share a weight panel run next to each other on one XCD and fetch it from memory once.
    int tm, tn, split;
    if (region) {
        // Many rows of tall tiles: the workgroups of a round (one per compute unit, P on each XCD) cover RM x RN tiles, as near to a square as the
        // tile counts allow, and each XCD 4 x P / 4 of them: a round reads 32 operand panels and an XCD 12 of them, where the run below
        // makes it 18 (16 rows of tiles).  Fills cost power, which is what bounds these: 4096 rows x 12288 x 16384 1187 -> 1134 us.
        // RM = 4: any number of blocks of 4 x P / 4 tiles one after the other, from top to bottom; the last round may lack some, and its
        // workgroups have nothing to do (5120 rows x 12288 x 16384 [out, in] 1851 -> 1527 us, 16384 x 12288 1489 -> 1442, 3072 x 12288 x 16384
        // 958 -> 911; blocks from left to right, which make a round read all of W's panels: 1612, 1527, 935).
        const int P = region >> 8, RM = region & 255, pw = P >> 2, RN = 8 * P / RM, xcols = RN / pw;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, round = slot / P, in = slot % P;
        int bm, bn;  // the block, in units of 4 and pw tiles
        if (RM > 4) {
            const int regions_n = tiles_n / RN;
            bm = round / regions_n * (RM / 4) + xcd / xcols;
            bn = round % regions_n * xcols + xcd % xcols;
        } else {
            const int block = round * 8 + xcd, blocks_m = tiles_m >> 2;
            bm = block % blocks_m;
            bn = block / blocks_m;
        }
        tm = bm * 4 + (in & 3);
        tn = bn * pw + (in >> 2);
        if (tn >= tiles_n) return;
        split = 0;
    } else {
        const int total = gridDim.x, q = total >> 3, r = total & 7;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        const int id = xcd * q + min(xcd, r) + slot;
        const int strip = id / tiles_m;  // (tile column, K-slice)
        tm = id - strip * tiles_m;
        tn = strip / nsplit;
        split = strip - tn * nsplit;
    }
    const int tile = tn * tiles_m + tm;
    if (grp.count > 1) {
        const int per = tiles_n / grp.count;
        const int member = tn / per;
        tn -= member * per;
        g.W = grp.W[member];
        g.Y = grp.Y[member];
        g.epi.bias = grp.bias[member];
        g.ldy = grp.ldy[member];
        g.epi.rows = grp.rows[member];
    }
    const int m0 = tm * TM, n0 = tn * TN;
    const int kt0 = split * kt_per_split;
    const int ktiles = min(g.K / MID_K - kt0, kt_per_split);
    const half_t* X = g.X + (int64_t)m0 * g.ldx + (int64_t)kt0 * MID_K;
    const half_t* W = (WL == W_KN)   ? g.W + n0 + (int64_t)kt0 * MID_K * g.ldw
                      : (WL == W_NK) ? g.W + (int64_t)n0 * g.ldw + (int64_t)kt0 * MID_K
                                     : g.W + (int64_t)n0 * g.ldw + (int64_t)kt0 * 1024;

    // per-lane byte offsets of the direct-to-LDS loads of one k-tile: MI + NJ chunks of 1 KiB per wave (X: 8 rows x 128 B each)
    unsigned xoff[MI], woff[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int q = i * 4 + wave;
        const int row = q * 8 + (lane >> 3), pos = lane & 7;
        const int xrow = min(row, g.M - 1 - m0);  // rows beyond M are read from row M-1 and never stored
        xoff[i] = (unsigned)(xrow * (int)g.ldx + swz_a(row, pos) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < NJ; ++i) {
        const int q = i * 4 + wave;
        if (WL == W_TILED) {
            woff[i] = ((unsigned)(q >> 1) * (unsigned)(g.K >> 5) * 512u + (unsigned)(q & 1) * 512u + (unsigned)lane * 8u) * 2u;
        } else if (WL == W_NK) {
            const int row = q * 8 + (lane >> 3), pos = lane & 7;
            woff[i] = (unsigned)(row * (int)g.ldw + swz_a(row, pos) * 8) * 2u;
        } else {
            constexpr int LPR = TN / 8;  // lanes to a k-row
            const int f = q * 64 + lane;
            const int k = f / LPR, p = f % LPR;
            woff[i] = (unsigned)(k * (int)g.ldw + (mid_swz_kn<NJ>(k, p >> 1) * 2 + (p & 1)) * 8) * 2u;
        }
    }
    const int64_t wstep = (WL == W_KN) ? (int64_t)MID_K * g.ldw : (WL == W_NK ? MID_K : 1024);
    const int slice = PAIR ? ktiles >> 1 : ktiles, start = n0 / MID_TURN_COLS * turn % ktiles;
    const bool other = PAIR && start >= slice;  // the second slice of the pair comes first
    const int first = start - (other ? slice : 0);
    // the tile index is clamped to the last one: the loop body is branch-free, the extra loads refill slots nobody reads
    auto at = [&](int kt) {
        const int c = kt < ktiles ? kt : ktiles - 1;
        const bool second = PAIR && c >= slice;
        const int t = c - (second ? slice : 0) + first;
        return (int64_t)((second != other ? slice : 0) + (t < slice ? t : t - slice));
    };
    auto x_tile = [&](int kt) { return reinterpret_cast<const char*>(X + at(kt) * MID_K); };
    auto w_tile = [&](int kt) { return reinterpret_cast<const char*>(W + at(kt) * wstep); };

    constexpr int NLOAD = MI + NJ;
    constexpr bool XFIRST = WS > XS;  // the operand with the shallower ring is issued first in a phase
    auto issue_x = [&](int i, const char* xg, half_t* xs) { load_lds16(reinterpret_cast<const half_t*>(xg + xoff[i]), xs + (i * 4 + wave) * 512); };
    auto issue_w = [&](int i, const char* wg, half_t* ws) { load_lds16<NT ? 2 : 0>(reinterpret_cast<const half_t*>(wg + woff[i]), ws + (i * 4 + wave) * 512); };
    // load l of the NLOAD of one k-tile of each operand
    auto issue_one = [&](int l, const char* xg, const char* wg, half_t* xs, half_t* ws) {
        const bool is_x = XFIRST ? l < MI : l >= NJ;
        const int i = is_x ? (XFIRST ? l : l - NJ) : (XFIRST ? l - MI : l);
        if (is_x) issue_x(i < MI ? i : 0, xg, xs);
        else issue_w(i < NJ ? i : 0, wg, ws);
    };

    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    // the second slice of a pair has sums of its own, all in registers
    float4_t more[PAIR ? MI : 1][PAIR ? NJ : 1];
    if constexpr (PAIR) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) more[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    }

    // LDS addresses of this lane's fragments inside a slot, per k-step (row groups 16 apart travel as instruction offsets)
    unsigned xaddr[2], waddr[2], wfrag[NJ];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        xaddr[ks] = lds_address(smem) + (unsigned)((wm * 16 * MI + l16) * 128 + (swz_a(l16, ks * 4 + lk) * 16));
        waddr[ks] = lds_address(wring) + (WL == W_TILED ? (unsigned)((wn * NJ * 2 + ks) * 1024 + lane * 16)
                                                        : (unsigned)((wn * 16 * NJ + l16) * 128 + (swz_a(l16, ks * 4 + lk) * 16)));
    }
#pragma unroll
    for (int u = 0; u < NJ; ++u) {
        const int k = lk * 8 + (l16 >> 2);
        wfrag[u] = lds_address(wring) + (unsigned)((k * TN + mid_unswz_kn<NJ>(k, wn * NJ + u) * 16 + (l16 & 3) * 4) * 2);
    }
    half4_t blo[2][NJ], bhi[2][NJ];
    constexpr int NDS = MI + NJ;  // LDS read units per k-step: u < NJ -> W fragment u, else X fragment u - NJ
    auto read_unit = [&](auto unit, auto kstep, unsigned xslot, unsigned wslot, half8_t (&a)[MI], half8_t (&b)[NJ]) {
        constexpr int u = decltype(unit)::value, ks = decltype(kstep)::value;
        if constexpr (u >= NJ) {
            lds_read16_issue_at<(u - NJ) * 2048>(a[u - NJ], xaddr[ks] + xslot);
        } else if constexpr (WL == W_KN) {
            lds_read_tr4_issue_at<ks * 64 * TN>(blo[ks][u], wfrag[u] + wslot);
            lds_read_tr4_issue_at<ks * 64 * TN + 8 * TN>(bhi[ks][u], wfrag[u] + wslot);
        } else {
            lds_read16_issue_at<u * 2048>(b[u], waddr[ks] + wslot);
        }
    };
    // waits for every LDS read in flight and names the fragments of k-step ks, so that nothing uses them earlier
    auto arrive = [&](auto kstep, half8_t (&a)[MI], half8_t (&b)[NJ]) {
        constexpr int ks = decltype(kstep)::value;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < MI; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
        for (int u = 0; u < NJ; ++u) {
            if (WL == W_KN) {
                asm volatile("" : "+v"(blo[ks][u]), "+v"(bhi[ks][u]));
                b[u] = join_half4(blo[ks][u], bhi[ks][u]);
            } else {
                asm volatile("" : "+v"(b[u]));
            }
        }
    };
    constexpr int NMFMA = MI * NJ;
    constexpr int DS_SPAN = NMFMA * 3 / 4;
    // One phase = the MFMAs of one k-step with the LDS reads of the next and NL loads of later k-tiles between them
    auto phase = [&](float4_t (&sum)[MI][NJ], auto loads, auto kstep, half8_t (&ma)[MI], half8_t (&mb)[NJ], half8_t (&ra)[MI], half8_t (&rb)[NJ], unsigned rx, unsigned rw, auto&& load) {
        constexpr int NL = decltype(loads)::value;
        constexpr int KS = decltype(kstep)::value;
        static_for<NMFMA>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            constexpr int i = m / NJ, j = m % NJ;
            mfma16_acc(sum[i][j], mb[j], ma[i]);
            static_for<NL>([&](auto lc) {
                constexpr int l = decltype(lc)::value;
                if constexpr (l * NMFMA / NL == m) load(l);
            });
            static_for<NDS>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                if constexpr (u * DS_SPAN / NDS == m) read_unit(uc, std::integral_constant<int, KS ^ 1>{}, rx, rw, ra, rb);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using Step0 = std::integral_constant<int, 0>;
    using Step1 = std::integral_constant<int, 1>;
    auto x_at = [](int slot) { return (unsigned)(slot * X_TILE * 2); };
    auto w_at = [](int slot) { return (unsigned)(slot * W_TILE * 2); };
    half8_t a0[MI], b0[NJ], a1[MI], b1[NJ];
    // tile kt + 1 has landed for every wave but IN_FLIGHT of this wave's loads, which are later, and this wave has all of tile kt in registers
    auto publish = [&](auto in_flight) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(in_flight)::value) : "memory");
        arrive(Step1{}, a1, b1);
        barrier_keep_loads_in_flight();
    };
    int kt = 0;
    if constexpr (ORDER == MID_PAIRS) {
        // Every second k-tile the W tiles of two k-tiles go out together, and then their X tiles.
        static_assert(XS == WS && XS >= 3, "one ring depth for both operands");
        constexpr int S = XS;
        constexpr int EVEN = (S - 2) * MI + (S - 3) * NJ, ODD = (S - 2) * NJ + (S - 3) * MI;  // loads issued after those of tile kt + 1
#pragma unroll
        for (int t = 0; t < S - 1; ++t) {
#pragma unroll
            for (int i = 0; i < MI; ++i) issue_x(i, x_tile(t), smem + t * X_TILE);
#pragma unroll
            for (int i = 0; i < NJ; ++i) issue_w(i, w_tile(t), wring + t * W_TILE);
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * NLOAD) : "memory");
        barrier_keep_loads_in_flight();
        static_for<NDS>([&](auto uc) { read_unit(uc, Step0{}, 0u, 0u, a0, b0); });
        arrive(Step0{}, a0, b0);
        int prev = S - 1, slot = 0, next = 1;
        auto advance = [&] {
            prev = slot;
            slot = next;
            next = next == S - 1 ? 0 : next + 1;
        };
        // (two loops, one after the other, for a pair: one loop over both would move the accumulators from registers to registers)
        auto run = [&](float4_t (&sum)[MI][NJ], int end) {
            for (;;) {
                {   // even k-tile: the second X tile of the last pair, then a pair of W tiles, into the slots of k-tiles kt - 1 and kt
                    const char* xg = x_tile(kt - 1 + S);
                    half_t* const xs = smem + prev * X_TILE;
                    phase(sum, std::integral_constant<int, MI>{}, Step0{}, a0, b0, a1, b1, x_at(slot), w_at(slot), [&](int l) { issue_x(l, xg, xs); });
                    publish(std::integral_constant<int, EVEN>{});
                    const char* wg0 = w_tile(kt - 1 + S);
                    const char* wg1 = w_tile(kt + S);
                    half_t* const ws0 = wring + prev * W_TILE;
                    half_t* const ws1 = wring + slot * W_TILE;
                    phase(sum, std::integral_constant<int, 2 * NJ>{}, Step1{}, a1, b1, a0, b0, x_at(next), w_at(next),
                          [&](int l) { l < NJ ? issue_w(l, wg0, ws0) : issue_w(l - NJ, wg1, ws1); });
                    arrive(Step0{}, a0, b0);
                }
                if (++kt >= end) break;
                advance();
                {   // odd k-tile: the first X tile of the pair
                    phase(sum, std::integral_constant<int, 0>{}, Step0{}, a0, b0, a1, b1, x_at(slot), w_at(slot), [](int) {});
                    publish(std::integral_constant<int, ODD>{});
                    const char* xg = x_tile(kt - 1 + S);
                    half_t* const xs = smem + prev * X_TILE;
                    phase(sum, std::integral_constant<int, MI>{}, Step1{}, a1, b1, a0, b0, x_at(next), w_at(next), [&](int l) { issue_x(l, xg, xs); });
                    arrive(Step0{}, a0, b0);
                }
                if (++kt >= end) break;
                advance();
            }
        };
        run(acc, slice);
        if constexpr (PAIR) {
            advance();
            run(more, ktiles);
        }
    } else {
        static_assert(!PAIR, "pairs of slices: only where loads go out in pairs");
        // The loads of k-tiles kt + XS and kt + WS go out once tile kt is done with: NOW of them under its second k-step and the others under
        // the first k-step of the next.
        constexpr int SMAX = XS > WS ? XS : WS, SMIN = XS < WS ? XS : WS;
        constexpr int NDEEP = XS == WS ? 0 : (XS > WS ? MI : NJ);  // loads of the deeper ring that may stay in flight besides whole tiles
        constexpr int NOW = ORDER == MID_BURST ? NLOAD : NLOAD / 2;
        // prologue: tiles 0 .. in the order the loop would have issued them
        static_for<SMAX>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
#pragma unroll
            for (int l = 0; l < NLOAD; ++l) {
                const bool is_x = XFIRST ? l < MI : l >= NJ;
                if (l >= NOW && t == (is_x ? XS : WS) - 1) continue;
                if (is_x ? t < XS : t < WS) issue_one(l, x_tile(t), w_tile(t), smem + t * X_TILE, wring + t * W_TILE);
            }
        });
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SMIN - 1) * NLOAD + NDEEP - (NLOAD - NOW)) : "memory");
        barrier_keep_loads_in_flight();
        static_for<NDS>([&](auto uc) { read_unit(uc, Step0{}, 0u, 0u, a0, b0); });
        arrive(Step0{}, a0, b0);
        int xslot = 0, wslot = 0, xprev = XS - 1, wprev = WS - 1;
        do {
            const char* xg0 = x_tile(kt - 1 + XS);
            const char* wg0 = w_tile(kt - 1 + WS);
            half_t* const xs0 = smem + xprev * X_TILE;
            half_t* const ws0 = wring + wprev * W_TILE;
            phase(acc, std::integral_constant<int, NLOAD - NOW>{}, Step0{}, a0, b0, a1, b1, x_at(xslot), w_at(wslot), [&](int l) { issue_one(l + NOW, xg0, wg0, xs0, ws0); });
            publish(std::integral_constant<int, (SMIN - 2) * NLOAD + NDEEP>{});
            const char* xg = x_tile(kt + XS);
            const char* wg = w_tile(kt + WS);
            half_t* const xs = smem + xslot * X_TILE;
            half_t* const ws = wring + wslot * W_TILE;
            xprev = xslot;
            wprev = wslot;
            xslot = xslot == XS - 1 ? 0 : xslot + 1;
            wslot = wslot == WS - 1 ? 0 : wslot + 1;
            phase(acc, std::integral_constant<int, NOW>{}, Step1{}, a1, b1, a0, b0, x_at(xslot), w_at(wslot), [&](int l) { issue_one(l, xg, wg, xs, ws); });
            arrive(Step0{}, a0, b0);
        } while (++kt < ktiles);
    }
    // The clamped refills of the last iterations land, and the last matrix instructions write their results: they are assembly, so the
    // compiler does not wait for them by itself.  The accumulators are named after the wait so that nothing reads one before it.
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            asm volatile("" : "+a"(acc[i][j]));
            if constexpr (PAIR) {
                asm volatile("" : "+a"(more[i][j]));
                acc[i][j] += more[i][j];
            }
        }

    // ---- epilogue: acc[i][j][r] = Y[m0 + wm*16*MI + i*16 + l16][n0 + wn*16*NJ + j*16 + 4*lk + r] ---------------------------
    // ---- K-slices: the slice of a tile that arrives last takes the others' fp32 sums from the stream's workspace (lane-contiguous),
    // adds all of them in slice order (four as two pairs, as workgroups that take a pair each do) and goes on to the epilogue.  Nobody waits
    // for a workgroup that may not be running: the wait below is for slices that have already arrived and are storing, microseconds.  It is
    // bounded (a second or so) for a caller who breaks the rule that one launch runs at a time on a workspace (a captured graph replayed on
    // two streams at once): wrong sums then, but the launch ends.  The counters are back at zero when the launch ends.
    if (nsplit > 1) {
        constexpr int SLICE = MI * NJ * MID_THREADS * 16;  // bytes
        // Small tiles: every slice stores its sums, then counts itself in (one trip to the counter).  Large ones: a slice first learns
        // whether it is the last, and the last one stores nothing, which saves a write of up to 256 KiB per tile.
        constexpr bool ASK_FIRST = MI * NJ > 16;
        const int tiles = tiles_m * tiles_n;
        const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(partial, 0, (int)LG_SPLITK_WORKSPACE_BYTES, 0x00027000);
        unsigned* const arrived = arrivals + tile;
        unsigned* const stored = arrivals + LG_ARRIVAL_COUNTERS / 2 + tile;
        unsigned* const flag = reinterpret_cast<unsigned*>(smem);
        auto count_in = [&](unsigned* counter) {  // every thread gets the count before this workgroup
            __syncthreads();
            if (tid == 0) *flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            return *flag;
        };
        auto store_sums = [&] {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4_t, acc[i][j]), ws, tid * 16 + (i * NJ + j) * (MID_THREADS * 16),
                                                           (split * tiles + tile) * SLICE, CACHE_DEVICE);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        };
        if (ASK_FIRST) {
            if (count_in(arrived) != (unsigned)nsplit - 1) {
                store_sums();
                __syncthreads();
                if (tid == 0) __hip_atomic_fetch_add(stored, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return;
            }
            if (tid == 0) {
                for (int spins = 0; spins < MID_MAX_SPINS && __hip_atomic_load(stored, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (unsigned)nsplit - 1; ++spins)
                    __builtin_amdgcn_s_sleep(1);
                __hip_atomic_store(stored, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
        } else {
            store_sums();
            if (count_in(arrived) != (unsigned)nsplit - 1) return;
        }
        if (tid == 0) __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        auto slice = [&](int sp, int f) {
            return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(ws, tid * 16 + f * (MID_THREADS * 16), (sp * tiles + tile) * SLICE, CACHE_DEVICE));
        };
        constexpr int MAXS = mid_max_splits(MI, NJ), G = MAXS == 2 ? 16 : 4;  // fragments whose slices are in flight together
#pragma unroll
        for (int f0 = 0; f0 < MI * NJ; f0 += G) {
            if (MAXS == 2 || nsplit == 2) {  // a + b == b + a
                float4_t p[G];
#pragma unroll
                for (int f = 0; f < G; ++f)
                    if (f0 + f < MI * NJ) p[f] = slice(split ^ 1, f0 + f);
#pragma unroll
                for (int f = 0; f < G; ++f)
                    if (f0 + f < MI * NJ) acc[(f0 + f) / NJ][(f0 + f) % NJ] += p[f];
            } else {
                float4_t p[MAXS][G];
#pragma unroll
                for (int sp = 0; sp < MAXS; ++sp)
#pragma unroll
                    for (int f = 0; f < G; ++f)
                        if (f0 + f < MI * NJ) p[sp][f] = slice(min(sp, nsplit - 1), f0 + f);
#pragma unroll
                for (int f = 0; f < G; ++f)
                    if (f0 + f < MI * NJ) {
                        float4_t v = p[0][f] + p[1][f];
#pragma unroll
                        for (int sp = 2; sp < MAXS; ++sp) {
                            const float4_t w = v + p[sp][f];
#pragma unroll
                            for (int r = 0; r < 4; ++r) v[r] = sp < nsplit ? w[r] : v[r];
                        }
                        const float4_t pairs = (p[0][f] + p[1][f]) + (p[2][f] + p[3][f]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] = nsplit == 4 ? pairs[r] : v[r];
                        acc[(f0 + f) / NJ][(f0 + f) % NJ] = v;
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    const int kind = g.epi.kind;
    if (kind == LG_EPI_BIAS_GEGLU) {
#pragma unroll
        for (int jp = 0; jp < NJ / 2; ++jp) {
            const int n = n0 + wn * (16 * NJ) + jp * 32 + 4 * lk;
            const half4_t g4 = *reinterpret_cast<const half4_t*>(g.epi.bias + n);
            const half4_t u4 = *reinterpret_cast<const half4_t*>(g.epi.bias + n + 16);
            const int col = (n >> 5) * 16 + (n & 15);
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int m = m0 + wm * 16 * MI + i * 16 + l16;
                if (m >= g.M) continue;
                half4_t o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = (half_t)(gelu_tanh(acc[i][2 * jp][r] + (float)g4[r]) * (acc[i][2 * jp + 1][r] + (float)u4[r]));
                *reinterpret_cast<half4_t*>(g.Y + (int64_t)m * g.ldy + col) = o;
            }
        }
        return;
    }
    // The tile goes through LDS and leaves in whole rows; rows that are not 16-byte aligned leave 8 bytes at a time.
    constexpr int PITCH = TN + 8;
    barrier_keep_loads_in_flight();  // every wave has read its last fragments
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int n = n0 + wn * (16 * NJ) + j * 16 + 4 * lk;
        float bv[4] = {-0.f, -0.f, -0.f, -0.f};  // x + -0 is x
        if (kind != LG_EPI_NONE) {
            const half4_t b4 = *reinterpret_cast<const half4_t*>(g.epi.bias + n);
#pragma unroll
            for (int r = 0; r < 4; ++r) bv[r] = (float)b4[r];
        }
        // one branch a column instead of one for every four outputs, which cost 256 x 256 tiles 1.2 us of their epilogue (4096 rows x 4096 x 1024 34.4
        // -> 33.3 us, 6144 x 8192 x 2048 167.7 -> 165)
        auto column = [&](auto act) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = act(acc[i][j][r] + bv[r]);
                const half4_t o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
                *reinterpret_cast<half4_t*>(&smem[(wm * 16 * MI + i * 16 + l16) * PITCH + wn * (16 * NJ) + j * 16 + 4 * lk]) = o;
            }
        };
        if (kind == LG_EPI_BIAS_GELU) column([](float v) { return gelu_tanh(v); });
        else column([](float v) { return v; });
    }
    __syncthreads();
    auto dest = [&](int m, int n) -> int64_t {
        if (kind == LG_EPI_BIAS_HEADS || kind == LG_EPI_BIAS_HEADS_ROWS) {
            int b, sq;
            if (kind == LG_EPI_BIAS_HEADS) { b = m / g.epi.seq; sq = m % g.epi.seq; }
            else { b = g.epi.rows ? rm.slot[m] : m; sq = g.epi.rows ? rm.pos[m] : 0; }
            return (((int64_t)b * g.epi.heads_total + n / g.epi.d) * g.ldy + sq) * (int64_t)g.epi.d + (n % g.epi.d);
        }
        return (int64_t)m * g.ldy + n;
    };
    constexpr int CPR = TN / 8;                         // 16-byte chunks per tile row
    constexpr int ITERS = (TM * CPR + MID_THREADS - 1) / MID_THREADS;  // (160 and 224 rows of 96: not a whole number of chunks a thread)
#pragma unroll 4
    for (int it = 0; it < ITERS; ++it) {
        const int c = it * MID_THREADS + tid;
        const int row = c / CPR, cc = c % CPR;
        const int m = m0 + row, n = n0 + cc * 8;
        if (m >= g.M || (TM * CPR % MID_THREADS && row >= TM)) continue;
        const half8_t o = *reinterpret_cast<const half8_t*>(&smem[row * PITCH + cc * 8]);
        if (wide_store) {
            *reinterpret_cast<half8_t*>(g.Y + dest(m, n)) = o;
        } else {
            *reinterpret_cast<half4_t*>(g.Y + dest(m, n)) = half4_t{o[0], o[1], o[2], o[3]};
            *reinterpret_cast<half4_t*>(g.Y + dest(m, n + 4)) = half4_t{o[4], o[5], o[6], o[7]};
        }
    }
}

// Ring depths: as many k-tiles as 160 KiB hold, at most 6.  Where they do not hold 3 of both: W, which comes from memory, gets the third
// (6 x 8 and 7 x 8: 0.90 of the time before, with 3 of X 0.94), but for 256 rows, where it makes no difference up to two rows of tiles and X
// gains by it above.
constexpr int mid_depth(int mi, int nj) { return 6 * (mi + nj) <= 40 ? 6 : 4 * (mi + nj) <= 40 ? 4 : 3 * (mi + nj) <= 40 ? 3 : 2; }
constexpr int mid_xs(int mi, int nj) { return mid_depth(mi, nj) > 2 ? mid_depth(mi, nj) : mi == 8 ? 3 : 2; }
constexpr int mid_ws(int mi, int nj) { return mid_depth(mi, nj) > 2 ? mid_depth(mi, nj) : mi == 8 ? 2 : 3; }
// Against all loads under the second k-step, over the problems that a tile is good for: in pairs 0.89 (6 x 4), 0.91 (4 x 3, 8 x 4), 0.95 (3 x 4,
// 4 x 4), 0.97-1.0 (the others of depth 4 and 6: bound by memory, or by few workgroups); at depth 3 spread 0.89-0.99, in pairs up to 1.05.
// 1 x 4 with weights contiguous along k, from two rows of tiles on: in pairs 1.00-1.04, spread 1.00-1.05 ([in, out]: in pairs 0.93-1.0).
// 4 x 6 with weights [in, out] above 256 rows: in pairs 1.00-1.07 (978 rows x 6144 x 12288 146 -> 156 us, 1968 x 9216 x 12288 433 -> 461), spread 0.99-1.05;
// up to 256 rows, with its K-slices, in pairs 0.95-0.98.
constexpr int mid_order(int wl, int mi, int nj) {
    return mi == 1 && nj == 4 && wl != W_KN ? MID_BURST : mid_depth(mi, nj) > 3 || nj == 4 ? MID_PAIRS : MID_SPREAD;
}

template <int WL, int MI, int NJ, int ORDER, bool NT, bool PAIR = false>
static void launch_mid_order(const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    constexpr int XS = mid_xs(MI, NJ), WS = mid_ws(MI, NJ);
    const int tiles_m = (g.M + 32 * MI - 1) / (32 * MI), tiles_n = g.N / (32 * NJ) * grp.count;
    constexpr size_t ring = (size_t)(XS * MI + WS * NJ) * 32 * MID_K * sizeof(half_t), tile = (size_t)(32 * MI) * (32 * NJ + 8) * sizeof(half_t);
    constexpr size_t smem = ring > tile ? ring : tile;
    static_assert(smem <= 160 * 1024, "a compute unit has 160 KiB of LDS");
    // whole-row stores need 16-byte aligned rows (heads epilogue: rows of size_per_head halves)
    int wide = 1;
    for (int i = 0; i < grp.count; ++i)
        if (!aligned16(grp.Y[i]) || (g.epi.kind == LG_EPI_BIAS_HEADS || g.epi.kind == LG_EPI_BIAS_HEADS_ROWS ? (g.epi.d % 8 != 0) : (grp.ldy[i] % 8 != 0))) wide = 0;
    // set once per instantiation; the initialisation of a function-local static is thread-safe
    static const hipError_t attr_rc = hipFuncSetAttribute((const void*)gemm_f16_mid<WL, MI, NJ, XS, WS, ORDER, NT, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    (void)attr_rc;
    // Tiles of 160 to 224 rows are placed where they make more than one round (2560 rows x 12288 x 16384 822 -> 788 us, 5120 x 4096 x 4096 152 ->
    // 142); in one round it gains nothing (1280 x 8192 x 2048 41 -> 41.5), and smaller tiles lose by it.
    int region = 0;
    int64_t blocks = (int64_t)tiles_m * tiles_n * l.nsplit;
    const int P = l.si.cus >> 3, pw = P >> 2;
    if ((MI == 8 || (MI >= 5 && blocks > 8 * P)) && l.nsplit == 1 && pw >= 1 && P % 4 == 0) {
        if (tiles_m % 16 == 0 && tiles_n % (2 * pw) == 0) region = 16;
        else if (tiles_m % 8 == 0 && tiles_n % (4 * pw) == 0) region = 8;
        else if (tiles_m % 4 == 0 && tiles_n % pw == 0) {
            region = 4;
            blocks = (blocks + 8 * P - 1) / (8 * P) * (8 * P);
        }
        if (region) region |= P << 8;
    }
    hipLaunchKernelGGL((gemm_f16_mid<WL, MI, NJ, XS, WS, ORDER, NT, PAIR>), dim3((unsigned)blocks), dim3(MID_THREADS), smem, l.stream, g, grp, rm, tiles_m, tiles_n,
                       l.si.ws, l.si.arrivals, l.nsplit, l.kt_per_split, l.turn, wide, region);
}

template <int WL, int MI, int NJ, bool NT>
static void launch_mid_tile(const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    if constexpr (WL != W_KN && MI == MID_PAIR_MI && NJ == MID_PAIR_NJ)
        if (l.pairs) return launch_mid_order<WL, MI, NJ, MID_PAIRS, NT, true>(g, grp, rm, l);
    if constexpr (WL == W_KN && MI == 4 && NJ == 6 && !NT)
        if (g.M >= kSequentialRows) return launch_mid_order<WL, MI, NJ, MID_BURST, NT>(g, grp, rm, l);
    launch_mid_order<WL, MI, NJ, mid_order(WL, MI, NJ), NT>(g, grp, rm, l);
}

// one instantiation per tile height MI of a list, with and without the non-temporal hint
template <int WL, int NJ, int... MI>
static bool launch_mid_heights(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return ((mi == MI && (nt ? launch_mid_tile<WL, MI, NJ, true>(g, grp, rm, l) : launch_mid_tile<WL, MI, NJ, false>(g, grp, rm, l), true)) || ...);
}

}  // namespace lg
