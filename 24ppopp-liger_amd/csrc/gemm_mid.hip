// gemm_mid.hip -- which tile, and how many K-slices, an fp16 GEMM takes: the instantiations of gemm_mid.hpp compared by a cost model,
// and the launch.
#include <stdlib.h>

#include "gemm_mid.hpp"

namespace lg {

#define LG_MID_DECL(L) bool launch_mid_##L(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l)
LG_MID_DECL(kn_128); LG_MID_DECL(kn_192); LG_MID_DECL(kn_256);
LG_MID_DECL(nk_96); LG_MID_DECL(nk_128); LG_MID_DECL(nk_192); LG_MID_DECL(nk_256);
LG_MID_DECL(tiled_96); LG_MID_DECL(tiled_128); LG_MID_DECL(tiled_192); LG_MID_DECL(tiled_256);
#undef LG_MID_DECL
void launch_gemm_fast_tile(const GemmArgs& g, const GemmGroup& grp, int wlayout, const StreamInfo& si, hipStream_t stream);

namespace {

struct Tile { signed char mi, nj; };
// the tiles that were the fastest, or within 1 % of it, for some problem of the sweep below; the 96-wide ones exist for K-contiguous weights,
// those of 160 rows and more for token counts above 256 that wider tiles cover with fewer workgroups than compute units (12288 features are 128
// columns of 96, two rows of them a full round): 384 rows x 12288 x 16384 151 -> 139 us, 420 rows 190 -> 154, 500 rows 192 -> 182.  Within a
// layer less is left of it, as more compute units at work lower the clock: two layers of 384 rows 1157 -> 1141 us.
constexpr Tile kTiles[] = {{1, 4}, {2, 4}, {3, 4}, {4, 4}, {6, 4}, {8, 4}, {2, 3}, {4, 3}, {5, 3}, {6, 3}, {7, 3}, {8, 3}, {4, 6}, {5, 6}, {6, 6}, {7, 6}, {8, 6}, {4, 8}, {5, 8}, {6, 8}, {7, 8}, {8, 8}};
constexpr int kMinSliceTiles = 8;     // k-tiles of a K-slice at least: below that its ramp costs more than it hides
constexpr int kMaxTiles = LG_ARRIVAL_COUNTERS / 2;

// Microseconds of one launch.  Fitted to 556 problems (M 8 .. 2048, 17 weight shapes from 1024 x 1024 to 32768 x 12288, all three
// layouts) x all tiles and slice counts, each measured with weights cycled out of the caches; picking by it costs 1 % against
// the best measured choice on average.  Terms: a k-tile costs its matrix work or its loads; a workgroup cannot pull more than 69 GB/s
// of weights (44 in pieces of 256 bytes: 128-wide tiles of [in, out] weights, few rows) and the chip 7.4 TB/s; what memory and matrix
// pipes do in the same time overlaps only in part; a K-slice meeting costs a trip to the counter and the transfer of the sums, in
// every round (three projections of 64 rows x 4096 x 4096 in four slices, three rounds: 40 us).
double tile_cost(int M, int N, int K, int count, int mi, int nj, int nsplit, int wlayout, int cus) {
    const int tiles_m = (M + 32 * mi - 1) / (32 * mi), tiles_n = N / (32 * nj) * count, ktiles = K / MID_K;
    const int kt = (ktiles + nsplit - 1) / nsplit;
    const long wgs = (long)tiles_m * tiles_n * nsplit;
    const double rounds = (double)((wgs + cus - 1) / cus);
    const double work = kt * (0.13 + 0.0192 * mi * nj), loads = kt * (0.0673 + 0.0292 * (mi + nj));
    const double compute = work > loads ? work : loads;
    const double rate = wlayout == W_KN && nj == 4 && M <= 64 ? 44e3 : 69.42e3;
    const double chip = 2.0 * N * K * count / (7.3735e6 * cus / 256.0) / rounds, own = kt * (64.0 * 32 * 2 / rate) * nj;
    double round = compute > chip ? compute + 0.6025 * chip : chip + 0.6025 * compute;
    if (round < own) round = own;
    double us = 3.67 + rounds * round;
    if (nsplit > 1) us += rounds * (2.13 + 0.1128 * mi * nj * (mi * nj <= 16 ? nsplit : 1));
    return us;
}

// 256-row tiles of 192 and 256 features above 256 token rows are 3 % faster against the others than the model says: 5120 rows x 6144 x 12288 in
// 480 tiles of 256 x 256 635 -> 559 us (768 of 160 x 256 592), 2560 x 12288 x 16384 815 -> 765 (790).
constexpr double kTallFactor = 0.97;

// K is sliced, and loops over it are turned, up to 256 token rows only.  Above that every output is one sum in the order of k: a row's
// bits do not depend on the rows and features around it in a call, on the layout or on the stream, so that a batch, its parts and the
// ranges of a decomposed call agree.  The price is what slices would give there, in microseconds at 384 rows ([out, in] weights):
// 6144 x 12288 79 -> 105, 12288 x 16384 140 -> 192, 16384 x 12288 157 -> 163, 2048 x 8192 30 -> 41 (256-row tiles: 160, 236, 197, 94).

// Where a workgroup starts in its loop over k.  If all start at the first k-tile, all of them read the same k of every weight row at
// the same time: pieces of 128 bytes, a row apart, and where the row is a multiple of many memory channels they come from a few of
// them.  Apart by 5 k-tiles, [out, in] weights 24576 x 12288 take 149 -> 107 us at 106 rows (the same as rows padded by 128 bytes),
// 164 -> 140 at 200; 12288 x 24576 139 -> 120 at 106; 6144 x 12288 43.0 -> 41.9.  Fragment blocks, read in pieces
// of 2 KiB, gain 0-3 % by 3 (16384 x 12288 at 80 rows 72.9 -> 70.8).  [in, out] rows are read over their whole length as it is: by 3,
// 12288 x 16384 loses 3 %.  Only where K may be sliced too (up to 256 rows, K of two slices or more).
int mid_turn(int M, int K, int wlayout) {
    if (M >= kSequentialRows || K < 2 * kMinSliceTiles * MID_K) return 0;
    return wlayout == W_NK ? 5 : wlayout == W_TILED ? 3 : 0;
}

}  // namespace

static TilePlan plan_gemm_tiles(const GemmArgs& g, int count, int wlayout, const StreamInfo& si) {
    const int cus = si.cus, ktiles = g.K / MID_K;
    const bool heads = g.epi.kind == LG_EPI_BIAS_HEADS || g.epi.kind == LG_EPI_BIAS_HEADS_ROWS;
    auto usable = [&](const Tile& t, int cnt, int sp) {
        if (g.N % (32 * t.nj)) return false;
        if (t.nj == 3 && (wlayout == W_KN || g.epi.kind == LG_EPI_BIAS_GEGLU)) return false;  // GeGLU: a wave must hold (gate, up) pairs
        if (t.nj == 3 && t.mi > 4 && g.M < kSequentialRows) return false;  // nothing gained where K may be sliced
        if (sp == 1) return true;
        const int64_t tiles = (int64_t)((g.M + 32 * t.mi - 1) / (32 * t.mi)) * (g.N / (32 * t.nj)) * cnt;
        if (t.mi * t.nj > 16 && sp > 2) return false;
        return sp <= 8 && ktiles >= sp * kMinSliceTiles && (ktiles + sp - 1) / sp * (sp - 1) < ktiles && tiles <= kMaxTiles &&
               (size_t)(tiles * sp) * (size_t)(t.mi * t.nj * 4096) <= si.ws_bytes;
    };
    // the best tile for a given number of members and slices (0: any number of slices that keeps one round of workgroups)
    auto pick = [&](int cnt, int fixed) {
        TilePlan p{};
        p.cost = 1e30;
        for (const Tile& t : kTiles) {
            const long tiles = (long)((g.M + 32 * t.mi - 1) / (32 * t.mi)) * (g.N / (32 * t.nj)) * cnt;
            const int fill = tiles > 0 ? (int)(cus / tiles) : 0;
            const int tries[4] = {1, 2, fill > 8 ? 8 : fill, 5};
            for (int c = 0; c < 4; ++c) {
                const int sp = fixed ? fixed : tries[c];
                if ((fixed && c) || sp < 1 || (c > 1 && sp <= 2) || (!fixed && sp > 1 && (!si.ws || tiles * sp > cus || g.M >= kSequentialRows))) continue;
                if (!usable(t, cnt, sp)) continue;
                const double factor = t.mi == 8 && t.nj >= 6 && g.M >= kSequentialRows ? kTallFactor : 1.0;
                const double us = factor * tile_cost(g.M, g.N, g.K, cnt, t.mi, t.nj, sp, wlayout, cus);
                if (us < p.cost) p = TilePlan{us, t.mi, t.nj, sp, false};
            }
        }
        return p;
    };
    // The members of a group (Q, K and V) come as one call or as several: how K is sliced, and with it every bit of the result, must not
    // depend on which.  So it is decided for one member alone or, for the heads epilogue, as suits three best (they are what a decode
    // step calls) among those slice counts with which a projection alone loses less than a half, above 64 rows (prompts, where it is as
    // likely to come alone) a quarter.  Without that limit it left most of the chip idle under one that comes alone, in microseconds:
    // 11 rows x 6144 x 12288 [in, out] 79 -> 31 (the three 93 -> 90), 64 rows x 4096 x 4096 30 -> 21 (33 -> 29), 96 rows x 3072 x 4096
    // 30 -> 18.  Where the weight-streaming kernel takes the three, in another order of the sum anyway, a projection alone is
    // sliced as suits it.
    const TilePlan alone = pick(1, 0);
    if (alone.nsplit == 0) return TilePlan{};
    int slices = alone.nsplit;
    if (heads && (alone.nsplit > 1 || pick(LG_MAX_GROUP, 0).nsplit > 1) && !skinny_takes_group(g, LG_MAX_GROUP, wlayout, cus)) {
        const double most = (g.M <= 64 ? 1.5 : 1.25) * alone.cost;
        double least = 1e30;
        for (int sp = 1; sp <= 8; ++sp) {
            const TilePlan a = pick(1, sp), t = pick(LG_MAX_GROUP, sp);
            if (a.nsplit && t.nsplit && a.cost < most && t.cost < least) { least = t.cost; slices = sp; }
        }
    }
    // Where three want two slices and one four, both have them: the sums of four slices are added as two pairs, and the workgroups of a group
    // compute a pair each.  6144 x 12288 alone, in two slices -> four: [out, in] 96 rows 42.4 -> 38.1 us, 128 rows 46.5 -> 39.7, fragment
    // blocks 41.0 -> 37.0 and 43.6 -> 40.1; a layer of 106 rows with three projections 413 -> 391.  The three of 80 rows as one launch, a
    // pair of slices to a workgroup instead of one slice: fragment blocks 100 -> 105, the step around them unchanged.  (Pairs need the loop
    // over k to take an even number of k-tiles for each slice.)
    if (heads && wlayout != W_KN && slices == 2 && alone.nsplit >= 4 && ktiles % 8 == 0) {
        const TilePlan one = pick(1, 4);
        TilePlan three = pick(LG_MAX_GROUP, 2);
        if (one.nsplit == 4 && three.mi == MID_PAIR_MI && three.nj == MID_PAIR_NJ) {
            three.pairs = true;
            return count == 1 ? one : count == LG_MAX_GROUP ? three : TilePlan{};
        }
    }
    // (where members are sliced and the slices of a group do not fit the workspace, the group is not taken as one launch)
    return pick(count, slices);
}

// alignment and shape that the tile kernels need of every member
static bool tiles_apply(const GemmArgs& g, const GemmGroup& grp, int wlayout, int batch) {
    if (batch != 1 || g.K % MID_K || g.M <= 0 || g.N <= 0 || g.K <= 0) return false;
    if (!aligned16(g.X) || (g.ldx % 8) || (g.ldw % 8)) return false;
    if (g.ldx >= (1 << 22) || g.ldw >= (1 << 22)) return false;  // 256 rows x ld must fit the 31-bit tile offsets
    if (wlayout == W_TILED && g.ldw != g.K) return false;
    const bool heads = g.epi.kind == LG_EPI_BIAS_HEADS || g.epi.kind == LG_EPI_BIAS_HEADS_ROWS;
    for (int i = 0; i < grp.count; ++i) {
        if (!aligned16(grp.W[i]) || (reinterpret_cast<uintptr_t>(grp.Y[i]) & 7u)) return false;
        if (heads ? (g.epi.d % 4 != 0) : (grp.ldy[i] % 4 != 0)) return false;
        if (g.epi.kind != LG_EPI_NONE && (reinterpret_cast<uintptr_t>(grp.bias[i]) & 7u)) return false;  // 8-byte bias loads
    }
    return true;
}

TilePlan plan_gemm_tiles_f16(const GemmArgs& g, const GemmGroup& grp, int wlayout, int batch, hipStream_t stream) {
    if (!tiles_apply(g, grp, wlayout, batch)) return TilePlan{};
    return plan_gemm_tiles(g, grp.count, wlayout, stream_info(stream));
}

int launch_gemm_tiles_f16(const GemmArgs& g, const GemmGroup& grp, const RowMap* rows, int wlayout, int batch, hipStream_t stream, bool* handled) {
    *handled = false;
    if (g.epi.kind == LG_EPI_BIAS_HEADS_ROWS && !rows) return LG_OK;
    TilePlan p = plan_gemm_tiles_f16(g, grp, wlayout, batch, stream);
    if (p.nsplit == 0) return LG_OK;
    const StreamInfo si = stream_info(stream);
    *handled = true;
    // LG_GEMM_TILE_WIDTH=2|3|4 in the environment (read once) overrides the width of 256-row tiles, in units of 64 features, where it
    // divides N: a measurement knob.  2 takes the kernel of gemm_fast.hip, which leaves registers and LDS for a second kernel's waves on
    // the same compute unit.
    static const int width = [] { const char* e = getenv("LG_GEMM_TILE_WIDTH"); return e ? atoi(e) : 0; }();
    if (width >= 2 && width <= 4 && p.mi == 8 && g.M >= kSequentialRows && g.N % (64 * width) == 0) {
        bool whole_rows = true;  // of 16 bytes
        for (int i = 0; i < grp.count; ++i) whole_rows = whole_rows && aligned16(grp.Y[i]);
        if (width > 2 && !(width == 3 && g.epi.kind == LG_EPI_BIAS_GEGLU)) p.nj = 2 * width;
        else if (width == 2 && whole_rows && g.epi.kind != LG_EPI_BIAS_HEADS_ROWS) {
            launch_gemm_fast_tile(g, grp, wlayout, si, stream);
            return check_launch("gemm_f16_fast");
        }
    }
    const int ktiles = g.K / MID_K, kt = (ktiles + p.nsplit - 1) / p.nsplit;
    const MidLaunch l{(ktiles + kt - 1) / kt, kt, mid_turn(g.M, g.K, wlayout), p.pairs, si, stream};
    const RowMap rm = rows ? *rows : RowMap{};
    // Weights that one row of tiles reads, or two whose workgroups run side by side on an XCD, need not stay in the L2: coming from memory, the
    // non-temporal hint is worth 7 % and 4 % with fragment blocks, 7 % and 2 % with [out, in], 5 % and nothing with [in, out], and costs up to
    // 4 % from three rows of tiles on.  Weights that the 256 MiB memory-side cache still holds from the last step lose by it (at two rows
    // 6144 x 2048 5 %, 12288 x 4096 20 %): two rows take it for weights that the cache cannot hold.
    const bool large = (int64_t)g.N * g.K * grp.count * (int64_t)sizeof(half_t) >= (int64_t)256 << 20;
    const bool nt = g.M <= 32 * p.mi || (g.M <= 64 * p.mi && wlayout != W_KN && large);
    bool ok = false;
    switch (p.nj) {
        case 3: ok = wlayout == W_NK ? launch_mid_nk_96(p.mi, nt, g, grp, rm, l) : launch_mid_tiled_96(p.mi, nt, g, grp, rm, l); break;
        case 4: ok = wlayout == W_KN ? launch_mid_kn_128(p.mi, nt, g, grp, rm, l) : wlayout == W_NK ? launch_mid_nk_128(p.mi, nt, g, grp, rm, l) : launch_mid_tiled_128(p.mi, nt, g, grp, rm, l); break;
        case 6: ok = wlayout == W_KN ? launch_mid_kn_192(p.mi, nt, g, grp, rm, l) : wlayout == W_NK ? launch_mid_nk_192(p.mi, nt, g, grp, rm, l) : launch_mid_tiled_192(p.mi, nt, g, grp, rm, l); break;
        case 8: ok = wlayout == W_KN ? launch_mid_kn_256(p.mi, nt, g, grp, rm, l) : wlayout == W_NK ? launch_mid_nk_256(p.mi, nt, g, grp, rm, l) : launch_mid_tiled_256(p.mi, nt, g, grp, rm, l); break;
    }
    if (!ok) { set_error("gemm_f16: no kernel for tile %d x %d", 32 * p.mi, 32 * p.nj); return LG_ERR_INVALID; }
    return check_launch("gemm_f16_mid");
}

}  // namespace lg
