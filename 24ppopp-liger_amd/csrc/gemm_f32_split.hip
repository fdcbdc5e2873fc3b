// gemm_f32_split.hip -- which tile of gemm_f32_split.hpp an fp32 GEMM takes.
#include "gemm_f32_split.hpp"

namespace lg {

namespace {

struct TileSplit { int mi, nj; double alone_k, alone, shared_k, shared, ahead; };  // microseconds, for each k and besides
// A tile on a compute unit of its own, and for each round of tiles when they are more than the compute units; `ahead`: what part of a round the
// last one costs on top of its tiles.  Fitted to 798 problems (M 1 .. 4096, N 64 .. 4096, K 256 .. 4096, both layouts, batches) x all tiles:
// picking by it costs 0.4 % on average, at worst 26 %.  8 x 8: the 128 x 128 kernel.
constexpr TileSplit kTilesSplit[] = {{1, 1, 0.00190, 0.07, 0.00186, 0.36, 0.37}, {1, 2, 0.00273, 0.39, 0.00267, 0.66, 0.48}, {2, 2, 0.00385, 1.01, 0.00396, 0.83, 0.55},
                                     {2, 4, 0.00625, 1.70, 0.00746, 2.54, 0.48}, {4, 4, 0.01120, 2.85, 0.01252, 4.38, 0.42}, {8, 8, 0.04864, 2.05, 0.03597, 2.11, 1.00}};
// The same for operands that go through registers, [K, N] and [N, K] weights (700 more problems, rows not 16-byte aligned: 0.4 % on average, at worst
// 24 %; by the table above 3.5 % and 70 %).  With the launch.
constexpr TileSplit kTilesSplitLoose[2][6] = {{{1, 1, 0.00241, 2.94, 0.00260, 0.94, 1.23}, {1, 2, 0.00381, 3.22, 0.00371, 1.23, 1.12}, {2, 2, 0.00674, 3.70, 0.00563, 1.61, 1.15},
                                               {2, 4, 0.00863, 4.41, 0.00915, 3.42, 0.63}, {4, 4, 0.01462, 5.19, 0.01609, 4.23, 0.54}, {8, 8, 0.04797, 7.75, 0.03772, 5.15, 1.40}},
                                              {{1, 1, 0.00336, 3.16, 0.00293, 1.27, 1.28}, {1, 2, 0.00510, 3.62, 0.00455, 1.68, 1.15}, {2, 2, 0.00706, 4.32, 0.00624, 2.21, 1.09},
                                               {2, 4, 0.01102, 5.70, 0.01023, 4.43, 0.79}, {4, 4, 0.01699, 5.16, 0.01799, 4.26, 0.56}, {8, 8, 0.04478, 7.33, 0.03784, 5.09, 1.28}}};

template <int WL>
void launch(const TileSplit& t, bool staged, const GemmArgsF32& g, int batch, hipStream_t stream) {
    switch (t.mi * 8 + t.nj) {
        case 1 * 8 + 1: staged ? launch_f32_split_tile<WL, 1, 1, true>(g, batch, stream) : launch_f32_split_tile<WL, 1, 1, false>(g, batch, stream); break;
        case 1 * 8 + 2: staged ? launch_f32_split_tile<WL, 1, 2, true>(g, batch, stream) : launch_f32_split_tile<WL, 1, 2, false>(g, batch, stream); break;
        case 2 * 8 + 2: staged ? launch_f32_split_tile<WL, 2, 2, true>(g, batch, stream) : launch_f32_split_tile<WL, 2, 2, false>(g, batch, stream); break;
        case 2 * 8 + 4: staged ? launch_f32_split_tile<WL, 2, 4, true>(g, batch, stream) : launch_f32_split_tile<WL, 2, 4, false>(g, batch, stream); break;
        case 4 * 8 + 4: staged ? launch_f32_split_tile<WL, 4, 4, true>(g, batch, stream) : launch_f32_split_tile<WL, 4, 4, false>(g, batch, stream); break;
        default: launch_f32_split128<WL>(g, batch, stream); break;
    }
}

}  // namespace

// The choice of this path looks at K alone: rows and features of a decomposed call have the bits of the whole.
int launch_gemm_f32_split(const GemmArgsF32& g, int wlayout, int batch, bool aligned, hipStream_t stream, bool* handled) {
    *handled = false;
    if (g.K < 256 || g.K % FS_K) return LG_OK;
    // direct-to-LDS loads are whole 16-byte vectors at 16-byte addresses, also where the last tile column of [K, N] weights is moved back;
    // they address the up to 64 rows of a tile by 32-bit element offsets
    const bool staged = aligned && g.ldx < (1 << 25) && g.ldw < (1 << 25) && (wlayout == W_NK || (g.N >= 16 && g.N % 4 == 0));
    const int cus = stream_info(stream).cus;
    const TileSplit* best = nullptr;
    double best_us = 1e30;
    for (const TileSplit& t : staged ? kTilesSplit : kTilesSplitLoose[wlayout == W_NK]) {
        const double tiles = (double)((g.M + 16 * t.mi - 1) / (16 * t.mi)) * ((g.N + 16 * t.nj - 1) / (16 * t.nj)) * batch;
        if (tiles > 1e9 || (wlayout == W_KN && t.nj > 1 && t.nj < 8 && g.N < 16 * t.nj)) continue;  // [K, N] weights are loaded nj features at a time
        const double alone = g.K * t.alone_k + t.alone, shared = tiles > cus ? (tiles / cus + t.ahead) * (g.K * t.shared_k + t.shared) : 0.0;
        const double us = alone > shared ? alone : shared;
        if (us < best_us) { best_us = us; best = &t; }
    }
    if (!best) return LG_OK;
    *handled = true;
    if (wlayout == W_NK) launch<W_NK>(*best, staged, g, batch, stream);
    else launch<W_KN>(*best, staged, g, batch, stream);
    return check_launch("gemm_f32_split");
}

}  // namespace lg
