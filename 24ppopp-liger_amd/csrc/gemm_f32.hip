// gemm_f32.hip -- which tile of gemm_f32.hpp an fp32 GEMM takes, or whether it stays on the 128 x 128 tiles of gemm.hip.
#include "gemm_f32.hpp"

namespace lg {

namespace {

struct TileF32 { int mi, nj; double alone, shared; };  // microseconds for each k: one tile on a compute unit, and with several sharing it
constexpr TileF32 kTilesF32[] = {{1, 1, 0.0016, 0.0030}, {1, 2, 0.0030, 0.0045}, {2, 2, 0.0048, 0.0074}, {2, 4, 0.0100, 0.0143}, {4, 4, 0.0175, 0.0257}};

// Estimated microseconds, fitted to 54 problems (M 8 .. 4096, K 32 .. 4096, batches up to 128, both layouts) x all tiles.
// 64 x 64 tiles of this kernel reach 82 TFLOP/s on a full chip (their operands come through the first-level cache), the 128 x 128
// tiles of gemm.hip 105-125, but only once there is one of them for every compute unit, and half of that if rows are not 16-byte
// aligned (K of 1024, which gemm_f32_split.hip takes now: 800 x 1024 80 us there, 23 here; 800 x 4096 81 and 102).  Both sum in the same
// order, so the choice changes no bit of a result.
double direct_cost(const TileF32& t, double tiles, int K, int cus) {
    const double load = (tiles + 0.25 * cus) / cus, fixed = 0.09 * t.mi * t.nj;  // fixed: the sums of the waves meet
    const double alone = K * t.alone + fixed, shared = load * (K * t.shared + fixed);
    return 3.5 + (alone > shared || tiles <= cus ? alone : shared);
}
double tile128_cost(double tiles, int K, bool aligned, int cus) {
    const double load = (tiles + 0.25 * cus) / cus;
    const double us = tiles <= cus ? 0.075 * K + 2.0 : load * (0.065 * K + 2.0);
    return 2.5 + (aligned ? us : 2.0 * us);
}

}  // namespace

int launch_gemm_f32_direct(const GemmArgsF32& g, int wlayout, int batch, bool aligned, hipStream_t stream, bool* handled) {
    *handled = false;
    const int cus = stream_info(stream).cus;
    auto tiles = [&](int rows, int cols) { return (double)((g.M + rows - 1) / rows) * ((g.N + cols - 1) / cols) * batch; };
    const TileF32* best = nullptr;
    double best_us = tile128_cost(tiles(128, 128), g.K, aligned, cus);
    for (const TileF32& t : kTilesF32) {
        const double n = tiles(16 * t.mi, 16 * t.nj);
        if (n > 1e9 || (wlayout == W_KN && t.nj > 1 && g.N < 16 * t.nj)) continue;  // [K, N] weights are loaded nj features at a time
        const double us = direct_cost(t, n, g.K, cus);
        if (us < best_us) { best_us = us; best = &t; }
    }
    if (!best) return LG_OK;
    *handled = true;
    const bool nk = wlayout == W_NK;
    switch (best->mi * 8 + best->nj) {
        case 1 * 8 + 1: nk ? launch_f32_direct_tile<W_NK, 1, 1, 4>(g, batch, stream) : launch_f32_direct_tile<W_KN, 1, 1, 4>(g, batch, stream); break;
        case 1 * 8 + 2: nk ? launch_f32_direct_tile<W_NK, 1, 2, 6>(g, batch, stream) : launch_f32_direct_tile<W_KN, 1, 2, 6>(g, batch, stream); break;
        case 2 * 8 + 2: nk ? launch_f32_direct_tile<W_NK, 2, 2, 2>(g, batch, stream) : launch_f32_direct_tile<W_KN, 2, 2, 2>(g, batch, stream); break;
        case 2 * 8 + 4: nk ? launch_f32_direct_tile<W_NK, 2, 4, 2>(g, batch, stream) : launch_f32_direct_tile<W_KN, 2, 4, 2>(g, batch, stream); break;
        default: nk ? launch_f32_direct_tile<W_NK, 4, 4, 3>(g, batch, stream) : launch_f32_direct_tile<W_KN, 4, 4, 3>(g, batch, stream); break;
    }
    return check_launch("gemm_f32_direct");
}

}  // namespace lg
