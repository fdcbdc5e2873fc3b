// gemm_skinny_kn.hip -- fp16 GEMM for few token rows with weights stored [in, out]: the 128-feature tiles of gemm_mid.hpp.
//
// A k-row of such a weight holds all features, so the B operand needs a transpose: tiles are read from LDS with
// ds_read_b64_tr_b16 (issued by hand).  With one row of tiles this is a stream of the weights (a decode step); it takes the place
// of a kernel of its own that sliced K over all compute units and summed the slices in a second launch (4096 x 4096 weight, 8-16
// rows: 15.3 -> 12.6 us; 16384 x 12288: 69.6 -> 67.3 us; Q, K and V are one launch instead of three and three sums).
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_kn_128(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_KN, 4, 1, 2, 3, 4, 6, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
