// gemm_mid_tiled_192.hip -- instantiations of gemm_mid.hpp for weights [out, in] in fragment blocks and tiles of 192 features.
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_tiled_192(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_TILED, 6, 4, 5, 6, 7, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
