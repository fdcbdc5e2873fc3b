// gemm_mid_nk_256.hip -- instantiations of gemm_mid.hpp for weights [out, in] and tiles of 256 features.
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_nk_256(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_NK, 8, 4, 5, 6, 7, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
