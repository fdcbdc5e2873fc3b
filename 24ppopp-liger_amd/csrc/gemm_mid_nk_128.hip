// gemm_mid_nk_128.hip -- instantiations of gemm_mid.hpp for weights [out, in] and tiles of 96 and 128 features.
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_nk_96(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_NK, 3, 2, 4, 5, 6, 7, 8>(mi, nt, g, grp, rm, l);
}
bool launch_mid_nk_128(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_NK, 4, 1, 2, 3, 4, 6, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
