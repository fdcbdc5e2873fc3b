// gemm_mid_kn_256.hip -- instantiations of gemm_mid.hpp for weights [in, out] and tiles of 256 features.
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_kn_256(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_KN, 8, 4, 5, 6, 7, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
