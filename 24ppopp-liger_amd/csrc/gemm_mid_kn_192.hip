// gemm_mid_kn_192.hip -- instantiations of gemm_mid.hpp for weights [in, out] and tiles of 192 features.
#include "gemm_mid.hpp"

namespace lg {

bool launch_mid_kn_192(int mi, bool nt, const GemmArgs& g, const GemmGroup& grp, const RowMap& rm, const MidLaunch& l) {
    return launch_mid_heights<W_KN, 6, 4, 5, 6, 7, 8>(mi, nt, g, grp, rm, l);
}

}  // namespace lg
