// K-split tiles of 32 x 32; see qgemm_ks.hpp.
#include "qgemm_ks.hpp"

namespace lq {
int launch_ks_c1(const GemmArgs& g, int conv, int groups, hipStream_t st) {
    return launch_ks_shape<KsCfg<2, 2, 8, 2>>(g, conv, groups, st);
}
}  // namespace lq
