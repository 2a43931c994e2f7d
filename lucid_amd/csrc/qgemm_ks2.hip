// K-split tiles of 64 x 32; see qgemm_ks.hpp.
#include "qgemm_ks.hpp"

namespace lq {
int launch_ks_c2(const GemmArgs& g, int conv, int groups, hipStream_t st) {
    return launch_ks_shape<KsCfg<4, 2, 4, 3>>(g, conv, groups, st);
}
}  // namespace lq
