// K-split tiles of 16 rows; see qgemm_ks.hpp.
#include "qgemm_ks.hpp"

namespace lq {
// As many columns per tile as give every CU one; 64 beyond (several rounds of them).
int launch_ks_c3(const GemmArgs& g, int conv, int groups, hipStream_t st) {
    if (conv) return fail(LQ_ERR_NOT_IMPLEMENTED, "K-split kernel: tiles of 16 rows are for plain GEMMs");
    const int cols = (g.N + 255) / 256;
    if (cols <= 16) return launch_ks<KsCfg<1, 1, 8, 4>, 128, 0>(g, groups, st);
    if (cols <= 32) return launch_ks<KsCfg<1, 2, 8, 3>, 128, 0>(g, groups, st);
    if (cols <= 48) return launch_ks<KsCfg<1, 3, 8, 2>, 128, 0>(g, groups, st);
    return launch_ks<KsCfg<1, 4, 8, 1>, 128, 0>(g, groups, st);
}
}  // namespace lq
