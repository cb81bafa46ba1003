// pg16 halo-tile 3x3 conv instances (a scale per 16 input channels).
#include "conv_halo.h"

namespace aexrt {
namespace halo {

hipError_t halo_launch_pg(const HaloParams& h, int jn, int pw, int np, int nw, hipStream_t stream) {
#define AEXRT_HALO_PG_CASE(J, P, N) \
    if (jn == J && pw == P && np == N) { \
        return nw == 8 ? halo_launch_cfg<true, J, P, N, igemm::kEpiAny, false, 8, true>(h, stream) \
                       : halo_launch_cfg<true, J, P, N, igemm::kEpiAny, false, 4, true>(h, stream); \
    }
    AEXRT_HALO_PG_CASE(1, 1, 1) AEXRT_HALO_PG_CASE(1, 1, 4) AEXRT_HALO_PG_CASE(1, 2, 2) AEXRT_HALO_PG_CASE(1, 2, 4)
    AEXRT_HALO_PG_CASE(2, 1, 1) AEXRT_HALO_PG_CASE(2, 1, 4) AEXRT_HALO_PG_CASE(2, 2, 2) AEXRT_HALO_PG_CASE(2, 2, 4)
    AEXRT_HALO_PG_CASE(4, 1, 1) AEXRT_HALO_PG_CASE(4, 1, 4) AEXRT_HALO_PG_CASE(4, 2, 2) AEXRT_HALO_PG_CASE(4, 2, 4)
#undef AEXRT_HALO_PG_CASE
    return hipErrorInvalidValue;
}

}  // namespace halo
}  // namespace aexrt
