// tbh_gemm_w4n.hip -- the prefill GEMM (tbh_gemm.h) for runtime-layout INT4 (scales per N-block and k).
#include "tbh_gemm.h"

namespace tbh {
namespace gemm {

hipError_t launch_w4n(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s) {
    if (zp || xp == 3) return hipErrorInvalidValue;   // no such weight, no such tile (tile_fits)
    return xp == 1 ? launch<W4N, 1, false>(a, tm, tn, blocks, s) : launch<W4N, 2, false>(a, tm, tn, blocks, s);
}

}  // namespace gemm
}  // namespace tbh
