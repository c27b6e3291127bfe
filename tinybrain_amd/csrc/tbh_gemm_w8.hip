// tbh_gemm_w8.hip -- the prefill GEMM (tbh_gemm.h) for INT8 rows.
#include "tbh_gemm.h"

namespace tbh {
namespace gemm {

hipError_t launch_w8(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s) {
    if (xp == 1) return zp ? launch<W8, 1, true>(a, tm, tn, blocks, s) : launch<W8, 1, false>(a, tm, tn, blocks, s);
    if (xp == 3) return zp ? launch<W8, 3, true>(a, tm, tn, blocks, s) : launch<W8, 3, false>(a, tm, tn, blocks, s);
    return zp ? launch<W8, 2, true>(a, tm, tn, blocks, s) : launch<W8, 2, false>(a, tm, tn, blocks, s);
}

}  // namespace gemm
}  // namespace tbh
