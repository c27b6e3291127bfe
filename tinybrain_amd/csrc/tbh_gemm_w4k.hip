// tbh_gemm_w4k.hip -- the prefill GEMM (tbh_gemm.h) for INT4 weights with scales along K.
#include "tbh_gemm.h"

namespace tbh {
namespace gemm {

hipError_t launch_w4k(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s) {
    if (xp == 1) return zp ? launch<W4K, 1, true>(a, tm, tn, blocks, s) : launch<W4K, 1, false>(a, tm, tn, blocks, s);
    if (xp == 3) return zp ? launch<W4K, 3, true>(a, tm, tn, blocks, s) : launch<W4K, 3, false>(a, tm, tn, blocks, s);
    return zp ? launch<W4K, 2, true>(a, tm, tn, blocks, s) : launch<W4K, 2, false>(a, tm, tn, blocks, s);
}

}  // namespace gemm
}  // namespace tbh
