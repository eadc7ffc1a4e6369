// Packed products in tiles of 128 tokens: Any-precision.
#include "qgemm_tile.h"

namespace decdec {

hipError_t launch_qgemm_anyprec(int dt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
    return qgemm_tiles<kAnyprec>(dt, bits, flag, p, g, s);
}

}  // namespace decdec
