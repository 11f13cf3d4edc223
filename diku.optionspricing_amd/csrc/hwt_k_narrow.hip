// hwt_k_narrow.hip -- mixed mode's narrow-tree kernel (trees up to 128 nodes
// wide, FP32 tree states).
#include "hwt_pricers.h"

namespace hwt {

template __global__ void k_price_narrow<float>(const OptConst *__restrict__, const double *__restrict__, const int32_t *__restrict__,
                                             int32_t *__restrict__, double *__restrict__, int32_t *__restrict__);

} // namespace hwt
