// elem_p3.hpp -- interface of the p = 3 element stiffness kernel (elem_p3.hip).
#pragma once

#include "common.hpp"

namespace yeti {

// COO values (and rows / columns, when Kr is given) of n elements from their geometry records
// (elem_geo_kernel<3, 4>), at entry offsets offs. cus: compute units of the device.
int launch_elem_p3(const double *geo, const int64_t *offs, int32_t n, double lam, double mu, int cus, double *Kd,
                   int32_t *Kr, int32_t *Kc, hipStream_t st);

}  // namespace yeti
