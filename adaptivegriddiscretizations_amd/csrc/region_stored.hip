// region_stored.hip -- one-launch solve of the models that run from a stored
// scheme: TTI2 and the curvature-penalised models, FP32.  (TTI3 has 126
// weights and codes a cell, FP64 twice the registers: pass solver.)
#include "region_kernels.hpp"

namespace agd {

RegionKernels<float> region_stored(int model, int d) {
  if (model == AGD_TTI && d == 2) return make_region_kernels<float, AGD_TTI, 2>();
  if (d != 3) return {};
  switch (model) {
    case AGD_REEDSSHEPP2: return make_region_kernels<float, AGD_REEDSSHEPP2, 3>();
    case AGD_REEDSSHEPPFWD2: return make_region_kernels<float, AGD_REEDSSHEPPFWD2, 3>();
    case AGD_ELASTICA2: return make_region_kernels<float, AGD_ELASTICA2, 3>();
    case AGD_DUBINS2: return make_region_kernels<float, AGD_DUBINS2, 3>();
  }
  return {};
}

}  // namespace agd
