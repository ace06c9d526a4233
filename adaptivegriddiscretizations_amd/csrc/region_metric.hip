// region_metric.hip -- one-launch solve of the Riemann and Rander models.
// Not the 2D ones in FP32: their stencils reach beyond the face neighbours that
// the pass solver re-lists, which leaves cells short of the fixed point; the
// exact marks here do not, and change the flow of riemann2 2000^2 by 1e-3 of
// its norm (its error against 64 bits from 1.0e-3 to 3e-4) for a gain of 1.24
// (rander2 501 x 403 with sensitivities: 4e-5, 1.14).  Callers keep the
// results they had.
#include "region_kernels.hpp"

namespace agd {

template <class S> RegionKernels<S> region_metric(int model, int d) {
  if constexpr (sizeof(S) == 8) {
    if (d == 2) return model == AGD_RIEMANN ? make_region_kernels<S, AGD_RIEMANN, 2>() : make_region_kernels<S, AGD_RANDER, 2>();
  }
  if (d == 2) return {};
  return model == AGD_RIEMANN ? make_region_kernels<S, AGD_RIEMANN, 3>() : make_region_kernels<S, AGD_RANDER, 3>();
}
template RegionKernels<float> region_metric<float>(int, int);
template RegionKernels<double> region_metric<double>(int, int);

}  // namespace agd
