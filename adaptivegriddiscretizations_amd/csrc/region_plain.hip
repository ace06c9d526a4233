// region_plain.hip -- one-launch solve of the Isotropic and Diagonal models.
#include "region_kernels.hpp"

namespace agd {

template <class S> RegionKernels<S> region_plain(int model, int d) {
  if (model == AGD_ISOTROPIC)
    return d == 2 ? make_region_kernels<S, AGD_ISOTROPIC, 2>() : make_region_kernels<S, AGD_ISOTROPIC, 3>();
  return d == 2 ? make_region_kernels<S, AGD_DIAGONAL, 2>() : make_region_kernels<S, AGD_DIAGONAL, 3>();
}
template RegionKernels<float> region_plain<float>(int, int);
template RegionKernels<double> region_plain<double>(int, int);

}  // namespace agd
