// Instantiations of the resident evolver: position Verlet, FP64 storage.
#include "scalar_resident.hpp"

namespace clmi {

const void *resident_kernel_pv_f64(int nf, const ResidentPlan &p, int pk)
{
  return nf == 1 ? resident_kernel<1, false, RES_PV>(p, pk) : resident_kernel<2, false, RES_PV>(p, pk);
}

}  // namespace clmi
