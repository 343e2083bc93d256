// Instantiations of the resident evolver: position Verlet, FP32-bulk storage.
#include "scalar_resident.hpp"

namespace clmi {

const void *resident_kernel_pv_f32(int nf, const ResidentPlan &p, int pk)
{
  return nf == 1 ? resident_kernel<1, true, RES_PV>(p, pk) : resident_kernel<2, true, RES_PV>(p, pk);
}

}  // namespace clmi
