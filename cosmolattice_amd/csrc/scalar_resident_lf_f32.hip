// Instantiations of the resident evolver: leapfrog, FP32-bulk storage.
#include "scalar_resident.hpp"

namespace clmi {

const void *resident_kernel_lf_f32(int nf, const ResidentPlan &p, int pk)
{
  return nf == 1 ? resident_kernel<1, true, RES_LF>(p, pk) : resident_kernel<2, true, RES_LF>(p, pk);
}

}  // namespace clmi
