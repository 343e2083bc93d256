// Instantiations of the plane-chunk scalar pass, FP32-bulk storage, 2 fields.
#include "scalar_flat.hpp"

namespace clmi {

hipError_t launch_scalar_flat_f32_nf2(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2)
{
  return poly_kind(a.poly, 2) == 1 ? dispatch_flat_shape<2, true, 1>(drift, kick, red, a, p, s, kick2)
                                    : dispatch_flat_shape<2, true, 0>(drift, kick, red, a, p, s, kick2);
}

}  // namespace clmi
