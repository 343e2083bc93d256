// Instantiations of the plane-chunk scalar pass, FP32-bulk storage, 1 field.
#include "scalar_flat.hpp"

namespace clmi {

hipError_t launch_scalar_flat_f32_nf1(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2)
{
  return poly_kind(a.poly, 1) == 1 ? dispatch_flat_shape<1, true, 1>(drift, kick, red, a, p, s, kick2)
                                    : dispatch_flat_shape<1, true, 0>(drift, kick, red, a, p, s, kick2);
}

}  // namespace clmi
