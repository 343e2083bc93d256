// Plan and launch of the plane-chunk scalar pass (kernel in scalar_flat.hpp).
#include "clmi_internal.hpp"

namespace clmi {

hipError_t launch_scalar_flat_f64_nf1(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2);
hipError_t launch_scalar_flat_f64_nf2(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2);
hipError_t launch_scalar_flat_f32_nf1(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2);
hipError_t launch_scalar_flat_f32_nf2(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                                      hipStream_t s, bool kick2);

// Even N from 24 (below, a lattice has fewer sites than a few workgroups' chunks) to 500, the largest measured (two
// fields: 66 168 bytes of LDS with the pass's tail, two workgroups a CU; the halo is two pairs a thread up to 512).  One site per lane up to N = 64, two above; the resident evolver's groups up to N = 128.  The x-chunk
// is one group: many short marches balance the CUs and keep the x-halo in L2 (us a step, two fields FP64, x-chunk 8
// / 16 / 24 / 32: 180^3 92 / 96 / 88 / 99, 200^3 119 / 140 / 138 / 158, 250^3 226 / 229 / 250 / 230; 300^3 from 16:
// 386 / - / 400).
bool scalar_flat_plan(int N, int nf, FlatPlan *p)
{
  if (nf < 1 || nf > 2 || (N & 1) || N < 24 || N > 500) return false;
  ResidentPlan r;
  p->VZ = N <= 64 ? 1 : 2;
  p->G = resident_plan(N, nf, &r) ? r.P : N <= 256 ? 8 : 16;
  const int C = kFlatThreads * p->VZ;
  p->chunks = (N * N + C - 1) / C;
  p->XC = p->G;
  p->blocks = p->chunks * ((N + p->XC - 1) / p->XC);
  p->rows = p->chunks * ((N + p->G - 1) / p->G);
  return true;
}

hipError_t launch_scalar_flat(int nf, bool f32, bool drift, bool kick, bool red, const ScalarPassArgs &a,
                              const FlatPlan &p, hipStream_t s, bool kick2)
{
  if (nf == 1)
    return f32 ? launch_scalar_flat_f32_nf1(drift, kick, red, a, p, s, kick2)
               : launch_scalar_flat_f64_nf1(drift, kick, red, a, p, s, kick2);
  if (nf == 2)
    return f32 ? launch_scalar_flat_f32_nf2(drift, kick, red, a, p, s, kick2)
               : launch_scalar_flat_f64_nf2(drift, kick, red, a, p, s, kick2);
  return hipErrorInvalidValue;
}

}  // namespace clmi
