// Plan and launch of the resident evolver (kernel in scalar_resident.hpp).
#include "clmi_internal.hpp"

namespace clmi {

const void *resident_kernel_lf_f64(int nf, const ResidentPlan &p, int pk);
const void *resident_kernel_lf_f32(int nf, const ResidentPlan &p, int pk);
const void *resident_kernel_vv_f64(int nf, const ResidentPlan &p, int pk);
const void *resident_kernel_vv_f32(int nf, const ResidentPlan &p, int pk);
const void *resident_kernel_pv_f64(int nf, const ResidentPlan &p, int pk);
const void *resident_kernel_pv_f32(int nf, const ResidentPlan &p, int pk);

namespace {
const void *kernel_of(int scheme, int nf, bool f32, int pk, const ResidentPlan &p)
{
  if (nf < 1 || nf > 2) return nullptr;
  switch (scheme) {
    case RES_LF: return f32 ? resident_kernel_lf_f32(nf, p, pk) : resident_kernel_lf_f64(nf, p, pk);
    case RES_VV: return f32 ? resident_kernel_vv_f32(nf, p, pk) : resident_kernel_vv_f64(nf, p, pk);
    case RES_PV: return f32 ? resident_kernel_pv_f32(nf, p, pk) : resident_kernel_pv_f64(nf, p, pk);
    default: return nullptr;
  }
}
}  // namespace

// One site per lane up to 64^3, two above (64 and 128 as the full-row pass has them).  64^3 and 128^3 take
// eight planes per tile, the full-row pass's group, so that their sums are the same.  Others take four where
// that gives at most 256 tiles, one per CU and half the sites per wave of eight (100^3 FP64: 13.3 us a step), else
// eight; up to 40^3 two, which the plane-chunk pass needs (its tile is the same): at 32^3, two fields FP64, a pass
// and its update take 11.1 us with two planes and 12.8 with four, the resident step 4.8 and 5.2.
bool resident_plan(int N, int nf, ResidentPlan *p)
{
  if (nf < 1 || nf > 2 || N < 24 || N > 128 || (N & 1)) return false;
  p->VZ = N <= 64 ? 1 : 2;
  const int C = kResThreads * p->VZ;
  p->chunks = (N * N + C - 1) / C;
  for (int P : {N <= 40 ? 2 : 4, 8}) {
    p->P = P;
    p->groups = (N + P - 1) / P;
    if (N % 64 != 0 && p->groups * p->chunks <= 256) break;
  }
  p->ragged = N % 64 != 0;  // (every tile of 64^3 and 128^3 is full)
  return p->groups * p->chunks <= 256;
}

hipError_t launch_scalar_resident(int scheme, int nf, bool f32, int pk, const ResidentPlan &p, const ResidentArgs &r,
                                  hipStream_t s)
{
  const void *k = kernel_of(scheme, nf, f32, pk, p);
  if (!k || r.groups != p.groups || r.chunks != p.chunks || r.passes < 1) return hipErrorInvalidValue;
  ResidentArgs args = r;
  void *params[] = {&args};
  return hipLaunchCooperativeKernel(k, dim3(p.groups * p.chunks), dim3(kResThreads), params, 0, s);
}

}  // namespace clmi
