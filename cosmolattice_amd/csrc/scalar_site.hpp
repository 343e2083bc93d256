// Per-site arithmetic of the scalar-singlet passes that keep plane-linear chunks of the lattice
// (scalar_flat.hpp, scalar_resident.hpp): the kick and the volume sums of one site from its drifted
// value and those of its six neighbours.  Every product and sum is formed as in scalar_rows.hpp and
// scalar_pass.hip, so fields and momenta are bit-identical to theirs.
#pragma once

#include "scalar_rows.hpp"

namespace clmi {
namespace {

// Constants of one pass, from the device background state.
struct SiteK {
  double ck, ck2, aK, aV, inv_dx, inv_dx2;  // FP64
  float kK, kV, kK2, kV2;                   // FP32-bulk
};

__device__ __forceinline__ SiteK site_consts(double ck, double ck2, double aK, double aV, double inv_dx,
                                             double inv_dx2)
{
  SiteK k;
  k.ck = ck;
  k.ck2 = ck2;
  k.aK = aK;
  k.aV = aV;
  k.inv_dx = inv_dx;
  k.inv_dx2 = inv_dx2;
  k.kK = (float)(ck * aK * inv_dx2);
  k.kV = (float)(ck * aV);
  k.kK2 = (float)(ck2 * aK * inv_dx2);
  k.kV2 = (float)(ck2 * aV);
  return k;
}

// Drift of one stored value: exactly Tr<F32>::value.
__device__ __forceinline__ void drift_value(double &v, double p, double fs, double cdt, float)
{
  v = __dadd_rn(v, __dmul_rn(fs, __dmul_rn(cdt, p)));
}
__device__ __forceinline__ void drift_value(float2 &v, float p, double, double, float cf) { pair_add(v.x, v.y, cf * p); }

// One site: c the drifted values of the NF fields, xp ... zm their neighbours', p the momenta (kicked
// in place).  kick2: kick a second time, by ck2, from the same fields, summing the momenta after each
// kick (p2, p2b).
template <int NF, bool F32, int PK, bool kick, bool kick2, bool red, class V = typename Tr<F32>::V,
          class M = typename Tr<F32>::P>
__device__ __forceinline__ void site_update(const ScalarPoly &poly, const SiteK &k, const V (&c)[NF], const V (&xp)[NF], const V (&xm)[NF],
                                            const V (&yp)[NF], const V (&ym)[NF], const V (&zp)[NF],
                                            const V (&zm)[NF], M (&p)[NF], double &p2, double &g2, double &vsum,
                                            double &p2b)
{
  if constexpr (!F32) {
    double lap[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if constexpr (kick) {
        double l = 0.0;
        l += xp[f] + xm[f] - 2 * c[f];
        l += yp[f] + ym[f] - 2 * c[f];
        l += zp[f] + zm[f] - 2 * c[f];
        lap[f] = l * k.inv_dx2;
      }
      if constexpr (red) {
        const double gx = (xp[f] - c[f]) * k.inv_dx, gy = (yp[f] - c[f]) * k.inv_dx, gz = (zp[f] - c[f]) * k.inv_dx;
        g2 += gx * gx;
        g2 += gy * gy;
        g2 += gz * gz;
      }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if constexpr (kick) {
        const double F = k.aK * lap[f] - k.aV * dpot<NF, PK, double>(poly, c, f);
        p[f] += k.ck * F;
        if constexpr (kick2) {
          p2 += p[f] * p[f];
          p[f] += k.ck2 * F;
          p2b += p[f] * p[f];
        } else {
          p2 += p[f] * p[f];
        }
      } else {
        p2 += p[f] * p[f];
      }
    }
    if constexpr (red) vsum += pot<NF, PK, double>(poly, c);
  } else {
    float lap[NF], phi[NF];
    float g2f = 0.0f, p2f = 0.0f, p2fb = 0.0f;  // per-site terms in FP32, accumulated over sites in FP64
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      phi[f] = c[f].x + c[f].y;
      const float dxp = (xp[f].x - c[f].x) + (xp[f].y - c[f].y);
      const float dyp = (yp[f].x - c[f].x) + (yp[f].y - c[f].y);
      const float dzp = (zp[f].x - c[f].x) + (zp[f].y - c[f].y);
      if constexpr (kick) {
        const float dxm = (xm[f].x - c[f].x) + (xm[f].y - c[f].y);
        const float dym = (ym[f].x - c[f].x) + (ym[f].y - c[f].y);
        const float dzm = (zm[f].x - c[f].x) + (zm[f].y - c[f].y);
        lap[f] = ((dxp + dxm) + (dyp + dym)) + (dzp + dzm);
      }
      if constexpr (red) g2f += (dxp * dxp + dyp * dyp) + dzp * dzp;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if constexpr (kick) {
        const float d = dpot<NF, PK, float>(poly, phi, f);
        p[f] += k.kK * lap[f] - k.kV * d;
        if constexpr (kick2) {
          p2f += p[f] * p[f];
          p[f] += k.kK2 * lap[f] - k.kV2 * d;
          p2fb += p[f] * p[f];
        } else {
          p2f += p[f] * p[f];
        }
      } else {
        p2f += p[f] * p[f];
      }
    }
    if constexpr (red) {
      p2 += (double)p2f;
      if constexpr (kick2) p2b += (double)p2fb;
      g2 += (double)g2f * k.inv_dx2;
      vsum += (double)pot<NF, PK, float>(poly, phi);
    }
  }
}

}  // namespace
}  // namespace clmi
