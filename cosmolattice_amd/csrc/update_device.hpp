// Device-side background update (used by the update kernel).
//
// sum_partials: fixed-order sum of the per-workgroup partial rows (bit-reproducible for a given
// block size).  apply_update: one thread advances the scale factor exactly as the reference's host
// code does and refreshes the kick/drift coefficients the next pass reads.
#pragma once

#include "clmi_internal.hpp"

namespace clmi {

// rpow(); INT: the exponent is known to be an integer of magnitude at most 32 (integer alpha), so the general
// pow(), which costs a kernel that keeps its state in registers about 100 of them, is not compiled in.
template <bool INT> __device__ __forceinline__ double bg_pow(double a, double e)
{
  if constexpr (!INT) return rpow(a, e);
  int n = (int)fabs(e);
  double p = 1.0, q = a;
  while (n) {
    if (n & 1) p *= q;
    q *= q;
    n >>= 1;
  }
  return e < 0 ? 1.0 / p : p;
}

// The scale-factor kernel of ScaleFactorKernels::get/getSI (evolvers/kernels/scalefactorkernels.h:27-124)
// with the energy normalisations of definitions/energies.h:37-85, from the given volume averages.
template <bool INT>
__device__ __forceinline__ double sf_kernel_of(double a, double pi2S, double grad2S, double pi2CS, double grad2CS,
                                      double pi2U1, double mag2U1, double pot, const ModelConsts &mc)
{
  // a^-2, a^-4, a^-6 from one division (a serial chain on the updating thread)
  const double ia = 1.0 / a, ia2 = ia * ia, ia4 = ia2 * ia2, ia6 = ia4 * ia2;
  double Eks = 0, Egs = 0, Ekcs = 0, Egcs = 0, Eel = 0, Emag = 0;
  if (mc.ns > 0) {
    Eks = 0.5 * pi2S * ia6;
    Egs = 0.5 * grad2S * ia2;
  }
  if (mc.ncs > 0) {
    Ekcs = pi2CS * ia6;
    Egcs = grad2CS * ia2;
  }
  if (mc.nu1 > 0) {
    const double w2 = (mc.omegaStar / mc.fStar) * (mc.omegaStar / mc.fStar);
    Eel = 0.5 * w2 * ia4 * pi2U1;
    Emag = 0.5 * w2 * ia4 * mag2U1;
  }
  const double fm = mc.fStar / mc.MPl;
  return bg_pow<INT>(a, 2 * mc.alpha + 1) / 3.0 * (fm * fm) *
         ((mc.alpha - 2) * (Eks + Ekcs) + mc.alpha * (Egs + Egcs) + (mc.alpha - 1) * (Eel + Emag) +
          (mc.alpha + 1) * pot);
}

// Fixed-order sum of `rows` partial rows by a block of NT threads: thread t adds rows t, t + NT, ... in
// that order, four rows in flight per batch (each row one 64-byte line, read as four 16-byte loads),
// then wavefront sums, then those in order.  Result in out[0..kNumRed)
// (shared memory); ends with a barrier.  The rows are 64-byte aligned (kNumRed = 8 doubles).
template <int NT>
__device__ inline void sum_partials(const double *partials, int rows, double *out)
{
  static_assert(kNumRed == 8, "a partial row is four 16-byte vectors");
  typedef double d2 __attribute__((ext_vector_type(2)));
  __shared__ double sh[NT / 64][kNumRed];
  const int t = threadIdx.x;
  const d2 *P = (const d2 *)partials;
  double v[kNumRed];
#pragma unroll
  for (int k = 0; k < kNumRed; ++k) v[k] = 0.0;
  // rows t, t + NT, t + 2 NT, ... in that order, U rows per batch with all their loads in flight (a
  // thread has at most U rows below U * NT rows, so those take one memory round trip)
  constexpr int U = 4;
  for (int r0 = t; r0 < rows; r0 += U * NT) {
    d2 q[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r0 + u * NT < rows)
#pragma unroll
        for (int k = 0; k < 4; ++k) q[u][k] = P[(size_t)(r0 + u * NT) * 4 + k];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r0 + u * NT < rows)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[2 * k] += q[u][k].x;
          v[2 * k + 1] += q[u][k].y;
        }
  }
#pragma unroll
  for (int k = 0; k < kNumRed; ++k) v[k] = wave_sum(v[k]);
  if ((t & 63) == 0)
#pragma unroll
    for (int k = 0; k < kNumRed; ++k) sh[t >> 6][k] = v[k];
  __syncthreads();
  if (t < kNumRed) {
    double s = 0.0;
    for (int w = 0; w < NT / 64; ++w) s += sh[w][t];
    out[t] = s;
  }
  __syncthreads();
}

// One background operation (UpdateOp), executed by one thread.  red: finished volume averages (sums / N^3) of
// the last pass.  a_drift > 0: the drift coefficients use this scale factor instead of aSI.
// Averages first, then one evaluation of the scale-factor kernel for every operation that needs it, then what it
// moves: this is compiled into every reducing pass (pass_tail.hpp), and seven copies of the kernel were 4 KB of it.
template <bool INT>
__device__ __forceinline__ void apply_op(DevState *st, const double *red, const ModelConsts &mc, const int op,
                                         const double w, double &a_drift)
{
  clmi_background &b = st->bg;
  const double dt = mc.dt;
  bool kernel = false;
  double g2 = b.grad2AvI, cg2 = b.CSgrad2AvI, b2 = b.U1Mag2AvI;  // the kernel's averages, where not the integer-time ones
  switch (op) {
    case OP_STORE_FIELDS:  // leapfrog.h:269-277
      if (mc.ns > 0) b.grad2AvI = red[RED_GRAD2S];
      if (mc.ncs > 0) b.CSgrad2AvI = red[RED_GRAD2CS];
      if (mc.nu1 > 0) b.U1Mag2AvI = red[RED_B2U1];
      b.potAvI = red[RED_POT];
      break;
    case OP_LF_MOMENTA:  // leapfrog.h:239-267
      if (mc.ns > 0) {
        b.pi2AvSIM = b.pi2AvSI;
        b.pi2AvSI = red[RED_PI2S];
        b.pi2AvI = 0.5 * (b.pi2AvSIM + b.pi2AvSI);
      }
      if (mc.ncs > 0) {
        b.CSpi2AvSIM = b.CSpi2AvSI;
        b.CSpi2AvSI = red[RED_PI2CS];
        b.CSpi2AvI = 0.5 * (b.CSpi2AvSIM + b.CSpi2AvSI);
      }
      if (mc.nu1 > 0) {
        b.U1pi2AvSIM = b.U1pi2AvSI;
        b.U1pi2AvSI = red[RED_PI2U1];
        b.U1pi2AvI = 0.5 * (b.U1pi2AvSIM + b.U1pi2AvSI);
      }
      kernel = true;
      break;
    case OP_LF_SYNC:  // leapfrog.h:105-112
      kernel = true;
      [[fallthrough]];
    case OP_VV_MOMENTA:  // velocityverlet.h:249-256
      if (mc.ns > 0) b.pi2AvI = red[RED_PI2S];
      if (mc.ncs > 0) b.CSpi2AvI = red[RED_PI2CS];
      if (mc.nu1 > 0) b.U1pi2AvI = red[RED_PI2U1];
      break;
    case OP_LF_INIT:      // leapfrog.h:35
    case OP_VV_SF_HALF:   // velocityverlet.h:165-168
    case OP_VV_SF_ONE:    // velocityverlet.h:171-174
    case OP_KERNEL_ONLY:
      kernel = true;
      break;
    case OP_VV_MOMENTA_KICK2:  // velocityverlet.h:249-256
      if (mc.ncs == 0) b.pi2AvI = red[RED_PI2S_KICK2];
      if (mc.ncs > 0) b.CSpi2AvI = red[RED_PI2CS_KICK2];
      if (mc.nu1 > 0) b.U1pi2AvI = red[RED_PI2U1_KICK2];
      break;
    case OP_VV_DRIFT_SF:  // velocityverlet.h:239-242
      b.aIM = b.aI;
      b.aI += dt * b.aDotSI * w;
      b.aSI = (b.aIM + b.aI) / 2.0;
      break;
    case OP_SET_ALL:  // averages.h:86-116
      b.potAvI = red[RED_POT];
      b.potAvSI = b.potAvI;
      if (mc.ns > 0) {
        b.pi2AvI = red[RED_PI2S];
        b.pi2AvSI = b.pi2AvI;
        b.grad2AvI = red[RED_GRAD2S];
      }
      if (mc.nu1 > 0) {
        b.U1pi2AvI = red[RED_PI2U1];
        b.U1pi2AvSI = b.U1pi2AvI;
        b.U1Mag2AvI = red[RED_B2U1];
      }
      if (mc.ncs > 0) {
        b.CSpi2AvI = red[RED_PI2CS];
        b.CSpi2AvSI = b.CSpi2AvI;
        b.CSgrad2AvI = red[RED_GRAD2CS];
      }
      break;
    case OP_PV_SF_FIRST:  // positionverlet.h:196-209; the first drift of the stage uses aI before it
      a_drift = b.aI;
      b.aIM = b.aI;
      b.aI += dt / 2.0 * b.aDotI * w;
      b.aSI = b.aI;
      break;
    case OP_PV_MID: {  // positionverlet.h:73-94
      // storeFieldsAveragesHalf (positionverlet.h:258-266): the half-step field averages feed getSI
      g2 = red[RED_GRAD2S], cg2 = red[RED_GRAD2CS], b2 = red[RED_B2U1];
      b.potAvSI = red[RED_POT];
      // storeMomentaAverages (positionverlet.h:238-256)
      const double pIM = b.pi2AvI, cIM = b.CSpi2AvI, uIM = b.U1pi2AvI;
      if (mc.ns > 0) b.pi2AvI = red[RED_PI2S];
      if (mc.ncs > 0) b.CSpi2AvI = red[RED_PI2CS];
      if (mc.nu1 > 0) b.U1pi2AvI = red[RED_PI2U1];
      b.pi2AvSI = 0.5 * (b.pi2AvI + pIM);
      b.CSpi2AvSI = 0.5 * (b.CSpi2AvI + cIM);
      b.U1pi2AvSI = 0.5 * (b.U1pi2AvI + uIM);
      kernel = true;
      break;
    }
    case OP_PV_DRIFT_AI:
      a_drift = b.aI;
      break;
    default:
      break;
  }
  if (!kernel) return;
  const bool si = op == OP_PV_MID;  // ScaleFactorKernels::getSI (positionverlet.h:151-154), else ::get
  const double K = sf_kernel_of<INT>(b.aI, si ? b.pi2AvSI : b.pi2AvI, g2, si ? b.CSpi2AvSI : b.CSpi2AvI, cg2,
                                     si ? b.U1pi2AvSI : b.U1pi2AvI, b2, si ? b.potAvSI : b.potAvI, mc);
  st->K = K;
  switch (op) {
    case OP_LF_MOMENTA:  // leapfrog.h:124-129 and 168-184
      b.aDotSIM = b.aDotSI;
      b.aDotSI += dt * K;
      b.aDotI = (b.aDotSIM + b.aDotSI) / 2.0;
      b.aIM = b.aI;
      b.aI += dt * b.aDotSI;
      b.aSI = (b.aIM + b.aI) / 2.0;
      break;
    case OP_LF_SYNC:
      b.aDotI = b.aDotSI + dt / 2.0 * K;
      break;
    case OP_LF_INIT:
      b.aDotSI = b.aDotI - dt / 2.0 * K;
      break;
    case OP_VV_SF_HALF:
      b.aDotSI = b.aDotI + (dt / 2) * K * w;
      break;
    case OP_VV_SF_ONE:
      b.aDotI = b.aDotSI + (dt / 2) * K * w;
      break;
    case OP_PV_MID:
      b.aDotI += dt * K * w;
      // driftScaleFactorSecondHalf (positionverlet.h:212-223); the second drift uses the new aI
      b.aI += dt / 2.0 * b.aDotI * w;
      b.aSI = (b.aIM + b.aI) / 2.0;
      a_drift = b.aI;
      break;
    default:
      break;
  }
}

// The kick and drift coefficients the next pass reads: a^(1+alpha) and a^(3+alpha) = a^(1+alpha) a^2,
// a^(alpha-1); the drift factors likewise share one power.
template <bool INT>
__device__ __forceinline__ void refresh_coefficients(DevState *st, const ModelConsts &mc, double a_drift)
{
  const clmi_background &b = st->bg;
  const double aK = bg_pow<INT>(b.aI, 1 + mc.alpha);
  st->aK = aK;
  st->aV = aK * (b.aI * b.aI);
  st->aG = bg_pow<INT>(b.aI, mc.alpha - 1);
  st->aJ = aK;
  const double ad = a_drift > 0.0 ? a_drift : b.aSI;
  const double fu = bg_pow<INT>(ad, mc.alpha - 1);
  st->fdrift_u = fu;
  st->fdrift_s = fu / (ad * ad);
}

// Executed by one thread: the operations in order, then the coefficients.
template <bool INT>
__device__ __forceinline__ void apply_update(DevState *st, const double *red, const ModelConsts &mc, const UpdateOps &ops)
{
  double a_drift = -1.0;
  for (int o = 0; o < ops.n; ++o) {
    apply_op<INT>(st, red, mc, ops.op[o], ops.w[o], a_drift);
    if (o == 0 && ops.snap) *ops.snap = st->bg;
  }
  refresh_coefficients<INT>(st, mc, a_drift);
}

}  // namespace clmi
