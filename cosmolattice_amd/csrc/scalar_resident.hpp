// Resident evolver of the scalar-singlet lattices of side N <= 128 (kernel template; instantiated in
// scalar_resident_*.hip): one cooperative launch advances the lattice by many passes, with the fields and
// momenta in registers throughout.
//
// What bounds these lattices pass by pass is not HBM (128^3, two fields: 50-67 MB, a pass of 26 us and an
// update of 7-9 us plus two launch gaps) but the traffic and the launches of a step that need not
// leave the chip: 256 CUs hold 128 MB in vector registers.  So a workgroup keeps a tile -- a chunk of
// C = 512 VZ consecutive sites of a plane (row-major, whole rows or not) by P planes -- of every array in
// registers, eight 64-lane waves, VZ sites a lane and plane, and per pass exchanges with the other
// workgroups only
//   - the kicked momenta of its boundary sites (the halo's fields are kept by every reader and drifted
//     by the same operations on the same values as their owner's, so they agree to the bit), and
//   - its partial sums, which every workgroup reads to finish the volume sums and to advance the background
//     by itself, in the order the update kernel uses, with the same bits.
// Each 8-byte word of the sums carries half a double and the pass's epoch, so it is data and flag in one trip
// (64-bit stores are single transactions): a workgroup waits until all tiles' words show the epoch.  Word w
// of all tiles is contiguous, so a wave reads 64 tiles' words with one 512-byte access.  A workgroup writes its
// words after the barrier that follows every thread's wait for its own momentum stores, and
// all exchanged data goes through agent-scope accesses, which bypass the incoherent L2s; no cache is
// written back or invalidated.  Buffers alternate by parity: a workgroup can reach epoch e + 2 only after all
// have written epoch e + 1, which they do after their last read of epoch e.  They are the arrays that take the
// final state: a workgroup stores that when it has seen every workgroup's words of the last pass, after which nobody
// reads or writes exchanged momenta.
//
// The launch is cooperative, but that check knows nothing of what else holds the device's CUs (another process's
// launch of this kind may wait for ours), so a workgroup first arrives at a gate.  The last to arrive opens it; one
// that waits there for kGateLimit polls (about a second) closes it, whichever comes first, and the host learns which.
// Behind a closed one every workgroup stores the state as it loaded it, so that what the host has queued meanwhile finds
// a state in the arrays that take it; the host then runs the same passes one by one.  Behind an open gate every
// workgroup is on the chip and every wait ends; kSpinLimit is there so that the grid drains even if the device itself
// fails, and the state is lost then (the host reports it).  The gate costs 1 to 2 us a launch.
//
// Measured (MI355X, us per leapfrog pass, resident against pass and update launches; VV2 in brackets):
//   64^3  one field  FP64 6.0 / 15.0 (6.6 / 16.6)    two fields FP32-bulk 7.3 / 18.2 (7.8 / 19.8)
//   128^3 one field  FP64 11.8 / 23.5 (12.6 / 25.1)  two fields FP32-bulk 16.0 / 36.8 (16.9 / 33.6)
//   128^3 two fields FP64 17.7 / 36.3 (19.0 / 40.3)
// A 128^3 FP64 pass of 40k cycles spends 16k on drift and stencil (issue of FP64 at two waves a SIMD), 4k on the
// tile's sums, 13-15k on the round trip of the sums (2.7 us at 256 workgroups for an empty exchange), 5k on the
// halo's and 2k on the background update's serial chain.
//
// Partial sums: one row per tile at row group * chunks + chunk, each thread summing its sites over the P
// planes, then the wave sums, those in order -- the rows of the full-row pass for N = 64 and 128
// (C = 8 rows, P = 8 = its G).
#pragma once

#include <type_traits>

#include "scalar_site.hpp"
#include "update_device.hpp"

namespace clmi {
namespace {

constexpr int kSpinLimit = 1 << 22, kGateLimit = 1 << 20;

__device__ __forceinline__ void decide_gate(const ResidentArgs &r, uint32_t want)
{
  uint32_t was = r.shut;
  if (__hip_atomic_compare_exchange_strong(&r.gate->word, &was, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT))
    __hip_atomic_store(&r.host->word, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// By one thread of every workgroup: arrive, and (later) wait for the decision; whether the gate opened.
__device__ __forceinline__ void arrive_at_gate(const ResidentArgs &r)
{
  const uint32_t n = __hip_atomic_fetch_add(&r.gate->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  if (r.refuse) decide_gate(r, r.shut + 2);
  else if (n == r.arrived) decide_gate(r, r.shut + 1);
}
__device__ __forceinline__ bool pass_gate(const ResidentArgs &r)
{
  for (int spin = 0;; ++spin) {
    const uint32_t w = __hip_atomic_load(&r.gate->word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (w != r.shut) return w == r.shut + 1;
    if (spin >= kGateLimit) decide_gate(r, r.shut + 2);  // (or somebody else has by now: the next poll shows it)
  }
}

__device__ __forceinline__ void xstore64(uint64_t *p, uint64_t v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t xload64(const uint64_t *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Exchanged momenta: VZ consecutive ones at uniform element offset o plus the lane's element offset i of an
// exchange buffer, through the coherence point.  Buffer accesses take the uniform part as a scalar, so a
// lane holds one 32-bit offset for all planes, and a lane's two FP64 momenta are one 16-byte access.
constexpr int kSc1 = 16;  // cache policy: device scope
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
template <int VZ, class M>
__device__ __forceinline__ void xstore(__amdgpu_buffer_rsrc_t b, uint32_t o, uint32_t i, const M (&v)[VZ])
{
  const int vo = (int)(i * (uint32_t)sizeof(M)), so = (int)(o * (uint32_t)sizeof(M));
  if constexpr (VZ * sizeof(M) == 16) {
    const u2v x = __builtin_bit_cast(u2v, v[0]), y = __builtin_bit_cast(u2v, v[1]);
    __builtin_amdgcn_raw_buffer_store_b128(u4v{x.x, x.y, y.x, y.y}, b, vo, so, kSc1);
  } else if constexpr (sizeof(M) == 8) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, v[0]), b, vo, so, kSc1);
  } else if constexpr (VZ == 2) {
    __builtin_amdgcn_raw_buffer_store_b64(u2v{__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1])}, b,
                                          vo, so, kSc1);
  } else {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[0]), b, vo, so, kSc1);
  }
}
template <int VZ, class M>
__device__ __forceinline__ void xload(__amdgpu_buffer_rsrc_t b, uint32_t o, uint32_t i, M (&v)[VZ])
{
  const int vo = (int)(i * (uint32_t)sizeof(M)), so = (int)(o * (uint32_t)sizeof(M));
  if constexpr (VZ * sizeof(M) == 16) {
    const u4v q = __builtin_amdgcn_raw_buffer_load_b128(b, vo, so, kSc1);
    v[0] = __builtin_bit_cast(M, u2v{q.x, q.y});
    v[1] = __builtin_bit_cast(M, u2v{q.z, q.w});
  } else if constexpr (sizeof(M) == 8) {
    const u2v q = __builtin_amdgcn_raw_buffer_load_b64(b, vo, so, kSc1);
    v[0] = __builtin_bit_cast(M, q);
  } else if constexpr (VZ == 2) {
    const u2v q = __builtin_amdgcn_raw_buffer_load_b64(b, vo, so, kSc1);
    const uint32_t x = q.x, y = q.y;  // (a bit cast of a vector's element takes its first one)
    v[0] = __builtin_bit_cast(M, x);
    v[1] = __builtin_bit_cast(M, y);
  } else {
    const uint32_t q = __builtin_amdgcn_raw_buffer_load_b32(b, vo, so, kSc1);
    v[0] = __builtin_bit_cast(M, q);
  }
}

// SZ bytes (4 or 16) per lane at byte offset bo + uniform byte offset uo of an exchange buffer, straight into LDS:
// lane l's bytes go to lds + l SZ (lds uniform over the wave).
template <int SZ>
__device__ __forceinline__ void xload_lds(__amdgpu_buffer_rsrc_t b, uint32_t uo, uint32_t bo, void *lds)
{
  const auto l = (__attribute__((address_space(3))) void *)lds;
  if constexpr (SZ == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(b, l, 16, (int)bo, (int)uo, 0, kSc1);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(b, l, 4, (int)bo, (int)uo, 0, kSc1);
}

// The value itself, which the compiler must take as new: an LDS address formed from it is not moved out of the
// pass loop.  Without this every plane's every neighbour address is a register for the whole launch (about
// 100 with eight planes of two fields) instead of an offset in the instruction.
__device__ __forceinline__ int fresh(int v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// Values that must have been computed by this point.  Within a basic block instruction selection places arithmetic
// near its use, also across barriers and scheduling barriers; without these the unrolled planes' neighbour
// values pile up (150 to 400 spilled registers with two fields).
__device__ __forceinline__ void settle(double &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void settle(float &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void settle(float2 &v)
{
  settle(v.x);
  settle(v.y);
}

// The factors of sf_kernel_of that depend on the scale factor alone, and the kernel of scalar singlets from them:
// the same operations in the same order, split so that the divisions and powers run while the sums travel.
struct ScaleTerms {
  double ia2, ia6, A;
};
__device__ __forceinline__ ScaleTerms scale_terms(double a, const ModelConsts &mc)
{
  ScaleTerms t;
  const double ia = 1.0 / a, ia2 = ia * ia, ia4 = ia2 * ia2;
  t.ia2 = ia2;
  t.ia6 = ia4 * ia2;
  const double fm = mc.fStar / mc.MPl;
  t.A = bg_pow<true>(a, 2 * mc.alpha + 1) / 3.0 * (fm * fm);
  return t;
}
__device__ __forceinline__ double scale_kernel(const ScaleTerms &t, double pi2, double grad2, double pot,
                                               const ModelConsts &mc)
{
  const double Eks = 0.5 * pi2 * t.ia6, Egs = 0.5 * grad2 * t.ia2;
  return t.A * ((mc.alpha - 2) * (Eks + 0.0) + mc.alpha * (Egs + 0.0) + (mc.alpha - 1) * (0.0 + 0.0) +
                (mc.alpha + 1) * pot);
}

// The background operations that the pass-by-pass evolvers put into a pass's update launch (apply_op's, for scalar
// singlets), then the coefficients.  t: of the aI before them.
template <int SCH, bool KICK>
__device__ __forceinline__ void resident_update(DevState &s, const double *red, const ModelConsts &mc,
                                                const ScaleTerms &t, double w, double w2, bool last)
{
  clmi_background &b = s.bg;
  const double dt = mc.dt;
  double a_drift = -1.0;
  if constexpr (SCH == RES_LF) {  // OP_STORE_FIELDS, OP_LF_MOMENTA
    const double g2 = red[RED_GRAD2S], pot = red[RED_POT], old = b.pi2AvSI, now = red[RED_PI2S];
    const double mid = 0.5 * (old + now);
    const double K = scale_kernel(t, mid, g2, pot, mc);
    const double d0 = b.aDotSI, d1 = d0 + dt * K, a0 = b.aI, a1 = a0 + dt * d1;
    b.grad2AvI = g2;
    b.potAvI = pot;
    b.pi2AvSIM = old;
    b.pi2AvSI = now;
    b.pi2AvI = mid;
    s.K = K;
    b.aDotSIM = d0;
    b.aDotSI = d1;
    b.aDotI = (d0 + d1) / 2.0;
    b.aIM = a0;
    b.aI = a1;
    b.aSI = (a0 + a1) / 2.0;
  } else if constexpr (SCH == RES_VV) {
    // OP_STORE_FIELDS, OP_VV_MOMENTA, OP_VV_SF_ONE, OP_VV_SF_HALF, OP_VV_MOMENTA_KICK2, OP_VV_DRIFT_SF
    const double g2 = red[RED_GRAD2S], pot = red[RED_POT];
    const double K = scale_kernel(t, red[RED_PI2S], g2, pot, mc);  // of both half-steps: only aDot changes between
    const double d1 = b.aDotSI + (dt / 2) * K * w, d2 = d1 + (dt / 2) * K * w2;
    const double a0 = b.aI, a1 = a0 + dt * d2 * w2;
    b.grad2AvI = g2;
    b.potAvI = pot;
    s.K = K;
    b.aDotI = d1;
    b.aDotSI = d2;
    b.pi2AvI = red[RED_PI2S_KICK2];
    b.aIM = a0;
    b.aI = a1;
    b.aSI = (a0 + a1) / 2.0;
  } else if constexpr (KICK) {  // OP_PV_MID
    const double g2 = red[RED_GRAD2S], pot = red[RED_POT], old = b.pi2AvI, now = red[RED_PI2S];
    const double mid = 0.5 * (now + old);
    const double K = scale_kernel(t, mid, g2, pot, mc);
    const double d1 = b.aDotI + dt * K * w, a1 = b.aI + dt / 2.0 * d1 * w;
    b.potAvSI = pot;
    b.pi2AvI = now;
    b.pi2AvSI = mid;
    b.CSpi2AvSI = 0.5 * (b.CSpi2AvI + b.CSpi2AvI);
    b.U1pi2AvSI = 0.5 * (b.U1pi2AvI + b.U1pi2AvI);
    s.K = K;
    b.aDotI = d1;
    b.aSI = (b.aIM + a1) / 2.0;
    b.aI = a1;
    a_drift = a1;
  } else {  // OP_STORE_FIELDS, OP_PV_SF_FIRST
    b.grad2AvI = red[RED_GRAD2S];
    b.potAvI = red[RED_POT];
    if (!last) {
      a_drift = b.aI;
      b.aIM = b.aI;
      b.aI += dt / 2.0 * b.aDotI * w2;
      b.aSI = b.aI;
    }
  }
  refresh_coefficients<true>(&s, mc, a_drift);
}

// SCH: the passes of a launch are all drift + kick passes (leapfrog; a.cdt, a.ckick), all double-kick passes
// (velocity Verlet: pass m drifts and kicks by stage m, then kicks by stage m + 1), or alternately
// drift + kick and drift passes (position Verlet, two per stage).  The single kick that opens or closes
// a call runs as an ordinary pass.  RAG: some tiles have fewer planes or sites than P and C.
template <int NF, bool F32, int VZ, int P, bool RAG, int PK, int SCH>
__global__ __launch_bounds__(kResThreads) void k_scalar_resident(const ResidentArgs r)
{
  using T = Tr<F32>;
  using V = typename T::V;
  using M = typename T::P;
  constexpr int NT = kResThreads, C = NT * VZ, NMAX = 64 * VZ, NW = NT / 64;
  constexpr bool K2 = SCH == RES_VV;
  constexpr int NS = K2 ? 4 : 3;  // sums: pi^2, |grad phi|^2, V, pi^2 after the second kick
  // Planes written to LDS before a barrier: all, or half where all would not fit beside the halo.
  constexpr int B = NF * VZ * P <= 16 ? P : P / 2;
  // Plane by plane, or (where the registers hold it) all planes of a batch interleaved: one site per lane
  // and plane alone is a serial chain of FP64 operations.
  constexpr bool STEP = NF * VZ * P > 8;
  // Where the state alone takes half the registers (two fields, two sites, eight planes), the halo's momenta
  // wait in LDS, in the planes' buffers, which are free between passes: x[side][field][site], then
  // y[pair of planes][site], one slot per thread.
  constexpr bool STAGE = NF * VZ * P >= 32;
  constexpr int XB = 2 * NF * VZ * NT * (int)sizeof(M);
  static_assert(!STAGE || VZ == 2, "16-byte pairs");
  static_assert(2 * NMAX * NF <= NT, "two halo sites per thread and pair of planes");
  __shared__ V tile[B][NF][C + 2 * NMAX];
  // halo fields, each thread its own slots: the planes before and after the tile (hx[0], hx[1]) and two
  // in-plane halo sites of every other plane; in LDS so that two FP64 fields leave room for the rest in registers
  __shared__ V hx[2][NF][VZ][NT];
  __shared__ V hy[P / 2][2][NT];
  __shared__ double wsum[NW][4];
  __shared__ DevState S;
  __shared__ ModelConsts MC;  // in LDS, and read through fresh(), so that nothing derived from it sits in registers
  __shared__ ScaleTerms pre;
  __shared__ int dead;

  const ScalarPassArgs &a = r.a;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int N = a.N;
  const uint32_t NN = (uint32_t)N * N;
  const int tiles = r.groups * r.chunks;
  const int grp = blockIdx.x / r.chunks, chk = blockIdx.x % r.chunks;
  const int start = chk * C, nc = RAG ? min(C, (int)NN - start) : C;
  const int x0 = grp * P, nx = RAG ? min(P, N - x0) : P;
  const int pf = RAG ? P - nx : 0;  // planes sit in slots pf .. P - 1
  // lanes past the chunk's end work on its first site again; their results are dropped
  const bool act = !RAG || tid * VZ < nc;
  const int i0 = act ? tid * VZ : 0;
  const int z = (start + i0) % N;
  // indices into a plane's LDS row: N halo sites, the chunk, N halo sites
  const int ic = N + i0;
  const int izl = ic + (z == 0 ? N - 1 : -1), izr = ic + VZ - 1 + (z + VZ == N ? 1 - N : 1);
  // this thread's in-plane halo: two consecutive sites of one field, of every other plane (slots 2 j + hp)
  const bool hact = tid < 2 * N * NF;
  const int hq = hact ? tid : 0, hp = hq / (N * NF), hf = hq % (N * NF) / N, hh = 2 * (hq % N);
  const int hidx = hh < N ? hh : nc + hh;
  uint32_t hs;
  {
    int h = hh < N ? start - N + hh : start + nc + hh - N;
    h = h < 0 ? h + (int)NN : (h >= (int)NN ? h - (int)NN : h);
    hs = (uint32_t)h;
  }
  // sites that another chunk's halo holds
  const bool edge = act && (i0 < N || i0 + VZ > nc - N);
  auto plane = [&](int x) -> uint32_t { return (uint32_t)(x < 0 ? x + N : (x >= N ? x - N : x)) * NN; };
  // array offsets: a uniform one of each plane plus this thread's site in it
  const uint32_t own = (uint32_t)(start + i0);
  const uint32_t offl = plane(x0 - 1), offr = plane(x0 + nx);
  const int off0 = (x0 - pf) * (int)NN;  // slot p: off0 + p NN
  auto slot = [&](int p) -> uint32_t { return (uint32_t)(off0 + p * (int)NN); };
  auto has = [&](int p) -> bool { return !RAG || p >= pf; };

  if (tid == 0) {
    arrive_at_gate(r);
    S = *r.st;
    MC = r.mc;
  }

  V phi[P][NF][VZ];
  M pi[P][NF][VZ];
  M xhp[2][NF][VZ], yhp[P / 2][2];  // halo momenta (not STAGE)
  char *const stage = (char *)&tile[0][0][0];
  static_assert(!STAGE || XB + P * NT * (int)sizeof(M) <= (int)sizeof(tile), "the halo's momenta fit the planes' buffers");
  // (FP64 pairs as the 16 bytes that one load to LDS writes, FP32 momenta one by one)
  auto xslot = [&](int d, int f, int k, int t) -> M & {
    if constexpr (sizeof(M) == 8) return ((M *)stage)[((d * NF + f) * NT + t) * VZ + k];
    else return ((M *)stage)[((d * NF + f) * VZ + k) * NT + t];
  };
  auto yslot = [&](int j, int k, int t) -> M & {
    if constexpr (sizeof(M) == 8) return ((M *)(stage + XB))[(j * NT + t) * 2 + k];
    else return ((M *)(stage + XB))[(j * 2 + k) * NT + t];
  };

  auto load_phi = [&](int f, uint32_t s, V (&o)[VZ]) {
    if constexpr (!F32) {
      vload<VZ>((const double *)a.phi_in[f], s, o);
    } else {
      float h[VZ], l[VZ];
      vload<VZ>((const float *)a.phi_in[f], s, h);
      vload<VZ>(a.philo_in[f], s, l);
#pragma unroll
      for (int k = 0; k < VZ; ++k) o[k] = make_float2(h[k], l[k]);
    }
  };
#pragma unroll
  for (int f = 0; f < NF; ++f) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const uint32_t s = (has(p) ? slot(p) : slot(P - 1)) + own;  // an unused slot repeats the last plane
      load_phi(f, s, phi[p][f]);
      vload<VZ>((const M *)a.pi_in[f], s, pi[p][f]);
    }
    V o[VZ];
    load_phi(f, offl + own, o);
#pragma unroll
    for (int k = 0; k < VZ; ++k) hx[0][f][k][tid] = o[k];
    load_phi(f, offr + own, o);
#pragma unroll
    for (int k = 0; k < VZ; ++k) hx[1][f][k][tid] = o[k];
    vload<VZ>((const M *)a.pi_in[f], offl + own, xhp[0][f]);
    vload<VZ>((const M *)a.pi_in[f], offr + own, xhp[1][f]);
    if constexpr (STAGE)
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int k = 0; k < VZ; ++k) xslot(d, f, k, tid) = xhp[d][f][k];
  }
#pragma unroll
  for (int j = 0; j < P / 2; ++j) {
    const bool on = hact && has(2 * j + hp);
    const uint32_t s = on ? slot(2 * j + hp) + hs : 0;
    M q[2];
    vload<2>((const M *)a.pi_in[hf], s, q);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if constexpr (!F32) hy[j][k][tid] = ((const double *)a.phi_in[hf])[s + k];
      else hy[j][k][tid] = make_float2(((const float *)a.phi_in[hf])[s + k], a.philo_in[hf][s + k]);
      if constexpr (STAGE) yslot(j, k, tid) = q[k];
      else yhp[j][k] = q[k];
    }
  }
  if (tid == 0) dead = !pass_gate(r);
  auto store_state = [&]() {
    if (act)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (has(p)) {
            const uint32_t s = slot(p) + own;
            vstore<VZ, false>((M *)a.pi_out[f], s, pi[p][f]);
            if constexpr (!F32) {
              vstore<VZ, false>((double *)a.phi_out[f], s, phi[p][f]);
            } else {
              float h[VZ], l[VZ];
#pragma unroll
              for (int k = 0; k < VZ; ++k) {
                h[k] = phi[p][f][k].x;
                l[k] = phi[p][f][k].y;
              }
              vstore<VZ, false>((float *)a.phi_out[f], s, h);
              vstore<VZ, false>(a.philo_out[f], s, l);
            }
          }
  };
  __syncthreads();
  if (dead) {
    store_state();
    if (blockIdx.x == 0 && tid == 0) *r.closed_st = S;
    return;
  }

  const bool red = r.mc.expansion != 0;
  const double dt = r.mc.dt;
  const int stages = 2 * (r.nws - 1) + 1;
  auto weight = [&](int k) {  // composition weight of stage k of the launch
    const int s = k % stages;
    return r.ws[s < r.nws ? s : stages - s - 1];
  };

  // One pass (its number, weights and coefficients); false: the workgroups lost each other.
  auto pass = [&](auto kickc, const int m, const double w, const double w2, const double cdt, const double ck,
                  const double ck2) -> bool {
    constexpr bool KICK = decltype(kickc)::value;
    const uint32_t epoch = r.epoch0 + 1 + (uint32_t)m;
    const bool last = m + 1 == r.passes;
    // momenta of this kick, or of the last one (position Verlet's drift passes): alternate buffers
    const bool odd = ((SCH == RES_PV ? m >> 1 : m) & 1) != 0;
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
        odd ? r.xch[1] : r.xch[0], 0, (int)((uint32_t)NF * a.V * (uint32_t)sizeof(M)), 0x00027000);
    const double fs = S.fdrift_s;
    const SiteK kc = site_consts(ck, ck2, S.aK, S.aV, a.inv_dx, a.inv_dx2);
    const int ft = fresh(tid);
    // Drift, the halo first: its momenta's registers are free for the rest of the pass.
    const float cf = (float)(fs * cdt);
    if constexpr (STAGE) __builtin_amdgcn_s_waitcnt(0);  // this wave's loads to LDS
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int k = 0; k < VZ; ++k) {
          M q;
          if constexpr (STAGE) q = xslot(d, f, k, ft);
          else q = xhp[d][f][k];
          V h = hx[d][f][k][ft];
          drift_value(h, q, fs, cdt, cf);
          hx[d][f][k][ft] = h;
        }
#pragma unroll
    for (int j = 0; j < P / 2; ++j)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        M q;
        if constexpr (STAGE) q = yslot(j, k, ft);
        else q = yhp[j][k];
        V h = hy[j][k][ft];
        drift_value(h, q, fs, cdt, cf);
        hy[j][k][ft] = h;
      }
    if constexpr (STAGE) __syncthreads();  // the planes take the buffers again
#pragma unroll
    for (int p = 0; p < P; ++p) {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int k = 0; k < VZ; ++k) {
          drift_value(phi[p][f][k], pi[p][f][k], fs, cdt, cf);
          if constexpr (STEP) settle(phi[p][f][k]);
        }
    }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    // boundary momenta: the first and last plane, and of the others the sites in a chunk's halo
    auto publish = [&](int p) {
      const bool face = p == P - 1 || (RAG ? p == pf : p == 0);
      if (has(p) && (edge || (face && act)))
#pragma unroll
        for (int f = 0; f < NF; ++f) xstore<VZ>(xb, (uint32_t)f * a.V + slot(p), own, pi[p][f]);
    };
#pragma unroll
    for (int b = 0; b < P; b += B) {
      if (b > 0) __syncthreads();  // every read of the planes before
#pragma unroll
      for (int p = b; p < b + B; ++p) {
        auto &t = tile[p - b];
        const int jc = fresh(i0) + N, jh = fresh(hidx), jt = fresh(tid);
        if (act)
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < VZ; ++k) t[f][jc + k] = phi[p][f][k];
        if (hact && hp == (p & 1)) {
          t[hf][jh] = hy[p / 2][0][jt];
          t[hf][jh + 1] = hy[p / 2][1][jt];
        }
      }
      __syncthreads();
#pragma unroll
      for (int p = b; p < b + B; ++p) {
        if (!has(p)) continue;
        const auto &t = tile[p - b];
        const int jm = fresh(i0), jl = fresh(izl), jr = fresh(izr), jt = fresh(tid);
        double p2 = 0.0, g2 = 0.0, vs = 0.0, p2b = 0.0;
#pragma unroll
        for (int k = 0; k < VZ; ++k) {
          V c[NF], xp[NF], xm[NF], yp[NF], ym[NF], zp[NF], zm[NF];
          M pk[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            c[f] = phi[p][f][k];
            xp[f] = p + 1 < P ? phi[p + 1 < P ? p + 1 : p][f][k] : hx[1][f][k][jt];
            if (p == 0 || (RAG && p == pf))
              xm[f] = hx[0][f][k][jt];
            else
              xm[f] = phi[p > 0 ? p - 1 : 0][f][k];
            yp[f] = t[f][jm + 2 * N + k];
            ym[f] = t[f][jm + k];
            zp[f] = k + 1 < VZ ? phi[p][f][k + 1 < VZ ? k + 1 : k] : t[f][jr];
            zm[f] = k > 0 ? phi[p][f][k > 0 ? k - 1 : k] : t[f][jl];
            pk[f] = pi[p][f][k];
          }
          site_update<NF, F32, PK, KICK, K2, true>(a.poly, kc, c, xp, xm, yp, ym, zp, zm, pk, p2, g2, vs, p2b);
#pragma unroll
          for (int f = 0; f < NF; ++f) pi[p][f][k] = pk[f];
        }
        acc[0] += p2;
        acc[1] += g2;
        acc[2] += vs;
        acc[3] += p2b;
        if constexpr (STEP) {
#pragma unroll
          for (int k = 0; k < NS; ++k) settle(acc[k]);
          if constexpr (KICK) {
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
              for (int k = 0; k < VZ; ++k) settle(pi[p][f][k]);
            publish(p);
          }
        }
      }
    }
    if constexpr (KICK && !STEP) {
#pragma unroll
      for (int p = 0; p < P; ++p) publish(p);
    }

    // partial sums of the tile (also without expansion: under a condition, the compiler would
    // move every site's energy terms, with the neighbours they read, behind it and out of the registers)
    double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NS; ++k) v[k] = wave_sum(act ? acc[k] : 0.0);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < 4; ++k) wsum[wave][k] = v[k];
    __builtin_amdgcn_s_waitcnt(0);  // this thread's exchange stores have reached the coherence point
    __syncthreads();
    uint64_t *const words = r.lines + (size_t)(epoch & 1) * tiles * 8;  // word w of tile t at w tiles + t
    if (tid < NS) {
      double sum = 0.0;
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) sum += wsum[wv][tid];
      const uint64_t bits = __builtin_bit_cast(uint64_t, sum);
      xstore64(words + (size_t)(2 * tid) * tiles + blockIdx.x, (bits << 32) | epoch);
      xstore64(words + (size_t)(2 * tid + 1) * tiles + blockIdx.x, (bits & 0xffffffff00000000ull) | epoch);
    }
    // What the background update takes from the scale factor alone, on a wave that has no words to read.
    if (red && tid == NT - 64) pre = scale_terms((&S)[fresh(0)].bg.aI, (&MC)[fresh(0)]);
    // all tiles' words
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = 0.0;
    if (tid < tiles) {
      for (int spin = 0;; ++spin) {
        uint64_t q[2 * NS];
#pragma unroll
        for (int k = 0; k < 2 * NS; ++k) q[k] = xload64(words + (size_t)k * tiles + tid);
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 2 * NS; ++k) ok = ok && (uint32_t)q[k] == epoch;
        if (ok) {
#pragma unroll
          for (int k = 0; k < NS; ++k)
            v[k] = __builtin_bit_cast(double, (q[2 * k] >> 32) | (q[2 * k + 1] & 0xffffffff00000000ull));
          break;
        }
        if (spin >= kSpinLimit) {
          dead = 1;
          break;
        }
      }
    }
    // the update kernel's order: thread t holds row t, wave sums, those in order
#pragma unroll
    for (int k = 0; k < NS; ++k) v[k] = wave_sum(v[k]);
    __syncthreads();  // every tile's words seen; wsum free
    if (dead) {
      if (tid == 0) __hip_atomic_store(&r.host->lost, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return false;
    }
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < NS; ++k) wsum[wave][k] = v[k];
    if (!last) {
      // halo momenta of the next drift (issued here so that they arrive during the background update)
      if constexpr (STAGE) {
        constexpr uint32_t MB = sizeof(M);
        const int uw = __builtin_amdgcn_readfirstlane(wave) * 64;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const uint32_t uo = ((uint32_t)f * a.V + (d ? offr : offl)) * MB;
            if constexpr (MB == 8) {
              xload_lds<16>(xb, uo, own * MB, &xslot(d, f, 0, uw));
            } else {
#pragma unroll
              for (int k = 0; k < VZ; ++k) xload_lds<4>(xb, uo, own * MB + 4u * k, &xslot(d, f, k, uw));
            }
          }
        if (hact)
#pragma unroll
          for (int j = 0; j < P / 2; ++j)
            if (has(2 * j + hp)) {
              const uint32_t bo = ((uint32_t)hf * a.V + (uint32_t)hp * NN + hs) * MB, uo = slot(2 * j) * MB;
              if constexpr (MB == 8) {
                xload_lds<16>(xb, uo, bo, &yslot(j, 0, uw));
              } else {
#pragma unroll
                for (int k = 0; k < 2; ++k) xload_lds<4>(xb, uo, bo + 4u * k, &yslot(j, k, uw));
              }
            }
      } else {
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int f = 0; f < NF; ++f) xload<VZ>(xb, (uint32_t)f * a.V + (d ? offr : offl), own, xhp[d][f]);
#pragma unroll
        for (int j = 0; j < P / 2; ++j)
          if (hact && has(2 * j + hp)) xload<2>(xb, slot(2 * j), (uint32_t)hf * a.V + (uint32_t)hp * NN + hs, yhp[j]);
      }
    }
    if (red) {
      __syncthreads();
      if (tid == 0) {
        double rd[kNumRed];
#pragma unroll
        for (int k = 0; k < kNumRed; ++k) rd[k] = 0.0;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
          double s = 0.0;
#pragma unroll
          for (int wv = 0; wv < NW; ++wv) s += wsum[wv][k];
          rd[k == 3 ? (int)RED_PI2S_KICK2 : k] = s * r.mc.invV;
        }
#pragma unroll
        for (int k = 0; k < kNumRed; ++k) S.red[k] = rd[k];
        resident_update<SCH, KICK>(S, rd, (&MC)[fresh(0)], pre, w, w2, last);
      }
    }
    __syncthreads();
    return true;
  };

  // (tested at the end: a loop that can end before its body keeps the state twice)
  int m = 0;
  bool ok;
  if constexpr (SCH == RES_LF) {
    do {
      ok = pass(std::true_type{}, m, 1.0, 1.0, dt, 1.0 * dt, 0.0);
    } while (++m < r.passes && ok);
  } else if constexpr (SCH == RES_VV) {
    do {
      const double w = weight(m), w2 = weight(m + 1);
      ok = pass(std::true_type{}, m, w, w2, dt * w, w * dt / 2, w2 * dt / 2);
    } while (++m < r.passes && ok);
  } else {
    do {
      const double w = weight(m >> 1);
      ok = pass(std::true_type{}, m, w, w, dt / 2 * w, w * dt, 0.0) &&
           pass(std::false_type{}, m + 1, w, weight((m >> 1) + 1), dt / 2 * w, 0.0, 0.0);
    } while ((m += 2) < r.passes && ok);
  }
  if (!ok) return;

  store_state();
  if (red && blockIdx.x == 0 && tid == 0) *r.st = S;
}

// The kernel for VZ sites per lane, P planes per tile and potential form pk (null: not instantiated).
template <int NF, bool F32, int SCH, int PK>
const void *resident_shape(const ResidentPlan &p)
{
  switch (p.VZ * 100 + p.P * 10 + (p.ragged ? 1 : 0)) {
    case 121: return (const void *)k_scalar_resident<NF, F32, 1, 2, true, PK, SCH>;
    case 141: return (const void *)k_scalar_resident<NF, F32, 1, 4, true, PK, SCH>;
    case 180: return (const void *)k_scalar_resident<NF, F32, 1, 8, false, PK, SCH>;
    case 241: return (const void *)k_scalar_resident<NF, F32, 2, 4, true, PK, SCH>;
    case 280: return (const void *)k_scalar_resident<NF, F32, 2, 8, false, PK, SCH>;
    case 281: return (const void *)k_scalar_resident<NF, F32, 2, 8, true, PK, SCH>;
    default: return nullptr;
  }
}
template <int NF, bool F32, int SCH>
const void *resident_kernel(const ResidentPlan &p, int pk)
{
  return pk == 1 ? resident_shape<NF, F32, SCH, 1>(p) : resident_shape<NF, F32, SCH, 0>(p);
}

}  // namespace
}  // namespace clmi
