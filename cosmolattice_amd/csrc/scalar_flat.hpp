// Plane-chunk scalar-singlet lattice pass (kernel template; instantiated in scalar_flat_*.hip): any even N up to
// 500 that the full-row and the 64-wide tiled passes do not take, with the same per-site arithmetic
// (bit-identical fields).
//
// Sides that are no multiple of 64 ran one site per thread with every neighbour read from cache: seven reads
// of the field and, drifting, seven of the momentum per site, which held 200^3 FP64 to 2.3 TB/s.  Here a
// workgroup owns C = 512 VZ consecutive sites of a plane in row-major order -- so every lane has work whatever
// N is, where tiles of rows or of 64 sites would leave 20-45 % of them idle at N = 100 or 200 -- and marches
// along x over XC planes like the full-row pass: x-neighbours in registers, the plane in a double-buffered
// LDS row of N halo sites, the chunk, and N halo sites, which holds all four in-plane neighbours of every site
// (rows wrap inside the halo).  Every array is read once per pass plus the halo (2 N / C of a plane, much of it
// from L2: the neighbouring chunk runs on the same XCD) and two planes per x-chunk.
//
// Measured (MI355X, leapfrog step, two fields; against one site per thread): 100^3 FP64 33.4 -> 21.5 us, 200^3 FP64
// 230 -> 119 us (4.3 TB/s of the arrays' bytes), 250^3 FP32-bulk 375 -> 190 us, 300^3 FP64 814 -> 386 us (4.5),
// 500^3 FP64 3906 -> 1744 us (4.6).  Non-temporal stores made no difference.  What bounds it is the memory path: halo rows that miss L2, and above 256^3
// the halo's share of the chunk.
//
// Volume sums are written per (group of G planes, chunk), independent of XC; for N <= 128 these are the tiles
// of the resident evolver, so its sums are the same.
#pragma once

#include "scalar_site.hpp"

namespace clmi {
namespace {

// NH: halo pairs per thread (N * NF pairs in all).
template <int NF, bool F32, int VZ, int NH, bool DRIFT, bool KICK, bool RED, int PK, bool KICK2 = false>
__global__ __launch_bounds__(kFlatThreads) void k_scalar_flat(const ScalarPassArgs a, const int XC, const int G,
                                                              const int chunks)
{
  static_assert(!KICK2 || (DRIFT && KICK), "a double kick follows a drift");
  using T = Tr<F32>;
  using V = typename T::V;
  using M = typename T::P;
  using Raw = typename T::template Raw<VZ>;
  using Raw2 = typename T::template Raw<2>;
  constexpr int NTH = kFlatThreads, C = NTH * VZ, NW = NTH / 64;
  extern __shared__ char lds_bytes[];
  V *const lds = (V *)lds_bytes;  // [2][NF][C + 2 N]

  const int N = a.N;
  const uint32_t NN = (uint32_t)N * N;
  const int W = C + 2 * N;
  const int nwg = gridDim.x, b = blockIdx.x;
  const int L = (nwg % 8 == 0) ? (b % 8) * (nwg / 8) + b / 8 : b;
  const int chk = L % chunks, x0 = L / chunks * XC, xe = min(x0 + XC, N);
  const int start = chk * C, nc = min(C, (int)NN - start);
  const int tid = threadIdx.x;
  // lanes past the chunk's end work on its first site again; their results are dropped
  const bool act = tid * VZ < nc;
  const int i0 = act ? tid * VZ : 0;
  const uint32_t own = (uint32_t)(start + i0);
  const int z = (int)(own % (uint32_t)N);
  const int ic = N + i0, izl = ic + (z == 0 ? N - 1 : -1), izr = ic + VZ - 1 + (z + VZ == N ? 1 - N : 1);
  // halo pairs of this thread: field, site in the plane, place in the LDS row
  bool hact[NH];
  int hf[NH], hidx[NH];
  uint32_t hs[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const int q = tid + h * NTH;
    hact[h] = q < N * NF;
    const int qq = hact[h] ? q : 0, hh = 2 * (qq % N);
    hf[h] = qq / N;
    hidx[h] = hf[h] * W + (hh < N ? hh : nc + hh);
    int s = hh < N ? start - N + hh : start + nc + hh - N;
    s = s < 0 ? s + (int)NN : (s >= (int)NN ? s - (int)NN : s);
    hs[h] = (uint32_t)s;
  }

  const double fs = DRIFT ? a.st->fdrift_s : 0.0;
  const float cf = DRIFT ? (float)(a.st->fdrift_s * a.cdt) : 0.0f;
  const SiteK kc = site_consts(a.ckick, a.ckick2, KICK ? a.st->aK : 0.0, KICK ? a.st->aV : 0.0, a.inv_dx, a.inv_dx2);
  auto plane = [&](int x) -> uint32_t { return (uint32_t)(x < 0 ? x + N : (x >= N ? x - N : x)) * NN; };

  V prev[NF][VZ], cur[NF][VZ], nxt[NF][VZ];
  M pic[NF][VZ], pin[NF][VZ];
  Raw pf[NF];
  Raw2 hq[NH];
  double acc[4] = {0.0, 0.0, 0.0, 0.0};

  auto load_halo = [&](uint32_t pl) {
#pragma unroll
    for (int h = 0; h < NH; ++h)
      if (hact[h]) T::template load<2>(a, hf[h], pl + hs[h], DRIFT, hq[h]);
  };
  auto put = [&](int buf) {  // plane in cur and its halo in hq
    V *const t = lds + buf * NF * W;
    if (act)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int k = 0; k < VZ; ++k) t[f * W + ic + k] = cur[f][k];
#pragma unroll
    for (int h = 0; h < NH; ++h)
      if (hact[h]) {
        t[hidx[h]] = T::template value<DRIFT>(hq[h], 0, fs, a.cdt, cf);
        t[hidx[h] + 1] = T::template value<DRIFT>(hq[h], 1, fs, a.cdt, cf);
      }
  };

  load_halo(plane(x0));
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    Raw q;
    T::load(a, f, plane(x0 - 1) + own, DRIFT, q);
#pragma unroll
    for (int k = 0; k < VZ; ++k) prev[f][k] = T::template value<DRIFT>(q, k, fs, a.cdt, cf);
    T::load(a, f, plane(x0) + own, true, q);
#pragma unroll
    for (int k = 0; k < VZ; ++k) {
      cur[f][k] = T::template value<DRIFT>(q, k, fs, a.cdt, cf);
      pic[f][k] = q.p[k];
    }
    T::load(a, f, plane(x0 + 1) + own, true, q);
#pragma unroll
    for (int k = 0; k < VZ; ++k) {
      nxt[f][k] = T::template value<DRIFT>(q, k, fs, a.cdt, cf);
      pin[f][k] = q.p[k];
    }
  }
  put(0);
  __syncthreads();

  for (int x = x0; x < xe; ++x) {
    const bool more = x + 1 < xe;
    if (more) {
#pragma unroll
      for (int f = 0; f < NF; ++f) T::load(a, f, plane(x + 2) + own, true, pf[f]);
      load_halo(plane(x + 1));
    }
    const V *const t = lds + ((x - x0) & 1) * NF * W;
    const uint32_t s0 = plane(x) + own;
    double p2 = 0.0, g2 = 0.0, vs = 0.0, p2b = 0.0;
    M pout[NF][VZ];
#pragma unroll
    for (int k = 0; k < VZ; ++k) {
      V c[NF], xp[NF], xm[NF], yp[NF], ym[NF], zp[NF], zm[NF];
      M pk[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const V *const tf = t + f * W;
        c[f] = cur[f][k];
        xp[f] = nxt[f][k];
        xm[f] = prev[f][k];
        yp[f] = tf[ic + N + k];
        ym[f] = tf[ic - N + k];
        zp[f] = k + 1 < VZ ? cur[f][k + 1 < VZ ? k + 1 : k] : tf[izr];
        zm[f] = k > 0 ? cur[f][k > 0 ? k - 1 : k] : tf[izl];
        pk[f] = pic[f][k];
      }
      site_update<NF, F32, PK, KICK, KICK2, RED>(a.poly, kc, c, xp, xm, yp, ym, zp, zm, pk, p2, g2, vs, p2b);
#pragma unroll
      for (int f = 0; f < NF; ++f) pout[f][k] = pk[f];
    }
    if (act) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if (KICK) vstore<VZ, false>((M *)a.pi_out[f], s0, pout[f]);
        if (DRIFT) {
          if constexpr (!F32) {
            vstore<VZ, false>((double *)a.phi_out[f], s0, cur[f]);
          } else {
            float h[VZ], l[VZ];
#pragma unroll
            for (int k = 0; k < VZ; ++k) {
              h[k] = cur[f][k].x;
              l[k] = cur[f][k].y;
            }
            vstore<VZ, false>((float *)a.phi_out[f], s0, h);
            vstore<VZ, false>(a.philo_out[f], s0, l);
          }
        }
      }
    }
    if (RED) {
      acc[0] += p2;
      acc[1] += g2;
      acc[2] += vs;
      if constexpr (KICK2) acc[3] += p2b;
      if ((x + 1) % G == 0 || x + 1 == N) {
        double v[kNumRed] = {act ? acc[0] : 0.0, act ? acc[1] : 0.0, act ? acc[2] : 0.0, 0, 0, 0, 0, 0};
        v[RED_PI2S_KICK2] = act ? acc[3] : 0.0;
        block_reduce_rows<NW, kNumRed>(v, a.partials + ((size_t)(x / G) * chunks + chk) * kNumRed);
        acc[0] = acc[1] = acc[2] = acc[3] = 0.0;
      }
    }
    if (more) {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int k = 0; k < VZ; ++k) {
          prev[f][k] = cur[f][k];
          cur[f][k] = nxt[f][k];
          pic[f][k] = pin[f][k];
          nxt[f][k] = T::template value<DRIFT>(pf[f], k, fs, a.cdt, cf);
          pin[f][k] = pf[f].p[k];
        }
      // the other buffer was last read in the previous iteration, before the barrier that ended it
      put((x + 1 - x0) & 1);
      __syncthreads();
    }
  }
  if constexpr (RED) finish_pass<NTH>(a.tail);
}

template <int NF, bool F32, int VZ, int NH, int PK>
hipError_t dispatch_flat(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p, hipStream_t s,
                         bool kick2)
{
  const size_t lds = 2 * (size_t)NF * (kFlatThreads * VZ + 2 * a.N) * 8;
  const dim3 grid(p.blocks), blk(kFlatThreads);
#define CLMI_SF(...) hipLaunchKernelGGL((k_scalar_flat<NF, F32, VZ, NH, __VA_ARGS__>), grid, blk, lds, s, a, p.XC, p.G, p.chunks)
  if (kick2) {
    if (!drift || !kick) return hipErrorInvalidValue;
    if (red) CLMI_SF(true, true, true, PK, true);
    else CLMI_SF(true, true, false, PK, true);
    return hipGetLastError();
  }
  switch ((drift ? 4 : 0) | (kick ? 2 : 0) | (red ? 1 : 0)) {
    case 7: CLMI_SF(true, true, true, PK); break;
    case 6: CLMI_SF(true, true, false, PK); break;
    case 5: CLMI_SF(true, false, true, PK); break;
    case 4: CLMI_SF(true, false, false, PK); break;
    case 3: CLMI_SF(false, true, true, PK); break;
    case 2: CLMI_SF(false, true, false, PK); break;
    case 1: CLMI_SF(false, false, true, PK); break;
    default: return hipErrorInvalidValue;
  }
#undef CLMI_SF
  return hipGetLastError();
}

template <int NF, bool F32, int PK>
hipError_t dispatch_flat_shape(bool drift, bool kick, bool red, const ScalarPassArgs &a, const FlatPlan &p,
                               hipStream_t s, bool kick2)
{
  if (a.N * NF > 2 * kFlatThreads) return hipErrorInvalidValue;
  if (p.VZ == 1) {
    if (a.N * NF > kFlatThreads) return hipErrorInvalidValue;
    return dispatch_flat<NF, F32, 1, 1, PK>(drift, kick, red, a, p, s, kick2);
  }
  if (a.N * NF <= kFlatThreads) return dispatch_flat<NF, F32, 2, 1, PK>(drift, kick, red, a, p, s, kick2);
  if constexpr (NF == 2) return dispatch_flat<NF, F32, 2, 2, PK>(drift, kick, red, a, p, s, kick2);
  else return hipErrorInvalidValue;
}

}  // namespace
}  // namespace clmi
