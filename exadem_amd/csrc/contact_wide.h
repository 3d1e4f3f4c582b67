// contact_wide.h — the sphere force pass with several lanes per particle, for particle counts that leave the chip
// idle at one lane per particle.
//
// With one lane per particle a pass lasts as long as the longest chain of one lane: its list entries one after the
// other (6 to 14 contacts of FP64 detection and law, each behind a gather), the walls, the mesh terms, the
// integration. Up to some tens of thousands of particles that chain, not bandwidth, is the time of a step (15 to
// 19 us at 1k to 36k spheres). Here L lanes share a particle: each evaluates one list entry of a round of L, writes
// the six terms it adds to the particle to LDS, and two threads per particle (force, moment) add them in list order, so
// the sums and their order, and with them every bit of the result, are those of the one-lane pass. Lanes without a
// contact write -0.0, which adds nothing to any value. The walls are a round of their own (one lane per wall); the
// mesh terms are added by the two threads, which then integrate the particle: the linear part on the one, the
// rotation on the other, in another wavefront.
//
// P (policy): Args, Entry, T (type of a pair's terms), Acc (their running sum: add, value), fetch, eval.
#pragma once

#include "contact_law.h"
#include "mesh.h"
#include "step.h"

namespace xdem {

struct Own {  // a particle's record as its lanes need it
  V3 r;
  double R;
  V3 v, w;
  double m;
};

// first record of a pass without an LDS tile: no partner lies in it (partner_global)
constexpr int64_t kNoTile = -(1ll << 40);

// Wall w of particle x (ContactLawDriverFunc<Surface / Cylinder / Ball>, contact_sphere.hpp:216-297, with the driver's
// detector): the terms it adds, history updated; nothing is added out of contact.
template <bool KR, class Args>
__device__ inline void wall_terms(const Args& a, int64_t x, int w, const Own& me, double (&c)[6]) {
  const Surface& sf = a.walls[w];
  const int64_t j = (int64_t)w * a.wstride + x;
  double dn;
  V3 nrm, cpos;
  if (!driver_detect(sf, me.r, me.R, dn, nrm, cpos)) {
    a.wl.hx[j] = 0.0; a.wl.hy[j] = 0.0; a.wl.hz[j] = 0.0;
    a.wl.mhx[j] = 0.0; a.wl.mhy[j] = 0.0; a.wl.mhz[j] = 0.0;
    return;
  }
  V3 ft{a.wl.hx[j], a.wl.hy[j], a.wl.hz[j]};
  V3 mint{0.0, 0.0, 0.0};
  if (KR) mint = {a.wl.mhx[j], a.wl.mhy[j], a.wl.mhz[j]};
  const V3 f = hooke_force<KR>(dn, nrm, a.dt, a.cpd, me.m, ft, mint, cpos, me.r, me.v, me.w, sf.center, sf.vel, sf.vrot);
  a.wl.hx[j] = ft.x; a.wl.hy[j] = ft.y; a.wl.hz[j] = ft.z;
  if (KR) {
    a.wl.mhx[j] = mint.x; a.wl.mhy[j] = mint.y; a.wl.mhz[j] = mint.z;
  }
  const V3 m = cross(cpos - me.r, f) + mint;
  c[0] = f.x; c[1] = f.y; c[2] = f.z;
  c[3] = m.x; c[4] = m.y; c[5] = m.z;
}

// Padded row of LDS terms: lane `sub` of particle p writes at sub * row + p, so the eight particles of a wavefront's
// lanes fall on distinct banks, and the adding threads read consecutive particles
constexpr int wide_row(int P) { return P + 8; }

template <class P, int L, bool FUSED, bool INTEG, bool GUARD>
__global__ __launch_bounds__(256) void k_force_wide(typename P::Args a) {
  constexpr int NP = 256 / L, ROW = wide_row(NP);
  // first thread of the moment role: a wavefront of its own
  constexpr int M0 = 64;
  typedef typename P::T T;
  static_assert(sizeof(T) <= sizeof(double), "terms are staged in slots of eight bytes");
  __shared__ double con[2][6][L * ROW];
  // what the integration reads (records, rebuild reference, inertia), staged with the first loads: held in registers
  // through the rounds it costs a wavefront per SIMD, read after them its latency
  __shared__ uint4 rec[FUSED ? NP * 8 : 1];
  __shared__ double aux[FUSED ? 6 : 1][NP];
  // the guard's flags with the first loads; nothing is stored before they are tested
  bool stop = false;
  if (GUARD) stop = (a.flags[1] | a.flags[a.trig_in]) != 0;
  const int tid = threadIdx.x;
  const int64_t b0 = xcd_block(blockIdx.x, gridDim.x) * NP;
  const int p = tid / L, sub = tid % L;
  const PState& s = a.s;
  const int64_t x = b0 + p;
  const int64_t xc = x < a.n ? x : a.n - 1;
  const uint32_t cnt = x < a.n ? a.nl.cnt[xc] : 0u;
  const uint64_t base = a.nl.base[xc >> 6] + (uint64_t)(xc & 63);
  static_assert(NP <= 64, "the block's particles lie in one list group of 64");
  const uint32_t kmax = a.nl.kmax[b0 >> 6];
  uint32_t mask = 0;
  if (a.nw && x < a.n) mask = a.wl.mask[xc];
  Own me;
  {
    const d4 xr = s.core[xc].xr, vm = s.core[xc].vm, w = s.core[xc].w;
    me = {V3{xr.x, xr.y, xr.z}, xr.w, V3{vm.x, vm.y, vm.z}, V3{w.x, w.y, w.z}, vm.w};
  }
  uint32_t wd = (uint32_t)sub < cnt ? a.nl.word[base + (uint64_t)sub * kWave] : 0u;
  constexpr int CH = NP * 8 / 256;  // 16-byte chunks of the block's records per thread
  uint4 ch[CH];
  constexpr int XD = (NP * 6 + 255) / 256;
  double ax[XD];
  if (FUSED) {
#pragma unroll
    for (int q = 0; q < CH; q++) {
      const int64_t at = b0 + ((tid + 256 * q) >> 3);
      ch[q] = ((const uint4*)(s.core + (at < a.n ? at : a.n - 1)))[tid & 7];
    }
#pragma unroll
    for (int q = 0; q < XD; q++) {
      const int i = tid + 256 * q, c = i / NP;
      const int64_t at0 = b0 + (i & (NP - 1)), at = at0 < a.n ? at0 : a.n - 1;
      ax[q] = 0.0;
      // (a load per array: a selected pointer would go through scratch memory)
      if (INTEG && c == 0) ax[q] = s.bx[at];
      if (INTEG && c == 1) ax[q] = s.by[at];
      if (INTEG && c == 2) ax[q] = s.bz[at];
      if (c == 3) ax[q] = s.ix[at];
      if (c == 4) ax[q] = s.iy[at];
      if (c == 5) ax[q] = s.iz[at];
    }
  }
  // the summing and integrating threads: the force and linear part of particle tid (threads 0 .. NP-1), the moment
  // and rotation of particle tid - M0
  const bool lin = tid < NP && b0 + tid < a.n;
  const bool rot = tid >= M0 && tid < M0 + NP && b0 + tid - M0 < a.n;
  const int sp = rot ? tid - M0 : (lin ? tid : 0);
  const int64_t xi = b0 + sp;
  const int c0 = rot ? 3 : 0;
  V3 start{0.0, 0.0, 0.0};
  if (lin && FUSED && a.gravity_on) {
    const double m = s.core[xi].vm.w;
    start = {0.0 + a.grav.x * m, 0.0 + a.grav.y * m, 0.0 + a.grav.z * m};
  } else if (!FUSED && (lin || rot)) {
    start = lin ? V3{s.ax[xi], s.ay[xi], s.az[xi]} : V3{s.mx[xi], s.my[xi], s.mz[xi]};
  }
  if (GUARD && stop) {
    if (blockIdx.x == 0 && tid == 0 && !a.flags[1]) {
      a.flags[1] = 1;
      a.flags[2] = a.step_tag;
    }
    return;
  }
  const uint32_t rounds = (kmax + L - 1) / L;
  uint32_t k = (uint32_t)sub;
  typename P::Acc acc[3];
  acc[0].init(start.x);
  acc[1].init(start.y);
  acc[2].init(start.z);
  if (FUSED) {  // these loads were issued with the list base, on which the word and then the partner wait
#pragma unroll
    for (int q = 0; q < CH; q++) rec[tid + 256 * q] = ch[q];
#pragma unroll
    for (int q = 0; q < XD; q++) {
      const int i = tid + 256 * q;
      if (i < NP * 6) aux[i / NP][i & (NP - 1)] = ax[q];
    }
    if (rounds == 0) __syncthreads();
  }
  int buf = 0;
  for (uint32_t r = 0; r < rounds; r++) {
    T c[6] = {(T)-0.0, (T)-0.0, (T)-0.0, (T)-0.0, (T)-0.0, (T)-0.0};
    if (k < cnt) {
      // (an entry fetched one round ahead costs 34 registers and with them a wavefront per SIMD)
      const uint64_t sl = base + (uint64_t)k * kWave;
      typename P::Entry e;
      P::fetch(a, sl, wd, e);
      if (k + L < cnt) wd = a.nl.word[sl + (uint64_t)L * kWave];
      P::eval(a, sl, e, me, c);
    }
    k += L;
#pragma unroll
    for (int q = 0; q < 6; q++) ((T*)con[buf][q])[sub * ROW + p] = c[q];
    __syncthreads();
    if (lin || rot) {
#pragma unroll
      for (int u = 0; u < L; u++)
#pragma unroll
        for (int q = 0; q < 3; q++) acc[q].add(((const T*)con[buf][c0 + q])[u * ROW + sp]);
    }
    buf ^= 1;  // the next round's terms are written while the slower threads still add these
  }
  V3 S{acc[0].value(), acc[1].value(), acc[2].value()};
  if (a.nw && __syncthreads_or((int)mask)) {
    for (int w0 = 0; w0 < a.nw; w0 += L) {
      double c[6] = {-0.0, -0.0, -0.0, -0.0, -0.0, -0.0};
      const int w = w0 + sub;
      if (w < a.nw && ((mask >> w) & 1u)) wall_terms<P::kKr>(a, xc, w, me, c);
#pragma unroll
      for (int q = 0; q < 6; q++) con[buf][q][sub * ROW + p] = c[q];
      __syncthreads();
      if (lin || rot) {
#pragma unroll
        for (int u = 0; u < L; u++)
          S = S + V3{con[buf][c0][u * ROW + sp], con[buf][c0 + 1][u * ROW + sp], con[buf][c0 + 2][u * ROW + sp]};
      }
      buf ^= 1;
    }
  }
  if (!lin && !rot) return;
  if (a.mt.ncand && a.mt.wcnt[xi >> 6] != 0u) mesh_add_half(a.mt, a.mt.idx[xi], c0, S);
  d4 ra{}, rb{};
  V3 ex{0.0, 0.0, 0.0};
  if (FUSED) {  // position and velocity halves of the record, or spin and orientation
    const uint4* row = rec + sp * 8 + (lin ? 0 : 4);
    __builtin_memcpy(&ra, row, sizeof(d4));
    __builtin_memcpy(&rb, row + 2, sizeof(d4));
    ex = {aux[c0][sp], aux[c0 + 1][sp], aux[c0 + 2][sp]};
  }
  if (lin) {
    if (!INTEG) {
      const V3 f = FUSED ? S / rb.w : S;
      s.ax[xi] = f.x;
      s.ay[xi] = f.y;
      s.az[xi] = f.z;
    } else {
      // the linear half of kick_prolog (the rotation's results are not used here)
      d4 w{}, qq{1.0, 0.0, 0.0, 0.0};
      kick_prolog<true>(ra, rb, w, qq, S.x / rb.w, S.y / rb.w, S.z / rb.w, 0.0, 0.0, 0.0, a.dt, a.kdt_2);
      a.core_out[xi].xr = ra;
      a.core_out[xi].vm = rb;
      const double dx = ra.x - ex.x, dy = ra.y - ex.y, dz = ra.z - ex.z;
      if (dx * dx + dy * dy + dz * dz >= a.thr2) a.flags[a.trig_out] = 1;
    }
  } else {
    if (!INTEG) {
      s.mx[xi] = S.x;
      s.my[xi] = S.y;
      s.mz[xi] = S.z;
    }
    if (FUSED) {
      const V3 al = angular_accel(Q4{rb.x, rb.y, rb.z, rb.w}, S, V3{ra.x, ra.y, ra.z}, ex);
      if (!INTEG) {
        s.alx[xi] = al.x;
        s.aly[xi] = al.y;
        s.alz[xi] = al.z;
      } else {
        d4 xr{}, vm{};
        kick_prolog<true>(xr, vm, ra, rb, 0.0, 0.0, 0.0, al.x, al.y, al.z, a.dt, a.kdt_2);
        a.core_out[xi].w = ra;
        a.core_out[xi].q = rb;
      }
    }
  }
}

// Lanes per particle of a pass over n spheres whose list has `slots` slots (a group of 64 particles has the rows of its
// longest list, so slots / n is the rows of an average wavefront) and whose longest row is `longest`; 1: the one-lane
// kernels. Per step of the engine, without rebuilds (us; one lane / four / eight):
//                     walled lattice (5.9 rows)    periodic packing (7.1 rows)    wide size distribution (8.1 rows)
//   FP64    5,000:    14.8 / 10.7 /  8.3           16.3 /  9.6 /  7.9
//          20,000:    14.7 / 13.0 / 11.3           17.2 / 12.6 / 12.1             22.8 / 14.4 / 12.3
//          36,000:    15.4 / 15.2 / 15.3           18.4 / 15.8 / 14.4             22.1 / 17.0 / 14.9
//          45,000:    15.9 / 16.0 / 17.5           19.0 / 16.6 / 17.7             23.2 / 18.1 / 18.6
//          49,000:    16.0 / 16.4 / 18.0           19.0 / 16.6 / 19.2             22.9 / 18.1 / 20.4
//          52,000:    16.4 / 18.5 / 18.7           18.9 / 18.9 / 19.3             24.3 / 21.6 / 20.1
//          64,000:    17.2 / 18.7 / 21.2           19.6 / 19.5 / 21.6             24.4 / 21.8 / 22.8
//          80,000:    22.1 / 24.5 / 24.8           24.9 / 25.0 / 25.6
//   FP32   20,000:    15.2 / 12.7 / 11.1           17.6 / 12.0 / 11.3             24.1 / 13.7 / 12.3
//          49,000:    16.3 / 15.6 / 17.7           19.2 / 15.1 / 18.4             23.5 / 16.8 / 20.0
//          52,000:    16.8 / 17.4 / 18.2           19.1 / 16.9 / 18.6             25.0 / 19.5 / 19.9
//          64,000:    17.5 / 17.4 / 20.8           19.5 / 17.6 / 21.3             24.5 / 19.8 / 22.3
//          80,000:    20.9 / 23.0 / 24.5           23.4 / 22.7 / 24.8
// The four-lane times step up where the blocks of 64 particles pass three and four per CU. One crowded sphere in the
// walled lattice (a row of 12) delays one wavefront of the one-lane pass: 49,000: 16.8 / 16.4, 60,000: 17.4 / 18.9 in
// FP64 and 17.7 / 17.8 in FP32; so the longest row alone decides only up to three blocks per CU in FP64 and four in FP32.
// With a rolling stiffness (more registers) four blocks are never worth it in FP64 nor, with short lists, in FP32: 64,000
// spheres, walled lattice 22.4 / 29.4 and 23.1 / 26.2, periodic 25.4 / 26.5 and 24.7 / 23.6.
constexpr int64_t kWide8Max = 36000, kWideShort = 45000;
constexpr int64_t kWide3 = 3 * 256 * 64, kWide4 = 4 * 256 * 64;  // spheres at three, four blocks of 64 per CU
inline int wide_lanes(int64_t n, int64_t slots, int longest, bool fp32, bool kr) {
  if (n <= kWide8Max) return 8;
  const bool mid = 2 * slots >= 13 * n, big = 2 * slots >= 15 * n;  // 6.5 and 7.5 rows
  int64_t most;
  if (fp32) most = mid || (longest > 8 && !kr) ? kWide4 : kWide3;
  else most = big && !kr ? kWide4 : mid || longest > 8 ? kWide3 : kWideShort;
  return n <= most ? 4 : 1;
}

template <class P>
void launch_wide(xdem_ctx* c, const typename P::Args& a, int lanes, bool fused, bool integ, bool guarded) {
  const dim3 grid(grid_blocks(a.n, 256 / lanes)), block(256);
#define WIDE(L, F, I, G) hipLaunchKernelGGL((k_force_wide<P, L, F, I, G>), grid, block, 0, c->stream, a)
#define WIDE_L(L)                                        \
  do {                                                   \
    if (integ) WIDE(L, true, true, true);                \
    else if (fused && guarded) WIDE(L, true, false, true); \
    else if (fused) WIDE(L, true, false, false);         \
    else WIDE(L, false, false, false);                   \
  } while (0)
  if (lanes == 8) WIDE_L(8);
  else WIDE_L(4);
#undef WIDE_L
#undef WIDE
}

}  // namespace xdem
