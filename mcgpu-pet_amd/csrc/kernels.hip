// kernels.hip — gfx950 photon-transport kernels.
//
// One lane runs one decay stream at a time: the reference's per-thread Poisson
// process (MCGPU-PET_kernel.cu:229-292) with its own RANECU stream. The kernels
// differ only in how lanes get streams:
//   plain      : lane i of the grid owns stream i (one pass, no queue);
//   persistent : a fixed grid of waves pulls stream indices from a device counter and
//                refills a lane as soon as its stream ends (streams are ordered by
//                decreasing voxel activity, so the long streams start first).
// Per lane the sequence of random numbers and the floating-point operations are those
// of the reference thread with the same id; integer tallies are order-independent, so
// both kernels produce the same tallies bit for bit.
//
// Memory layout (MI355X-first):
//   - voxels: a u8 (or u16) index per voxel into a palette of (density, material)
//     words when the phantom has few distinct pairs (the volume then stays in each XCD's
//     L2), else one 8-byte word per voxel; activity is only read once per stream from a
//     compacted, activity-sorted list of emitting voxels;
//   - cross sections: total (a,b) pairs in an 8-byte table read in the Woodcock loop,
//     Compton/Rayleigh (a,b) in a separate 16-byte table read only at real events;
//   - the Compton shells of the phantom's materials, the energy spectrum and the per-material dose
//     are kept in LDS and flushed once per workgroup;
//   - per-lane state touched by only some phases of the persistent kernel (the pair kept
//     between the two photons, the Compton sampler between rejection trials) lives in
//     LDS slots, so that registers hold only the stream and the current photon.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <climits>

#include "devutil.h"
#include "fastmath.h"
#include "fmath.h"
#include "kparams.h"

#define K_PI 3.14159265358979323846
#define K_EPS 0.00015f
#define K_INV_C (1.0 / 29979245800e-12)
#define K_E511 510998.95f
#define K_MAXMAT 15
// LDS address space: the wave's stream-queue range is passed to a non-inlined function, which
// would otherwise see a generic pointer and use flat accesses.
#define K_LDS __attribute__((address_space(3)))
// Upper bound on the iterations of each rejection loop (GRAa, GCOa). Valid tables accept
// within a few trials; the bound only guarantees that no lane can loop forever on
// corrupt input. The oracle applies the same bound.
#define K_MAX_TRIALS (1 << 20)

// Woodcock steps a lane may take in one STEP phase while its steps stay virtual, and GCOa
// rejection trials (tau loop, p_z loop) in one CTAU / CPZ phase: the phase selection's ballots
// are paid once for several. 3 and 2 measured best on the head workload (1-4 steps, 1-3
// trials); more inflate the register pressure of every phase.
#ifndef MCPET_STEPS_PER_PHASE
#define MCPET_STEPS_PER_PHASE 3
#endif
#ifndef MCPET_TRIALS_PER_PHASE
#define MCPET_TRIALS_PER_PHASE 2
#endif
// Blocks chained after the selected phase's (bit flags): 1 GCOa's tau trials after an
// interaction, 2 its p_z trials after the tau trials, 4 Woodcock steps after the p_z trials,
// 8 Woodcock steps after an emission, 16 the next decay after a pair tally. All five measured
// best on the head workload (6.8 % fewer cycles than none; results are the same bit for bit,
// since a lane's own sequence of operations does not depend on when its blocks run).
#ifndef MCPET_CHAIN
#define MCPET_CHAIN 31
#endif
// Occupancy target of the persistent transport kernels: five waves per SIMD (96 registers, none spilled, up to
// 32 KB of LDS a workgroup). Waves hide the dependent gathers until the vector ALUs' issue bounds the
// kernel; six have 80 registers, which spill. With four / five / six, streams made ready by the wave and
// pairs tallied from the queue: head, 1e8 decays, 29.7 / 26.9 / 28.2 ms; 4e7 torso decays with singles 35.7 /
// 32.7 / 36.8; eight phantoms 7.05 / 6.58 / 7.08; 5e6 decays 1.49 / 1.46 / 1.51; 4e6 ragged 1.06 / 1.07 / 1.13.
#ifndef MCPET_WAVES_PER_EU
#define MCPET_WAVES_PER_EU 5
#endif
#define K_OCCUPANCY __attribute__((amdgpu_waves_per_eu(MCPET_WAVES_PER_EU, 8)))
// Per-phase execution statistics of the persistent kernel (diagnostic builds only).
#ifndef MCPET_SM_STATS
#define MCPET_SM_STATS 0
#endif
// Rarely executed physics (Compton, Rayleigh, tallies) as real calls instead of inlined code.
#ifndef MCPET_NOINLINE_RARE
#define MCPET_NOINLINE_RARE 0
#endif
#if MCPET_NOINLINE_RARE
#define K_RARE __device__ __noinline__
#else
#define K_RARE __device__
#endif

namespace {

struct Rng {
  int x, y;
};

// Skip-ahead in digits of 11 bits: y[j][d] = (a1, a2)^(L d 2^(11 j)) mod (m1, m2), L = 555555 x
// 256, for the three digits of a stream number below 2^33 (built by the compiler, 48 KB, read
// through L2). A stream's start is then the product of three entries and the seed; with one
// factor per set bit, a DECAY phase in which three or four of thirty lanes took a new stream
// spent more than a third of its instructions there (head, 1e8 decays: 41.6 -> 39.7 ms;
// eight phantoms of 3e7 decays in all in one launch: 14.0 -> 12.0 ms).
struct JumpDigits {
  static constexpr int kBits = 11, kDigits = 3;
  alignas(8) unsigned y[kDigits << kBits][2];
};
constexpr JumpDigits jump_digits()
{
  JumpDigits t{};
  const unsigned long long a[2] = {MCR_A1, MCR_A2}, m[2] = {MCR_M1, MCR_M2};
  for (int g = 0; g < 2; g++) {
    unsigned long long base = 1, sq = a[g];
    for (unsigned long long e = (unsigned long long)MCR_HIST_PER_THREAD * MCR_LEAP_DISTANCE; e; e >>= 1) {
      if (e & 1) base = base * sq % m[g];
      sq = sq * sq % m[g];
    }
    for (int j = 0; j < JumpDigits::kDigits; j++) {   // base = a^(L 2^(11 j))
      unsigned long long v = 1;
      for (int d = 0; d < (1 << JumpDigits::kBits); d++) {
        t.y[(j << JumpDigits::kBits) + d][g] = (unsigned)v;
        v = v * base % m[g];
      }
      base = v;
    }
  }
  return t;
}
__device__ const JumpDigits k_jump = jump_digits();

// mcr_init_stream (ranecu.h) with the digit table; j1, j2: the bit tables for the bits above it.
__device__ __forceinline__ void init_stream_seeds(long long id, int seed, const uint32_t* j1, const uint32_t* j2, int* sx, int* sy)
{
  constexpr uint32_t c1 = 0x80000000u - (uint32_t)MCR_M1, c2 = 0x80000000u - (uint32_t)MCR_M2;
  constexpr int B = JumpDigits::kBits;
  const unsigned long long n = (unsigned long long)(id + 1);
  uint32_t y1 = 0, y2 = 0;
#pragma unroll
  for (int j = 0; j < JumpDigits::kDigits; j++) {
    const unsigned d = (j << B) + ((unsigned)(n >> (B * j)) & ((1u << B) - 1u));
    const unsigned long long e = gld(reinterpret_cast<const unsigned long long*>(k_jump.y), d);
    y1 = j ? mcr_mulmod_pm(y1, (uint32_t)e, c1) : (uint32_t)e;
    y2 = j ? mcr_mulmod_pm(y2, (uint32_t)(e >> 32), c2) : (uint32_t)(e >> 32);
  }
  int k = B * JumpDigits::kDigits;
  for (unsigned long long h = n >> k; h && k < MCR_JUMP_BITS; k++, h >>= 1)
    if (h & 1ull) {
      y1 = mcr_mulmod_pm(y1, j1[k], c1);
      y2 = mcr_mulmod_pm(y2, j2[k], c2);
    }
  if (seed > 0 && seed < MCR_M2) {
    *sx = (int)mcr_mulmod_pm((uint32_t)seed, y1, c1);
    *sy = (int)mcr_mulmod_pm((uint32_t)seed, y2, c2);
  } else {
    *sx = mcr_abmodm(MCR_M1, seed, (int)y1);
    *sy = mcr_abmodm(MCR_M2, seed, (int)y2);
  }
}

// Event counters, a compile-time policy of every device function below.
// FullCounters (instrumented instantiation): every event count, per lane in registers,
// flushed once per lane. LiteCounters (production): only decays, streams, tallied pairs
// and coincidences, as workgroup counters in LDS, so that the transport keeps no counter
// registers. Both instantiations perform the same arithmetic on the same random numbers.
struct FullCounters {
  unsigned c[KC_N];
  __device__ __forceinline__ void init(unsigned*)
  {
#pragma unroll
    for (int i = 0; i < KC_N; i++) c[i] = 0;
  }
  __device__ __forceinline__ void inc(int k) { c[k]++; }
  __device__ __forceinline__ void add(int k, unsigned v) { c[k] += v; }
  __device__ __forceinline__ void flush(const KParams& P, const unsigned*)
  {
#pragma unroll
    for (int i = 0; i < KC_N; i++)
      if (c[i]) gatomic_add(&P.counters[i], (unsigned long long)c[i]);
  }
};
struct LiteCounters {
  unsigned* s;  // KC_N workgroup counters in LDS
  __device__ __forceinline__ void init(unsigned* lds) { s = lds; }
  __device__ __forceinline__ void inc(int k)
  {
    if (k == KC_DECAYS || k == KC_STREAMS || k == KC_PAIRS || k == KC_COINC) atomicAdd(&s[k], 1u);
  }
  __device__ __forceinline__ void add(int, unsigned) {}
  __device__ __forceinline__ void flush(const KParams&, const unsigned*) {}
};

template <class CN>
__device__ __forceinline__ float rn(Rng& r, CN& C)
{
  C.inc(KC_RNDRAWS);
  return mcr_ranecu(&r.x, &r.y);
}
template <class CN>
__device__ __forceinline__ double rnd(Rng& r, CN& C)
{
  C.inc(KC_RNDRAWS);
  return mcr_ranecu_double(&r.x, &r.y);
}

// Voxel index x + nx (y + ny z).
__device__ __forceinline__ int voxel_index(const StepParams& P, int x, int y, int z)
{
  if (P.index24) return (int)(__umul24(__umul24(z, P.ny) + y, P.nx) + x);
  return x + P.nx * (y + P.ny * z);
}

// locate_voxel (K:1097-1124). NaN positions count as outside and indices are clamped
// to the grid (the reference would read out of bounds in both cases). Evaluated without
// branches: positive floats order as their bits, so one unsigned comparison per axis tests both
// bounds, and fails for negative numbers and NaN; inside the box floor(p * inverse size) lies in
// [0, n], so only n is clamped. The same index as the reference's early returns and
// __float2int_rd.
__device__ __forceinline__ int locate(const StepParams& P, const float* p)
{
  const bool inside = (__float_as_uint(p[0]) - P.box_lo <= P.box_span[0]) & (__float_as_uint(p[1]) - P.box_lo <= P.box_span[1]) &
                      (__float_as_uint(p[2]) - P.box_lo <= P.box_span[2]);
  const int vx = min(floor_i32(p[0] * P.ivx), P.nx - 1), vy = min(floor_i32(p[1] * P.ivy), P.ny - 1),
            vz = min(floor_i32(p[2] * P.ivz), P.nz - 1);
  return inside ? voxel_index(P, vx, vy, vz) : -100;
}

// rotate_double (K:1159-1200): PENELOPE DIRECT in double precision on a float vector.
__device__ __forceinline__ void rotate_double(float* d, double costh, double phi)
{
  double DXY, NORM, cosphi, sinphi, SDT;
  DXY = (double)(d[0] * d[0] + d[1] * d[1]);
  sincos_n(phi, &sinphi, &cosphi);   // 0 <= phi < 2 pi
  NORM = DXY + (double)(d[2] * d[2]);
  if (fabs(NORM - 1.0) > 1.0e-14) {
    NORM = div_n(1.0, sqrt_n(NORM));   // a unit vector up to rounding
    d[0] = (float)(NORM * d[0]);
    d[1] = (float)(NORM * d[1]);
    d[2] = (float)(NORM * d[2]);
    DXY = (double)(d[0] * d[0] + d[1] * d[1]);
  }
  if (DXY > 1.0e-28) {
    // zero or above 2^-53 (negative, and the direction undefined, only where a table gives |costh| > 1);
    // DXY lies in (1e-28, 1]
    const double sin2 = 1.0 - costh * costh;
    SDT = sin2 != 0.0 ? sqrt_n(div_n(sin2, DXY)) : 0.0;
    float xin = d[0];
    float yz = d[1] * d[2];
    float xz = xin * d[2];
    d[0] = (float)(d[0] * costh + SDT * ((double)xz * cosphi - d[1] * sinphi));
    d[1] = (float)(d[1] * costh + SDT * ((double)yz * cosphi + xin * sinphi));
    d[2] = (float)(d[2] * costh - DXY * SDT * cosphi);
  } else {
    SDT = sqrt(1.0 - costh * costh);
    d[1] = (float)(SDT * sinphi);
    if (d[2] > 0.0) {
      d[0] = (float)(SDT * cosphi);
      d[2] = (float)costh;
    } else {
      d[0] = (float)(-SDT * cosphi);
      d[2] = (float)(-costh);
    }
  }
}

// The Rayleigh (GRAa) and Compton (GCOa) samplers below follow the PENELOPE 2006 algorithms
// as the reference states them (MCGPU-PET_kernel.cu:1216-1228, 1318-1330), which carry this
// notice:
//   PENELOPE/PENGEOM (version 2006)
//     Copyright (c) 2001-2006
//     Universitat de Barcelona
//   Permission to use, copy, modify, distribute and sell this software and its documentation
//   for any purpose is hereby granted without fee, provided that the above copyright notice
//   appears in all copies and that both that copyright notice and this permission notice
//   appear in all supporting documentation. The Universitat de Barcelona makes no
//   representations about the suitability of this software for any purpose. It is provided
//   "as is" without express or implied warranty.

// GRAa (K:1230-1296): Rayleigh angle by RITA inverse cumulative + Thomson rejection.
template <class CN>
K_RARE void graa(float energy, double* costh, int mat, float pmax_current, Rng& r, CN& C,
                     const mcpet_rayleigh_table* __restrict__ cgra_in)
{
  const DU_GLOBAL mcpet_rayleigh_table* cgra = (const DU_GLOBAL mcpet_rayleigh_table*)cgra_in;
  double xmax = ((double)energy) * 8.065535669099010e-5;
  double x2lim = (double)cgra->xco[(mat + 1) * MCPET_NP_RAYLEIGH - 1];
  double x2max = (xmax * xmax) < x2lim ? (xmax * xmax) : x2lim;
  if (xmax < 0.01) {
    int trials = 0;
    do {
      *costh = 1.0 - rnd(r, C) * 2.0;
    } while (rnd(r, C) > (((*costh) * (*costh) + 1.0) * 0.5) && ++trials < K_MAX_TRIALS);
    return;
  }
  *costh = 1.0;
  for (int trial = 0; trial < K_MAX_TRIALS; trial++) {
    double ru = rnd(r, C) * (double)pmax_current;
    int itn = (int)(ru * (MCPET_NP_RAYLEIGH - 1));
    itn = min(max(itn, 0), MCPET_NP_RAYLEIGH - 1);
    int i__ = (int)cgra->itlco[itn + mat * MCPET_NP_RAYLEIGH];
    int j = (int)cgra->ituco[itn + mat * MCPET_NP_RAYLEIGH];
    if ((j - i__) > 1) {
      do {
        int k = (i__ + j) >> 1;
        if (ru > cgra->pco[k - 1 + mat * MCPET_NP_RAYLEIGH]) i__ = k;
        else j = k;
      } while ((j - i__) > 1);
    }
    int index = i__ - 1 + mat * MCPET_NP_RAYLEIGH;
    double rr = ru - cgra->pco[index];
    double xx;
    if (rr > 1e-16) {
      double d__ = (double)(cgra->pco[index + 1] - cgra->pco[index]);
      float aco_index = cgra->aco[index], bco_index = cgra->bco[index], xco_index = cgra->xco[index];
      xx = (double)xco_index + (double)(aco_index + 1.0f + bco_index) * d__ * rr /
                                   (d__ * d__ + (aco_index * d__ + bco_index * rr) * rr) *
                                   (double)(cgra->xco[index + 1] - xco_index);
    } else {
      xx = cgra->xco[index];
    }
    if (xx < x2max) {
      *costh = 1.0 - 2.0 * xx / x2max;
      if (rnd(r, C) < (((*costh) * (*costh) + 1.0) * 0.5)) break;
    }
  }
}

// Compton shells in LDS: the shells of every distinct material file in turn, each (ionisation
// energy U, occupation f, profile J0, U x 510998.918) in one 16-byte read, and per material slot
// (first shell << 8) | number of shells.
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
struct Shells {
  const K_LDS v4f* table;
  const K_LDS unsigned* of;
  const K_LDS v2f* pal;        // the u8 voxel palette (density, material word), where it is in LDS
};

// Compton profile term of shell i at momentum transfer factor `cdtf` (the inner body of
// the incoherent-scattering-function loops, K:1407-1449); 0 for inaccessible shells.
__device__ __forceinline__ float shell_term(v4f sh, float energy, float cdtf, bool use_cdt)
{
  float temp = sh.x;
  if (!(temp < energy)) return 0.0f;
  float pzomc;
  if (!use_cdt) {
    float aux = energy * (energy - temp) * 2.f;
    pzomc = div_n(sh.z * (aux - sh.w), sqrt_nz(aux + aux + temp * temp) * 510998.918f);
    const float m = (pzomc > 0.0f) ? 0.707106781186545f + pzomc * 1.4142135623731f : 0.707106781186545f - pzomc * 1.4142135623731f;
    temp = 0.5f * exp_n(0.5f - m * m);
    if (pzomc > 0.0f) temp = 1.0f - temp;
    return temp;
  }
  float aux = (energy) * (energy - temp) * cdtf;
  pzomc = div_n(sh.z * (aux - sh.w), sqrt_nz(aux + aux + temp * temp) * 510998.918f);
  if (!((aux > 1.0e-12f) || (temp > 1.0e-12f))) pzomc = 0.002f;
  temp = pzomc * 1.4142135623731f;
  const float m = (pzomc > 0.0f) ? temp + 0.70710678118654502f : 0.70710678118654502f - temp;
  temp = 0.5f * exp_n(0.5f - m * m);
  if (pzomc > 0.0f) temp = 1.0f - temp;
  return temp;
}

// GCOa (K:1334-1563): Compton scattering, relativistic impulse approximation with
// analytical one-electron profiles, split into resumable pieces so that the persistent
// kernel can run one rejection trial per phase: gcoa_init (S(theta=pi) over the shells),
// gcoa_tau_trial (one trial of the tau/shell-profile loop, K:1389-1459), gcoa_pz_trial
// (one trial of the p_z loop, K:1463-1539) and gcoa_finish (the final energy, K:1543-1557).
// The per-shell values rn[i] of the accepted tau trial are kept for the first four shells
// and recomputed for later shells instead of a 30-entry array (same values).
struct ComptonState {
  float a1, s0, taumin;            // set by gcoa_init
  float tau, s;                    // accepted tau trial
  float rc0, rc1, rc2, rc3;        // its profile terms of shells 0..3
  float pzomc;
  double cdt1;
  int trials;
};

__device__ __forceinline__ void gcoa_init(float E, int mat, const Shells& cg, ComptonState& cs)
{
  const unsigned of = cg.of[mat];
  const K_LDS v4f* table = cg.table + (of >> 8);
  const int my_noscco = of & 0xff;
  const float ek = E * 1.956951306108245e-6f;
  const float ek2 = ek * 2.f + 1.f;
  cs.taumin = div_n(1.f, ek2);
  cs.a1 = log_n(ek2);
  float s0 = 0.0f;
  for (int i = 0; i < my_noscco; i++) {
    const v4f sh = table[i];
    if (sh.x < E) s0 += sh.y * shell_term(sh, E, 0.0f, false);
  }
  cs.s0 = s0;
  cs.trials = 0;
}

// One trial of the tau loop; true when the loop is over (accepted or trial cap).
template <class CN>
__device__ __forceinline__ bool gcoa_tau_trial(float E, int mat, Rng& r, CN& C, const Shells& cg,
                                               ComptonState& cs)
{
  const unsigned of = cg.of[mat];
  const K_LDS v4f* table = cg.table + (of >> 8);
  const int my_noscco = of & 0xff;
  const float ek = E * 1.956951306108245e-6f;
  const float ek2 = ek * 2.f + 1.f;
  const float ek3 = ek * ek;
  const float taumin = cs.taumin, a1 = cs.a1;
  float tau;
  if (rn(r, C) * (a1 + 2. * ek * (ek + 1.f) * taumin * taumin) < a1)
    tau = exp_n(rn(r, C) * log_n(taumin));   // taumin^u: 0 < taumin < 1, u > 0
  else
    tau = sqrt_nz(1.f + rn(r, C) * (taumin * taumin - 1.f));
  double cdt1 = div_n((double)(1.f - tau), ((double)tau) * ((double)E) * 1.956951306108245e-6);
  if (cdt1 > 2.0) cdt1 = 1.99999999;
  const float cdtf = (float)cdt1;
  float s = 0.0f;
  C.add(KC_SHELLEVAL, (unsigned)my_noscco);
  float rc0 = 0.0f, rc1 = 0.0f, rc2 = 0.0f, rc3 = 0.0f;
  for (int i = 0; i < my_noscco; i++) {
    const v4f sh = table[i];
    if (sh.x < E) {
      const float t = shell_term(sh, E, cdtf, true);
      s += sh.y * t;
      rc0 = (i == 0) ? t : rc0;
      rc1 = (i == 1) ? t : rc1;
      rc2 = (i == 2) ? t : rc2;
      rc3 = (i == 3) ? t : rc3;
    }
  }
  cs.tau = tau;
  cs.cdt1 = cdt1;
  cs.s = s;
  cs.rc0 = rc0;
  cs.rc1 = rc1;
  cs.rc2 = rc2;
  cs.rc3 = rc3;
  const bool reject =
      (rn(r, C) * cs.s0) > div_n(s * (1.0f + tau * ((ek3 - ek2 - 1.0f) + tau * (ek2 + tau * ek3))), ek3 * tau * (tau * tau + 1.0f));
  if (!reject) return true;
  return ++cs.trials >= K_MAX_TRIALS;
}

__device__ __forceinline__ float gcoa_rnv(float E, const K_LDS v4f* table, const ComptonState& cs, int i)
{
  if (i < 4) return i == 0 ? cs.rc0 : i == 1 ? cs.rc1 : i == 2 ? cs.rc2 : cs.rc3;
  return shell_term(table[i], E, (float)cs.cdt1, true);
}

// One trial of the p_z loop; true when the loop is over (accepted or trial cap).
template <class CN>
__device__ __forceinline__ bool gcoa_pz_trial(float E, int mat, Rng& r, CN& C, const Shells& cg,
                                              ComptonState& cs)
{
  const unsigned of = cg.of[mat];
  const K_LDS v4f* table = cg.table + (of >> 8);
  const int my_noscco = of & 0xff;
  const double costh = 1.0 - cs.cdt1;
  const float tau = cs.tau;
  float temp = cs.s * rn(r, C);
  float pac = 0.0f;
  int ishell = my_noscco - 1;
  for (int i = 0; i < (my_noscco - 1); i++) {
    pac += table[i].y * gcoa_rnv(E, table, cs, i);
    if (pac > temp) {
      ishell = i;
      break;
    }
  }
  temp = rn(r, C) * gcoa_rnv(E, table, cs, ishell);
  const float fj = table[ishell].z;
  // both halves of the profile through one logarithm and root; its argument is below 1
  const bool low = temp < 0.5f;
  const float y = low ? temp + temp : 2.0f - 2.0f * temp, den = fj * 1.4142135623731f;
  const float dev = sqrt_nz(0.5f - log_n(y)) - 0.70710678118654502f;
  float pzomc = div_n(low ? -dev : dev, den);
  // y below 2^-126: the profile term underflows; no number: a profile of zero or hardly any width
  if (!(y >= 0x1p-126f) || pzomc != pzomc) {
    const float gdev = sqrtf(0.5f - mcf_logf(y)) - 0.70710678118654502f;
    pzomc = (low ? -gdev : gdev) / den;
  }
  cs.pzomc = pzomc;
  if (!(pzomc < -1.0f)) {
    float af;
    temp = (float)(tau * (tau - costh * 2.f) + 1.f);
    if (temp > 1.0e-20f)
      af = sqrt_nz(temp) * (div_n(tau * (tau - ((float)costh)), temp) + 1.f);
    else
      af = 0.00200f;
    if (af > 0.0f) temp = af * 0.2f + 1.f;
    else temp = 1.f - af * 0.2f;
    float pzc = pzomc < 0.2f ? pzomc : 0.2f;
    pzc = pzc > -0.2f ? pzc : -0.2f;
    if (rn(r, C) * temp < (af * pzc + 1.f)) return true;
  }
  return ++cs.trials >= K_MAX_TRIALS;
}

// Final energy (K:1543-1557); returns cos(theta) of the accepted trial.
__device__ __forceinline__ double gcoa_finish(float* energy, const ComptonState& cs)
{
  const double costh = 1.0 - cs.cdt1;
  const float tau = cs.tau, pzomc = cs.pzomc;
  float t, b1, b2, temp;
  t = pzomc * pzomc;
  b1 = 1.f - t * tau * tau;
  b2 = 1.f - t * tau * ((float)costh);
  temp = sqrtf(fabsf(b2 * b2 - b1 * (1.0f - t)));
  if (pzomc < 0.0f) temp *= -1.0f;
  t = (tau / b1) * (b2 + temp);
  if (t > 1.0f) t = 1.0f;
  (*energy) *= t;
  return costh;
}

struct Stream {
  Rng r;
  unsigned long long remaining;  // acquisition time left (ps)
  double inv_act;                // tpb / activity, decayed per emission
  int absvox;
  unsigned long long event;      // (reference thread id << 32) | number of the current decay
};

// Staging of appended records. A returning atomic on a list's one counter costs about 5 ns for
// the whole device however few lanes ask (other XCDs' caches are in between), so a wave keeps its
// records in a buffer of its own and moves them to the list 64 at a time, with one atomic and
// coalesced copies (4e6 decays with a phase-space file 1.71 -> 1.20 ms, 4e7 torso decays with a
// singles list 47.6 -> 38.4 ms). The number of staged records is in LDS (wq[2], as the stream
// range below).
__device__ __forceinline__ char* stage_of(const KParams& P)
{
  if (!P.stage) return nullptr;
  const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
  return P.stage + (size_t)wave * P.stage_stride;
}
// The first of n staging places for every calling lane.
__device__ __forceinline__ int stage_append(volatile K_LDS long long* wq, int n)
{
  const unsigned long long here = __ballot(1);
  const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(here >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)here, 0u));
  const int c = __builtin_amdgcn_readfirstlane((int)wq[2]);
  if (rank == 0) wq[2] = c + n * __popcll(here);
  return c + n * rank;
}
// Move the last m <= 64 of the wave's c staged records to its list (the whole wave).
__device__ __attribute__((noinline)) void stage_flush(const KParams& P, const char* stage, volatile K_LDS long long* wq, int c, int m)
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the records were written by other lanes
  const int lane = (int)(threadIdx.x & 63);
  const bool singles = P.mode == MCPET_TALLY_SINGLES;
  unsigned long long base = 0;
  if (lane == 0) {
    wq[2] = c - m;
    if (singles) {
      base = gatomic_add(P.singles_n, (unsigned long long)m);
    } else {
      base = (unsigned long long)(unsigned)gatomic_add(P.psf_index, m);
      if (base > 2000000000ull) gatomic_min(P.psf_index, 2000000000);
    }
  }
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)base);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
  base = ((unsigned long long)hi << 32) | lo;
  const long long cap = singles ? P.singles_cap : (P.psf ? (long long)P.psf_size : 0ll);
  const int keep = base >= (unsigned long long)cap ? 0 : (int)min((long long)m, cap - (long long)base);
  const int words = (singles ? (int)sizeof(mcpet_single) : (int)sizeof(mcpet_psf_record)) / 4;
  const DU_GLOBAL unsigned* src = (const DU_GLOBAL unsigned*)stage + (c - m) * words;
  DU_GLOBAL unsigned* dst = (DU_GLOBAL unsigned*)(singles ? (void*)P.singles : (void*)P.psf) + base * words;
  for (int i = lane; i < keep * words; i += 64) dst[i] = src[i];
}

// Cylinder intersection of both photons (K:1645-1707 / K:536-577).
__device__ __forceinline__ float cyl_dist(const KParams& P, float x0, float y0, const float* dir)
{
  float A = dir[0] * dir[0] + dir[1] * dir[1];
  float B = 2.0f * (x0 * dir[0] + y0 * dir[1]);
  float Cc = x0 * x0 + y0 * y0 - P.radius * P.radius;
  if (A == 0.0f) return 99999999.9f;
  return (-B + sqrtf(B * B - 4.0f * A * Cc)) / (2.0f * A);
}

__device__ __forceinline__ void spectrum_add(const KParams& P, int* s_spec, int iE)
{
  if (P.lds_spectrum) __hip_atomic_fetch_add((K_LDS int*)s_spec + iE, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else gatomic_add(&P.spectrum[iE], 1);
}

// Pairs whose bin is known wait in LDS for the rest of their tally, HIT_LEN a wave: about one decay in
// ten gets that far, three lanes of a wave at a time, and the energy blur of 64 lanes costs as much.
// An entry holds what is left to compute with, the four random numbers (drawn in their turn) among it;
// the tallies are integer sums, whose order does not matter. The number of entries is wq[3]. Not with
// lists (kExt), whose registers it would cost more than it gives (torso 34.0 -> 34.2 ms). Head, 1e8
// decays, 29.3 -> 28.5 ms; 5e6 decays on the estimate's phantom 1.67 -> 1.61.
#define HIT_LEN 24
#define HIT_FULL 16   // enough to take them all
enum HitWord { HIT_E1 = 0, HIT_E2, HIT_R1, HIT_R2, HIT_R3, HIT_R4, HIT_BIN, HIT_VOX, HIT_WORDS };   // HIT_VOX: voxel, sign: scattered
typedef K_LDS float* HitQueue;   // [HIT_WORDS][HIT_LEN]

template <class CN>
__device__ __forceinline__ void tally_hit(const KParams& P, float energy, float energyFirst, float randno1, float randno2,
                                          float randno3, float randno4, int ibin, int absvox, bool scattered, CN& C, int* s_spec)
{
  // -2 log(u) is zero or above 1e-7; the doubling is exact
  float g1 = sqrt_nz(-2.0f * log_n(randno1 + 1e-8f)) * cos_n((float)(2.0f * K_PI * (double)randno2));
  float g2 = sqrt_nz(-2.0f * log_n(randno3 + 1.0e-8f)) * cos_n((float)(2.0f * K_PI * (double)randno4));
  float Energia1 = energy + ((P.e_resol) / 2.35f) * energy * g1;
  float Energia2 = energyFirst + ((P.e_resol) / 2.35f) * energyFirst * g2;
  int iE1 = floor_i32_nan(div_r(Energia1, 1000.0f, 1.0f / 1000.0f));   // (no bin for an undefined energy)
  int iE2 = floor_i32_nan(div_r(Energia2, 1000.0f, 1.0f / 1000.0f));
  if ((iE1 < P.ne) && (iE1 >= 0)) spectrum_add(P, s_spec, iE1);
  if ((iE2 < P.ne) && (iE2 >= 0)) spectrum_add(P, s_spec, iE2);
  C.inc(KC_PAIRS);
  if ((Energia1) > (P.e_low) && (Energia1) < (P.e_high) && (Energia2) > (P.e_low) && (Energia2) < (P.e_high)) {
    C.inc(KC_COINC);
    gatomic_add(scattered ? &P.scatter[ibin] : &P.trues[ibin], 1);
    gatomic_add(scattered ? &P.img_sc[absvox] : &P.img_t[absvox], 1);
    if (P.rb_trues) {   // the same event on the rebinning grid (sinogram, angle, radial bin of ibin)
      const int per = P.nangles * P.nrad;
      const int izm = ibin / per, rem = ibin - izm * per;
      const int ith = rem / P.nrad, ir = rem - ith * P.nrad;
      const int cb = (P.rb_plane[izm] * P.rb_H + ith / P.rb_gh) * P.rb_W + ir / P.rb_gw;
      gatomic_add(scattered ? &P.rb_scatter[cb] : &P.rb_trues[cb], 1);
    }
  }
}

// every waiting entry; by the whole wave
template <class CN>
__device__ __forceinline__ void hits_take(const KParams& P, HitQueue hq, volatile K_LDS long long* wq, CN& C, int* s_spec)
{
  const int lane = (int)(threadIdx.x & 63);
  const int c = __builtin_amdgcn_readfirstlane((int)wq[3]);
  __builtin_amdgcn_wave_barrier();
  if (lane < c) {
    float e[HIT_WORDS];
#pragma unroll
    for (int k = 0; k < HIT_WORDS; k++) e[k] = ((volatile K_LDS float*)hq)[k * HIT_LEN + lane];
    const int v = __float_as_int(e[HIT_VOX]);
    tally_hit(P, e[HIT_E1], e[HIT_E2], e[HIT_R1], e[HIT_R2], e[HIT_R3], e[HIT_R4], __float_as_int(e[HIT_BIN]), v & 0x7fffffff,
              v < 0, C, s_spec);
  }
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) wq[3] = 0;
}

// tally_Sinogram (K:1623-1836).
template <class CN>
K_RARE void tally_sinogram(const KParams& P, float energy, float energyFirst, const float* pos, const float* posf,
                               const float* dir, const float* dirf, int ss, int ssf, Stream& st, CN& C, int* s_spec,
                               HitQueue hq, volatile K_LDS long long* wq)
{
  float x0 = pos[0] - P.cx, y0 = pos[1] - P.cy;
  float dist = cyl_dist(P, x0, y0, dir);
  float pxn = x0 + dist * dir[0];
  float pyn = y0 + dist * dir[1];
  float pzn = (pos[2] - P.cz) + dist * dir[2];
  if (!(fabsf(pzn) < 0.5f * P.height)) return;
  x0 = posf[0] - P.cx;
  y0 = posf[1] - P.cy;
  dist = cyl_dist(P, x0, y0, dirf);
  float pfxn = x0 + dist * dirf[0];
  float pfyn = y0 + dist * dirf[1];
  float pfzn = (posf[2] - P.cz) + dist * dirf[2];
  if (!(fabsf(pfzn) < 0.5f * P.height)) return;
  // the azimuths only matter once both hits are inside the detector height (K:1669,1700)
  const float phi = mcf_atan2f(pyn, pxn);
  const float phi1 = mcf_atan2f(pfyn, pfxn);
  int ibin = sino_bin(P, phi, pzn, phi1, pfzn);
  if (ibin < 0) return;
  const float randno1 = rn(st.r, C);
  const float randno2 = rn(st.r, C);
  const float randno3 = rn(st.r, C);
  const float randno4 = rn(st.r, C);
  const bool scattered = ss > 0 || ssf > 0;
  if (hq) {
    const unsigned long long here = __ballot(1);
    const int n = __popcll(here), rank = __popcll(here & ((1ull << __lane_id()) - 1ull));
    const int at = __builtin_amdgcn_readfirstlane((int)wq[3]);
    __builtin_amdgcn_wave_barrier();
    if (at + n <= HIT_LEN) {
      const float e[HIT_WORDS] = {energy, energyFirst, randno1, randno2, randno3, randno4, __int_as_float(ibin),
                                  __int_as_float(st.absvox | (scattered ? (int)0x80000000 : 0))};
#pragma unroll
      for (int k = 0; k < HIT_WORDS; k++) ((volatile K_LDS float*)hq)[k * HIT_LEN + at + rank] = e[k];
      if (rank == 0) wq[3] = at + n;
      return;
    }
  }
  tally_hit(P, energy, energyFirst, randno1, randno2, randno3, randno4, ibin, st.absvox, scattered, C, s_spec);
}

__device__ __forceinline__ void write_psf(DU_GLOBAL mcpet_psf_record* rec, unsigned long long t_ps, float travel_ps, int vox, float e,
                                          float z, float phi, const float* v, int idx1)
{
  rec->emission_time_ps = t_ps;
  rec->travel_time_ps = travel_ps;
  rec->emission_absvox = vox;
  rec->energy = e;
  rec->z = z;
  rec->phi = phi;
  rec->vx = v[0];
  rec->vy = v[1];
  rec->vz = v[2];
  rec->index1 = (int16_t)idx1;
  rec->index2 = 0;
}

// tally_PSF_coincidences (K:530-644).
template <class CN>
K_RARE void tally_psf(const KParams& P, float energy, float energyFirst, const float* pos_in, const float* posf_in,
                          const float* dir, const float* dirf, int ss, int ssf, float travel, float travelFirst, Stream& st,
                          CN& C, char* stage, volatile K_LDS long long* wq)
{
  float position[3], positionFirst[3];
  float x0 = pos_in[0] - P.cx, y0 = pos_in[1] - P.cy;
  float dist = cyl_dist(P, x0, y0, dir);
  travel += dist;
  position[0] = x0 + dist * dir[0];
  position[1] = y0 + dist * dir[1];
  position[2] = (pos_in[2] - P.cz) + dist * dir[2];
  if (!(fabsf(position[2]) < 0.5f * P.height)) return;
  x0 = posf_in[0] - P.cx;
  y0 = posf_in[1] - P.cy;
  dist = cyl_dist(P, x0, y0, dirf);
  travelFirst += dist;
  positionFirst[0] = x0 + dist * dirf[0];
  positionFirst[1] = y0 + dist * dirf[1];
  positionFirst[2] = (posf_in[2] - P.cz) + dist * dirf[2];
  float randno1 = rn(st.r, C);
  float randno2 = rn(st.r, C);
  float g1 = sqrt_nz(-2.0f * log_n(randno1 + 1e-8f)) * cos_n((float)(2.0f * K_PI * (double)randno2));
  float randno3 = rn(st.r, C);
  float randno4 = rn(st.r, C);
  float g2 = sqrt_nz(-2.0f * log_n(randno3 + 1.0e-8f)) * cos_n((float)(2.0f * K_PI * (double)randno4));
  float Energia1 = energy + ((P.e_resol) * (1.0f / 2.35f)) * energy * g1;
  float Energia2 = energyFirst + ((P.e_resol) * (1.0f / 2.35f)) * energyFirst * g2;
  if (fabsf(positionFirst[2]) < 0.5f * P.height && (Energia1 > P.e_low) && (Energia1 < P.e_high) && (Energia2 > P.e_low) &&
      (Energia2 < P.e_high)) {
    mcpet_psf_record* list;
    int index, room;
    if (stage) {
      list = (mcpet_psf_record*)stage;
      index = stage_append(wq, 2);
      room = K_STAGE_RECORDS;
    } else {
      list = P.psf;
      index = gatomic_add(P.psf_index, 2);
      if (index > 2000000000) gatomic_min(P.psf_index, 2000000000);
      room = P.psf ? P.psf_size : 0;
    }
    if (index < room) {
      int i0, i1;
      if (travel < travelFirst) {
        i0 = index;
        i1 = index + 1;
      } else {
        i0 = index + 1;
        i1 = index;
      }
      unsigned long long t_ps = P.acq_ps - st.remaining;
      // azimuths of the two records (K:554,577), needed only for a stored pair
      const float phi = mcf_atan2f(position[1], position[0]);
      const float phi1 = mcf_atan2f(positionFirst[1], positionFirst[0]);
      if (i0 < room)
        write_psf((DU_GLOBAL mcpet_psf_record*)(list + i0), t_ps, (float)(travel * K_INV_C), st.absvox, Energia1, position[2], phi, dir, ss);
      if (i1 < room)
        write_psf((DU_GLOBAL mcpet_psf_record*)(list + i1), t_ps, (float)(travelFirst * K_INV_C), st.absvox, Energia2, positionFirst[2], phi1, dirf, ssf);
    }
  }
}

// Singles list (no reference counterpart; the reference tallies pairs only): a photon that
// leaves the phantom and hits the detector cylinder within its height gets the detector's
// energy blur (the PSF path's form, K:580-587, two draws), joins the singles spectrum and,
// inside the energy window, is appended with its detection time = emission time + flight
// time to the cylinder.
template <class CN>
__device__ __forceinline__ void record_single(const KParams& P, const float* pos, const float* dir, float energy, float travel,
                                              int ss, int kind, Stream& st, CN& C, int* s_spec, char* stage,
                                              volatile K_LDS long long* wq)
{
  const float x0 = pos[0] - P.cx, y0 = pos[1] - P.cy;
  const float dist = cyl_dist(P, x0, y0, dir);
  const float z = (pos[2] - P.cz) + dist * dir[2];
  if (!(fabsf(z) < 0.5f * P.height)) return;
  const float randno1 = rn(st.r, C);
  const float randno2 = rn(st.r, C);
  const float g = sqrt_nz(-2.0f * log_n(randno1 + 1e-8f)) * cos_n((float)(2.0f * K_PI * (double)randno2));
  const float e = energy + ((P.e_resol) * (1.0f / 2.35f)) * energy * g;
  const int iE = floor_i32_nan(div_r(e, 1000.0f, 1.0f / 1000.0f));
  if ((iE < P.ne) && (iE >= 0)) spectrum_add(P, s_spec, iE);
  if (!(e > P.e_low && e < P.e_high)) return;
  const float phi = mcf_atan2f(y0 + dist * dir[1], x0 + dist * dir[0]);
  const unsigned long long flight = d2ull_rn((double)(travel + dist) * K_INV_C);
  const unsigned long long t = (P.acq_ps - st.remaining) + (flight < (1ull << 40) ? flight : (1ull << 40) - 1ull);
  const unsigned long long k = stage ? (unsigned long long)stage_append(wq, 1) : gatomic_add(P.singles_n, 1ull);
  if (stage || (long long)k < P.singles_cap) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    DU_GLOBAL u32x4* rec = (DU_GLOBAL u32x4*)((stage ? (mcpet_single*)stage : P.singles) + k);
    rec[0] = u32x4{(unsigned)t, (unsigned)(t >> 32), (unsigned)st.event, (unsigned)(st.event >> 32)};
    rec[1] = u32x4{__float_as_uint(e), __float_as_uint(z), __float_as_uint(phi), ((unsigned)ss & 0xffffu) | ((unsigned)kind << 16)};
  }
}

__device__ __forceinline__ void tally_dose(const KParams& P, float Edep, int mat, const float* pos, unsigned long long* s_mat)
{
  if (P.material_dose) {
    atomicAdd(&s_mat[2 * mat], f2ull_rn(Edep * 1.0f));
    atomicAdd(&s_mat[2 * mat + 1], f2ull_rn(Edep * Edep));
  }
  if (P.voxel_dose) {
    short vx = (short)floor_i32(pos[0] * P.ivx);
    short vy = (short)floor_i32(pos[1] * P.ivy);
    short vz = (short)floor_i32(pos[2] * P.ivz);
    if ((vx < P.roi[0]) || (vx > P.roi[1]) || (vy < P.roi[2]) || (vy > P.roi[3]) || (vz < P.roi[4]) || (vz > P.roi[5])) return;
    int DX = 1 + (int)(P.roi[1] - P.roi[0]);
    int num = (int)(vx - P.roi[0]) + ((int)(vy - P.roi[2])) * DX + ((int)(vz - P.roi[4])) * DX * (1 + (int)(P.roi[3] - P.roi[2]));
    gatomic_add(&P.voxel_edep[2 * (size_t)num], f2ull_rn(Edep * 1.0f));
    gatomic_add(&P.voxel_edep[2 * (size_t)num + 1], f2ull_rn(Edep * Edep));
  }
}

// ---------------------------------------------------------------------------------- photon transport
// Transport is split into three per-lane building blocks so that the same arithmetic
// serves the nested (plain) kernel and the state-machine (persistent) kernel:
// photon_start (energy bin, Woodcock mean free path), woodcock_step (one delta-tracking
// step, K:319-342) and real_interaction (K:348-413).

struct Photon {
  float pos[3], dir[3];
  float E, travel, mfpW, mfp_density, prob, randno;
  float2 tab;            // (a, b) of the total cross section at (index, material of mat_old)
  int index;
  int mat_old;           // voxel material word of the last step (< 0: reload the cross section)
  int mat0, ss;
};

__device__ __forceinline__ void photon_start(const KParams& P, Photon& ph, float energy = K_E511)
{
  ph.E = energy;
  ph.ss = 0;
  ph.travel = 0.0f;
  ph.index = floor_i32((ph.E - P.e0) * P.ide);
  const float2 w = gld32(P.woodcock, ph.index);
  ph.mfpW = w.x + ph.E * w.y;
  ph.mat_old = -1;
}

enum StepOutcome { STEP_ESCAPED = 0, STEP_VIRTUAL = 1, STEP_REAL = 2 };

// The total-cross-section row (a, b) of every material slot at the annihilation energy's bin,
// copied to LDS per workgroup: unscattered photons (most Woodcock steps) reload (a, b) from
// here on a table change instead of from global memory. The same values as P.tot's row.
__shared__ float2 k_tot511[K_MAXMAT];

// Fill k_tot511 (all lanes of the workgroup; a barrier must follow).
__device__ __forceinline__ void load_tot511(const KParams& P)
{
  const int idx = f2i_rd((K_E511 - P.e0) * P.ide);
  if (threadIdx.x < K_MAXMAT) k_tot511[threadIdx.x] = gld(P.tot, idx * K_MAXMAT + threadIdx.x);
}

// The (density, material) word of voxel absvox in the device layout chosen at set-up.
__device__ __forceinline__ float2 voxel_word(const StepParams& P, const K_LDS v2f* pal, int absvox)
{
  if (P.vox_fmt == 1) {
    const unsigned i = gld32(P.vox8, absvox);
    if (!P.lds_palette) return gld32(P.palette, i);
    const v2f v = pal[i];
    return make_float2(v.x, v.y);
  }
  if (P.vox_fmt == 2) return gld32(P.palette, gld32(P.vox16, absvox));
  return gld(P.vox, absvox);
}

template <class CN>
__device__ __forceinline__ int woodcock_step(const StepParams& P, const K_LDS v2f* pal, Photon& ph, Rng& r, CN& C)
{
  const float step = -(ph.mfpW)*log_n(rn(r, C));
  C.inc(KC_WOODCOCK);
  ph.travel += step;
  ph.pos[0] += step * ph.dir[0];
  ph.pos[1] += step * ph.dir[1];
  ph.pos[2] += step * ph.dir[2];
  const int absvox = locate(P, ph.pos);
  if (absvox < 0) return STEP_ESCAPED;
  const float2 md = voxel_word(P, pal, absvox);
  // material word: slot (bits 0-7) | id of its total cross-section table (bits 8-15); slots
  // whose tables are bitwise identical share an id, so a change between them (a material
  // change of the reference, K:331-336) keeps the (a, b) already loaded: the same values
  const int w = __float_as_int(md.y);
  ph.mat0 = w & 0xff;
  if (w != ph.mat_old) {
    if (ph.mat_old < 0 || (w >> 8) != (ph.mat_old >> 8))
      ph.tab = ph.index == P.idx511 ? k_tot511[ph.mat0] : gld32(P.tot, ph.index * K_MAXMAT + ph.mat0);
    ph.mat_old = w;
    C.inc(KC_MATCHANGE);
  }
  ph.mfp_density = ph.mfpW * md.x;
  ph.prob = 1.0f - ph.mfp_density * (ph.tab.x + ph.E * ph.tab.y);
  ph.randno = rn(r, C);
  return (ph.randno < ph.prob) ? STEP_VIRTUAL : STEP_REAL;
}

// Real event at the photon's position (K:348-413), in two halves around GCOa's loops:
// interaction_begin picks the process; Rayleigh and photoelectric events complete there
// (with their dose), a Compton event starts GCOa and is completed by compton_end after
// its rejection loops. interaction_begin returns IA_ALIVE, IA_ABSORBED or IA_COMPTON.
enum InteractionOutcome { IA_ALIVE = 0, IA_ABSORBED = 1, IA_COMPTON = 2 };

template <class CN>
__device__ __forceinline__ int interaction_begin(const KParams& P, Photon& ph, Rng& r, CN& C,
                                                 const Shells& cg, ComptonState& cs, unsigned long long* s_mat)
{
  const float4 cr = gld32(P.cr, ph.index * K_MAXMAT + ph.mat0);
  float prob = ph.prob + ph.mfp_density * (cr.x + ph.E * cr.y);
  const float randno = ph.randno;
  if (randno < prob) {
    C.inc(KC_COMPTON);
    gcoa_init(ph.E, ph.mat0, cg, cs);
    return IA_COMPTON;
  }
  prob += ph.mfp_density * (cr.z + ph.E * cr.w);
  if (randno < prob) {
    double costh_Rayleigh;
    C.inc(KC_RAYLEIGH);
    const float pmax_current = gld(P.ray->pmax, (ph.index + 1) * K_MAXMAT + ph.mat0);
    graa(ph.E, &costh_Rayleigh, ph.mat0, pmax_current, r, C, P.ray);
    rotate_double(ph.dir, costh_Rayleigh, 6.28318530717958647693 * rnd(r, C));
    ph.ss = (ph.ss == 0) ? 2 : 3;
    return IA_ALIVE;
  }
  C.inc(KC_PHOTO);
  const float randno_pe = -ph.E;
  ph.index = -11;
  if (randno_pe < -0.001f) tally_dose(P, -1.0f * randno_pe, ph.mat0, ph.pos, s_mat);
  return IA_ABSORBED;
}

// Completion of a Compton event once both GCOa loops are done: new energy and direction,
// energy bin, Woodcock mean free path, scatter state and dose. False if absorbed (energy
// below the tables).
template <class CN>
__device__ __forceinline__ bool compton_end(const KParams& P, Photon& ph, Rng& r, CN& C, const ComptonState& cs,
                                            unsigned long long* s_mat)
{
  const float e_before = ph.E;
  const double costh_Compton = gcoa_finish(&ph.E, cs);
  rotate_double(ph.dir, costh_Compton, 6.28318530717958647693 * rnd(r, C));
  const float randno = ph.E - e_before;
  ph.index = floor_i32_nan((ph.E - P.e0) * P.ide);   // an undefined energy lies below the tables: absorbed
  if (ph.index > -1) {
    const float2 w = gld32(P.woodcock, ph.index);
    ph.mfpW = w.x + ph.E * w.y;
    ph.mat_old = -2;
    ph.ss = (ph.ss == 0) ? 1 : 3;
  }
  if (randno < -0.001f) tally_dose(P, -1.0f * randno, ph.mat0, ph.pos, s_mat);
  return ph.index >= 0;
}

// Whole real event, nested form. False when the photon is absorbed.
template <class CN>
__device__ __forceinline__ bool real_interaction(const KParams& P, Photon& ph, Rng& r, CN& C, const Shells& cg,
                                                 unsigned long long* s_mat)
{
  ComptonState cs;
  const int o = interaction_begin(P, ph, r, C, cg, cs, s_mat);
  if (o != IA_COMPTON) return o == IA_ALIVE;
  while (!gcoa_tau_trial(ph.E, ph.mat0, r, C, cg, cs)) {
  }
  cs.trials = 0;
  while (!gcoa_pz_trial(ph.E, ph.mat0, r, C, cg, cs)) {
  }
  return compton_end(P, ph, r, C, cs, s_mat);
}

// Whole photon (K:297-415), nested loops: escape or absorption.
template <class CN>
__device__ __forceinline__ void transport_photon(const KParams& P, Photon& ph, Stream& st, CN& C,
                                                 const Shells& cg, unsigned long long* s_mat)
{
  if (locate(P, ph.pos) < 0) return;   // an interaction leaves the photon inside the box
  for (;;) {
    int o;
    do {
      o = woodcock_step(P, cg.pal, ph, st.r, C);
    } while (o == STEP_VIRTUAL);
    if (o == STEP_ESCAPED) return;
    if (!real_interaction(P, ph, st.r, C, cg, s_mat)) return;
  }
}

// Pair emission at a uniform point of the stream's voxel (K:665-773).
// q = n / d for 0 <= n < 2^31 and 1 <= d < 2^20 with inv = 1/d in double: the product's
// error is below 2^-21 < 1/d, so its truncation is q, or q - 1 when n / d is an integer and the
// product rounds below it; one comparison fixes that. Replaces a 32-bit integer division (tens
// of instructions). Grid dimensions are far below 2^20.
__device__ __forceinline__ int div_by_inv(int n, int d, double inv)
{
  int q = (int)((double)n * inv);
  if (n - q * d >= d) q++;
  return q;
}
// (x, y, z) of voxel index v (x fastest), the reference's v % nx, (v / nx) % ny, v / (nx ny).
__device__ __forceinline__ void voxel_coords(const KParams& P, int v, int& ix, int& iy, int& iz)
{
  const int q = div_by_inv(v, P.nx, P.inv_nx);
  iz = div_by_inv(q, P.ny, P.inv_ny);
  iy = q - iz * P.ny;
  ix = v - q * P.nx;
}

template <class CN>
__device__ __forceinline__ void source_first(const KParams& P, Stream& st, CN& C, float* pos, float* dir)
{
  dir[2] = 1.0f - 2.0f * rn(st.r, C);
  float phi_sampled = 6.28318530716f * rn(st.r, C);
  float sin_theta = sqrt_nz(1.0f - dir[2] * dir[2]);
  float sp, cp;
  sincos_n(phi_sampled, &sp, &cp);
  dir[1] = sin_theta * sp;
  dir[0] = sin_theta * cp;
  float r1 = rn(st.r, C);
  float r2 = rn(st.r, C);
  float r3 = rn(st.r, C);
  r1 = (K_EPS > r1 - K_EPS) ? K_EPS : r1 - K_EPS;
  r2 = (K_EPS > r2 - K_EPS) ? K_EPS : r2 - K_EPS;
  r3 = (K_EPS > r3 - K_EPS) ? K_EPS : r3 - K_EPS;
  int ix, iy, iz;
  voxel_coords(P, st.absvox, ix, iy, iz);
  pos[0] = div_r((float)ix + r1, P.ivx, P.rvx);
  pos[1] = div_r((float)iy + r2, P.ivy, P.rvy);
  pos[2] = div_r((float)iz + r3, P.ivz, P.rvz);
}

// Isotropic direction (K:711-720, the BG-mode second photon).
template <class CN>
__device__ __forceinline__ void isotropic_dir(Stream& st, CN& C, float* dir)
{
  dir[2] = 1.0f - 2.0f * rn(st.r, C);
  float phi_sampled = 6.28318530716f * rn(st.r, C);
  float sin_theta = sqrt_nz(1.0f - dir[2] * dir[2]);
  float sp, cp;
  sincos_n(phi_sampled, &sp, &cp);
  dir[1] = sin_theta * sp;
  dir[0] = sin_theta * cp;
}

template <class CN>
__device__ __forceinline__ void source_second(const KParams& P, Stream& st, CN& C, const float* dir1, float* dir)
{
  if (P.bg_mode) {
    isotropic_dir(st, C, dir);
    return;
  }
  float phi_sampled2 = (float)((double)mcf_atan2f(dir1[1], dir1[0]) + K_PI);
  float theta_sampled2 = (float)(K_PI - (double)mcf_acosf(dir1[2]));
  float V1 = rn(st.r, C);
  float V2 = rn(st.r, C);
  float THETA_NC = (float)((2.0 * 0.21276 * K_PI / 180.0) * (double)sqrt_nz(-2.0f * log_n(V2 + 1e-8f)) *
                           (double)cos_n((float)((2.0 * K_PI) * (double)V1)));
  float PHI_NC = (float)((2.0 * K_PI) * (double)rn(st.r, C));
  float ST, CT, CP, SP, ST1, CT1, CP1, SP1;
  sincos_n(THETA_NC, &ST, &CT);
  sincos_n(PHI_NC, &SP, &CP);
  sincos_n(theta_sampled2, &ST1, &CT1);
  sincos_n(phi_sampled2, &SP1, &CP1);
  float GX = CP * ST;
  float GY = SP * ST;
  float GZ = CT;
  dir[0] = GX * CT1 * CP1 - GY * SP1 + GZ * ST1 * CP1;
  dir[1] = GX * CT1 * SP1 + GY * CP1 + GZ * ST1 * SP1;
  dir[2] = -GX * ST1 + GZ * CT1;
}

// Time to the next annihilation of the stream (K:261-292). False when the stream's
// acquisition time is exhausted.
template <class CN>
__device__ __forceinline__ bool decay_time(const KParams& P, Stream& st, CN& C)
{
  const double Dt = -log_n(rnd(st.r, C)) * st.inv_act;
  const unsigned long long Dt_ps = d2ull_rn(Dt * 1e12);
  if (!(Dt_ps < st.remaining)) return false;
  st.remaining -= Dt_ps;
  st.event++;
  C.inc(KC_DECAYS);              // 2 photon histories per decay (K:282)
  st.inv_act = st.inv_act * exp_nonneg(Dt * P.inv_mean_life);
  return true;
}

// Pair state kept between the two photons of an annihilation (K:200-203, 418-441).
struct Pair {
  float p1[3], d1[3];              // emission point and photon-1 direction
  float EF, travelF;               // photon 1 at escape (EF = -10 if absorbed)
  float posF[3], dirF[3];
  int ssF;
};

__device__ __forceinline__ bool pair_selected(const KParams& P, int ss, int ssF)
{
  return P.type == 0 || (P.type == 1 && ss == 0 && ssF == 0) || (P.type == 2 && (ss != 0 || ssF != 0));
}

template <class CN, bool kLists = true>
__device__ __forceinline__ void tally_pair(const KParams& P, const Photon& ph, const Pair& pr, Stream& st, CN& C, int* s_spec, char* stage = nullptr,
                                           volatile K_LDS long long* wq = nullptr, HitQueue hq = nullptr)
{
  if (!kLists || P.mode == 0 || P.mode == 2)
    tally_sinogram(P, ph.E, pr.EF, ph.pos, pr.posF, ph.dir, pr.dirF, ph.ss, pr.ssF, st, C, s_spec, hq, wq);
  if (kLists && (P.mode == 0 || P.mode == 1))
    tally_psf(P, ph.E, pr.EF, ph.pos, pr.posF, ph.dir, pr.dirF, ph.ss, pr.ssF, ph.travel, pr.travelF, st, C, stage, wq);
}

__device__ __forceinline__ void keep_first(Pair& pr, const Photon& ph)
{
  if (ph.index > -1) {
    pr.EF = ph.E;
    pr.travelF = ph.travel;
    pr.ssF = ph.ss;
    for (int k = 0; k < 3; k++) {
      pr.posF[k] = ph.pos[k];
      pr.dirF[k] = ph.dir[k];
    }
  }
}

// One annihilation, both photons, nested loops (reference main loop body, K:259-449).
template <class CN>
__device__ bool decay(const KParams& P, Stream& st, CN& C, const Shells& cg, int* s_spec,
                      unsigned long long* s_mat)
{
  if (!decay_time(P, st, C)) return false;
  C.inc(KC_EMIT_PAIR);
  Pair pr;
  Photon ph;
  source_first(P, st, C, pr.p1, pr.d1);
  pr.EF = -10.0f;
  for (int k = 0; k < 3; k++) {
    ph.pos[k] = pr.p1[k];
    ph.dir[k] = pr.d1[k];
  }
  photon_start(P, ph);
  transport_photon(P, ph, st, C, cg, s_mat);
  keep_first(pr, ph);
  source_second(P, st, C, pr.d1, ph.dir);
  for (int k = 0; k < 3; k++) ph.pos[k] = pr.p1[k];
  photon_start(P, ph);
  transport_photon(P, ph, st, C, cg, s_mat);
  if (ph.index > -1 && pr.EF > -0.5f && pair_selected(P, ph.ss, pr.ssF)) tally_pair(P, ph, pr, st, C, s_spec);
  return true;
}

__device__ __forceinline__ void stream_init(const KParams& P, long long s, Stream& st)
{
  int k;
  long long tid, per_voxel;
  if (P.stream_start) {   // balanced layout: the voxel owning stream s (binary search)
    int lo = 0, hi = P.n_active - 1;
    if (P.stream_hint) {  // narrowed to the owners of the first streams of s's block and the next
      const long long b = s >> P.hint_shift;
      lo = gld(P.stream_hint, b);
      hi = gld(P.stream_hint, b + 1);
    }
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (gld(P.stream_start, mid) <= s) lo = mid;
      else hi = mid - 1;
    }
    k = lo;
    const long long s0 = gld(P.stream_start, k);
    per_voxel = gld(P.stream_start, k + 1) - s0;
    tid = gld(P.stream_id, k) + (s - s0);
  } else {
    k = (int)((double)s * P.inv_tpb);   // s / tpb: exact, or one too small where tpb divides s
    if ((long long)(k + 1) * P.tpb <= s) k++;
    per_voxel = P.tpb;
    tid = (long long)gld(P.active_vox, k) * P.tpb + (s - (long long)k * P.tpb);
  }
  st.absvox = gld(P.active_vox, k);
  const float act = gld(P.active_act, k);
  init_stream_seeds(tid, P.seed, P.j1, P.j2, &st.r.x, &st.r.y);
  st.event = (unsigned long long)tid << 32;
  st.remaining = P.acq_ps;
  st.inv_act = div_n((double)per_voxel, (double)act);
}

__device__ __forceinline__ void stream_finish(const KParams& P, const Stream& st)
{
  if ((long long)(st.event >> 32) == P.last_thread_id) *(DU_GLOBAL int*)P.final_seed = st.r.x;
}

// Workgroup prologue/epilogue shared by the kernels: Compton table, spectrum, material
// dose and workgroup counters in LDS; counters flushed once per lane / per workgroup.
// Dynamic LDS of the single-phantom kernels: the shells, the palette and the spectrum (the last
// two where the layout keeps them in LDS), of the sizes this phantom needs.
#define K_PROLOGUE(CN)                                                                           \
  __shared__ unsigned s_shell_of[K_MAXMAT];                                                      \
  __shared__ unsigned long long s_mat[2 * K_MAXMAT];                                             \
  __shared__ unsigned s_cnt[KC_N];                                                               \
  extern __shared__ v4f s_dyn[];                                                                 \
  const bool use_pal = P.vox_fmt == 1 && P.lds_palette;                                          \
  v2f* const s_pal = (v2f*)(s_dyn + P.n_shells);                                                 \
  int* const s_spec = (int*)(s_pal + (use_pal ? P.n_palette : 0));                               \
  {                                                                                              \
    for (int i = threadIdx.x; i < P.n_shells; i += blockDim.x) {                                 \
      const float4 v = gld(P.shells, i);                                                         \
      s_dyn[i] = v4f{v.x, v.y, v.z, v.w};                                                        \
    }                                                                                            \
    if (threadIdx.x < K_MAXMAT) s_shell_of[threadIdx.x] = P.shell_of[threadIdx.x];               \
    if (threadIdx.x < 2 * K_MAXMAT) s_mat[threadIdx.x] = 0ull;                                   \
    if (threadIdx.x < KC_N) s_cnt[threadIdx.x] = 0u;                                             \
    if (use_pal)                                                                                 \
      for (int i = threadIdx.x; i < P.n_palette; i += blockDim.x) {                              \
        const float2 v = gld(P.palette, i);                                                      \
        s_pal[i] = v2f{v.x, v.y};                                                                \
      }                                                                                          \
    load_tot511(P);                                                                              \
    if (P.lds_spectrum)                                                                          \
      for (int i = threadIdx.x; i < P.ne; i += blockDim.x) s_spec[i] = 0;                        \
  }                                                                                              \
  __syncthreads();                                                                               \
  const Shells s_cmp{(const K_LDS v4f*)s_dyn, (const K_LDS unsigned*)s_shell_of, (const K_LDS v2f*)s_pal}; \
  CN C;                                                                                          \
  C.init(s_cnt);

#define K_EPILOGUE                                                                               \
  C.flush(P, s_cnt);                                                                             \
  __syncthreads();                                                                               \
  if (threadIdx.x < KC_N && s_cnt[threadIdx.x])                                                  \
    gatomic_add(&P.counters[threadIdx.x], (unsigned long long)s_cnt[threadIdx.x]);               \
  if (P.lds_spectrum)                                                                            \
    for (int i = threadIdx.x; i < P.ne; i += blockDim.x)                                         \
      if (s_spec[i]) gatomic_add(&P.spectrum[i], s_spec[i]);                                     \
  if (threadIdx.x < 2 * K_MAXMAT && s_mat[threadIdx.x]) gatomic_add(&P.mat_edep[threadIdx.x], s_mat[threadIdx.x]);

// Plain kernel: lane i of the grid runs stream i to the end (nested loops, no queue).
#ifndef MCPET_PLAIN_WAVES
#define MCPET_PLAIN_WAVES 4
#endif
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MCPET_PLAIN_WAVES, 8))) void k_transport_plain(KParams P)
{
  K_PROLOGUE(FullCounters)
  const long long sid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (sid < P.n_streams) {
    Stream st;
    stream_init(P, sid, st);
    C.inc(KC_STREAMS);
    while (decay(P, st, C, s_cmp, s_spec, s_mat)) {
    }
    stream_finish(P, st);
  }
  K_EPILOGUE
}

// Persistent kernel: every lane is a small state machine over the phases of a decay
//   DECAY    : (refill a stream from the device queue,) sample the decay time, emit photon 1
//   STEP     : one Woodcock step of the current photon
//   INTERACT : one real interaction (Compton / Rayleigh / photoelectric + dose)
//   SOURCE2  : emit photon 2 of the pair
//   TALLY    : detector, energy blur, sinogram / PSF tallies of the pair
//   CTAU     : one trial of GCOa's tau loop
//   CPZ      : one trial of GCOa's p_z loop (+ completion of the Compton event)
//   DETECT   : singles list: detector hit, energy blur and record of the photon just ended
//   SOURCE3  : emit the decay's prompt gamma (isotropic)
// and each iteration the wave executes the one phase held by the most lanes (ballot
// counts). Lanes in other phases wait, so expensive phases (Compton rejection trials,
// detector geometry) run with many lanes at once instead of one or two, and a lane that
// needs more rejection trials than its neighbours does not hold them back. The phases that
// follow the selected one along a photon's path (GCOa's trials after an interaction, Woodcock
// steps after a Compton event or an emission, the next decay after a pair tally) run in the
// same iteration for every lane that has reached them. A lane's own sequence of random
// numbers and operations is unchanged.
enum LaneState {
  LS_DECAY = 0, LS_SOURCE2 = 1, LS_STEP = 2, LS_INTERACT = 3, LS_TALLY = 4, LS_CTAU = 5, LS_CPZ = 6, LS_DETECT = 7,
  LS_SOURCE3 = 8, LS_N = 9, LS_DONE = 10
};

// Per-lane state that only some phases touch lives in LDS slots instead of registers
// (structure of arrays, slot k of lane i at [k][i]: consecutive lanes, consecutive banks):
// the pair kept between the two photons and the Compton sampler's state between its rejection
// trials (22 words in all). Only the stream, the current photon and a ready next stream stay in
// registers across iterations.
#define K_BLOCK 256
// Slots whose contents are never needed together share a place: photon 1's direction waits for
// photon 2's emission where the pair's first hit goes later, and moves to the Compton sampler's
// slots when photon 1 has ended.
enum PairSlot { PS_P1 = 0, PS_POSF = 3, PS_DIRF = 6, PS_EF = 9, PS_SSF = 10, PS_N = 11, PS_D1 = PS_POSF };
enum ComptonSlot {
  CS_A1 = PS_N, CS_S0, CS_TAUMIN, CS_TAU, CS_S, CS_RC0, CS_RC1, CS_RC2, CS_RC3, CS_CDT1_LO, CS_CDT1_HI, LANE_SLOTS,
  CS_PROB = CS_A1, CS_MFPD, CS_RANDNO,   // a real interaction's inputs until GCOa starts
  PS_D1_LATER = CS_A1,                   // photon 1's direction between the two photons
  PS_TRAVELF = LANE_SLOTS, LANE_SLOTS_EXT   // photon 1's path, only where records are listed
};

struct LaneSlots {
  float* p;  // &slots[0][lane]
  __device__ __forceinline__ float& operator[](int k) const { return p[k * K_BLOCK]; }
};

__device__ __forceinline__ void pair_store_source(const LaneSlots& L, const Pair& pr)
{
  for (int k = 0; k < 3; k++) {
    L[PS_P1 + k] = pr.p1[k];
    L[PS_D1 + k] = pr.d1[k];
  }
  L[PS_EF] = pr.EF;
}
__device__ __forceinline__ void pair_keep_d1(const LaneSlots& L)
{
  for (int k = 0; k < 3; k++) L[PS_D1_LATER + k] = L[PS_D1 + k];
}
template <bool kExt>
__device__ __forceinline__ void pair_store_first(const LaneSlots& L, const Photon& ph)
{
  if (ph.index > -1) {   // as keep_first
    L[PS_EF] = ph.E;
    if (kExt) L[PS_TRAVELF] = ph.travel;
    L[PS_SSF] = __int_as_float(ph.ss);
    for (int k = 0; k < 3; k++) {
      L[PS_POSF + k] = ph.pos[k];
      L[PS_DIRF + k] = ph.dir[k];
    }
  }
}
template <bool kExt>
__device__ __forceinline__ void pair_load(const LaneSlots& L, Pair& pr)
{
  for (int k = 0; k < 3; k++) {
    pr.posF[k] = L[PS_POSF + k];
    pr.dirF[k] = L[PS_DIRF + k];
  }
  pr.EF = L[PS_EF];
  pr.travelF = kExt ? L[PS_TRAVELF] : 0.0f;
  pr.ssF = __float_as_int(L[PS_SSF]);
}
__device__ __forceinline__ void cs_store(const LaneSlots& L, const ComptonState& cs)
{
  L[CS_A1] = cs.a1;
  L[CS_S0] = cs.s0;
  L[CS_TAUMIN] = cs.taumin;
  L[CS_TAU] = cs.tau;
  L[CS_S] = cs.s;
  L[CS_RC0] = cs.rc0;
  L[CS_RC1] = cs.rc1;
  L[CS_RC2] = cs.rc2;
  L[CS_RC3] = cs.rc3;
  const unsigned long long b = (unsigned long long)__double_as_longlong(cs.cdt1);
  L[CS_CDT1_LO] = __uint_as_float((unsigned)b);
  L[CS_CDT1_HI] = __uint_as_float((unsigned)(b >> 32));
}
__device__ __forceinline__ void cs_load(const LaneSlots& L, ComptonState& cs)
{
  cs.a1 = L[CS_A1];
  cs.s0 = L[CS_S0];
  cs.taumin = L[CS_TAUMIN];
  cs.tau = L[CS_TAU];
  cs.s = L[CS_S];
  cs.rc0 = L[CS_RC0];
  cs.rc1 = L[CS_RC1];
  cs.rc2 = L[CS_RC2];
  cs.rc3 = L[CS_RC3];
  const unsigned long long b = (unsigned long long)__float_as_uint(L[CS_CDT1_LO]) |
                               ((unsigned long long)__float_as_uint(L[CS_CDT1_HI]) << 32);
  cs.cdt1 = __longlong_as_double((long long)b);
}

// Next state once the current photon has escaped or was absorbed (K:418-442). Photons are
// numbered 1, 2 (annihilation pair) and 3 (prompt gamma); the singles pipeline records every
// photon in DETECT instead of pairing them here.
template <bool kExt>
__device__ __forceinline__ int after_photon(const KParams& P, bool singles, int photon_no, bool prompt, const Photon& ph, const LaneSlots& L)
{
  if (photon_no == 1) pair_keep_d1(L);
  if (singles) return LS_DETECT;
  if (photon_no == 1) {
    pair_store_first<kExt>(L, ph);
    return LS_SOURCE2;
  }
  if (photon_no == 2 && ph.index > -1 && L[PS_EF] > -0.5f && pair_selected(P, ph.ss, __float_as_int(L[PS_SSF])))
    return LS_TALLY;
  return (photon_no == 2 && prompt) ? LS_SOURCE3 : LS_DECAY;
}

// The state machine of one wave on one phantom, until the phantom's stream queue is empty
// and every lane of the wave has finished its stream. kExt: a phase-space file, the singles list
// or prompt gammas are in use (staged records, phases DETECT and SOURCE3 exist); otherwise the
// wave only ballots over the seven phases of the sinogram's pair tallies.
// Streams are claimed from the queue by the wave, many indices per atomic, and handed to
// the lanes that need one in lane order; the wave's unused range (next index wq[0], count
// wq[1]) lives in LDS
// (a single global counter updated once per stream was the limit of short runs). The range
// is read by every lane and written by the lowest one; volatile keeps each access an LDS
// operation in program order, which a wave executes in order. Dealt thinly (shares > 0), the
// queue counts shares: one atomic claims the streams share, share + shares, ... of `lanes` lanes.
// A wave's first chunk (share) is that of its own number, without an atomic (`first` chunks are
// given out that way; the queue counts the others).
// Index (from the queue's origin) of the next stream for every calling lane.
__device__ __forceinline__ long long claim_stream(unsigned long long* queue, volatile K_LDS long long* wq, int lanes,
                                                               int shares, int first, int chunk0, int chunk_min, int shift,
                                                               long long n)
{
  // the lanes here all need a stream: rank among them, claim a new chunk if short
  // (the range is wave-uniform: read into scalar registers)
  const unsigned long long need = __ballot(1);
  const int cnt = __popcll(need);
  const int rank = __popcll(need & ((1ull << __lane_id()) - 1ull));
  const int step = shares ? shares : 1;
  const long long q0 = wq[0];
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)q0);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long long)q0 >> 32));
  const long long qn = (long long)(((unsigned long long)hi << 32) | lo);
  const int avail = __builtin_amdgcn_readfirstlane((int)wq[1]);
  long long idx;
  if (avail >= cnt) {
    idx = qn + rank * step;
    if (rank == 0) {
      wq[0] = qn + cnt * step;
      wq[1] = avail - cnt;
    }
  } else {
    unsigned long long base = 0;
    // a part of the rest as far as this wave knows it (from its last claim)
    const int more = shares ? lanes : max(cnt - avail, (int)min(512ll, max((long long)chunk_min, (n - qn) >> shift)));
    if (rank == 0) base = gatomic_add(queue, shares ? 1ull : (unsigned long long)more);
    const unsigned blo = __builtin_amdgcn_readfirstlane((unsigned)base);
    const unsigned bhi = __builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
    long long b = (long long)(((unsigned long long)bhi << 32) | blo) + (long long)first * (shares ? 1 : chunk0);
    if (shares && b >= shares) b = 1ll << 62;   // no share is left
    idx = rank < avail ? qn + rank * step : b + (rank - avail) * step;
    if (rank == 0) {
      wq[0] = b + (cnt - avail) * step;
      wq[1] = more - (cnt - avail);
    }
  }
  return idx;
}

// Streams made ready by the whole wave: the lanes' next streams, each advanced to its first decay. Only a
// few lanes of a wave ask at a time, and many streams of a low activity have no decay at all; seeding
// (skip-ahead, voxel, first decay time) costs the same for 64 lanes as for the one that asks. They wait in
// eight registers and go to the lanes that ask by a cross-lane read. Head, 1e8 decays, 28.5 -> 27.3 ms;
// eight phantoms, 3.2e7 decays, 7.9 -> 6.7; 4e6 ragged 1.19 -> 1.08.
// `flags` bit 0: the index was a stream of this run, bit 1: it has a decay.
struct NextStream {
  int x, y;                       // generator state after the first decay time
  unsigned remaining[2], inv_act[2];
  unsigned tid;
  int absvox, flags;
};
struct NoCounters {
  __device__ __forceinline__ void inc(int) {}
  __device__ __forceinline__ void add(int, unsigned) {}
};
// Claims for as many lanes as the queue's rest allows (the claims' own rule: at its end a wave must not
// hold streams that others could run). Not inlined: in the state machine its registers would be
// every phase's.
__device__ __attribute__((noinline)) NextStream next_streams(const KParams* Pp, volatile K_LDS long long* wq, int first)
{
  const KParams& P = *Pp;
  NextStream q;
  q.flags = 0;
  const long long q0 = wq[0];
  const int rest = (int)min(64ll, (P.n_claims - q0) >> P.chunk_shift);
  // what the wave already holds, without a claim; else as many as a claim
  const int held = __builtin_amdgcn_readfirstlane((int)wq[1]);
  const int width = held > 0 ? min(64, held)
                             : P.shares ? P.lanes : max(min(P.chunk_min, 64), __builtin_amdgcn_readfirstlane(rest));
  if ((int)__lane_id() < width) {
    const long long idx = claim_stream(P.queue, wq, P.lanes, P.shares, first, P.chunk0, P.chunk_min, P.chunk_shift, P.n_claims);
    const long long sid = P.stream_base + (P.stream_stride > 1 ? idx * P.stream_stride : idx);
    if (sid < P.n_streams) {
      Stream st;
      NoCounters none;
      stream_init(P, sid, st);
      q.flags = 1;
      if (decay_time(P, st, none)) q.flags = 3;
      else stream_finish(P, st);
      const unsigned long long a = (unsigned long long)__double_as_longlong(st.inv_act);
      q.x = st.r.x;
      q.y = st.r.y;
      q.remaining[0] = (unsigned)st.remaining;
      q.remaining[1] = (unsigned)(st.remaining >> 32);
      q.inv_act[0] = (unsigned)a;
      q.inv_act[1] = (unsigned)(a >> 32);
      q.tid = (unsigned)(st.event >> 32);
      q.absvox = st.absvox;
    }
  }
  return q;
}
// position of the k-th (from 0) set bit of m; k < popcount(m)
__device__ __forceinline__ int nth_bit(unsigned long long m, int k)
{
  unsigned w = (unsigned)m;
  int c = __popc(w), at = 0;
  if (k >= c) {
    k -= c;
    w = (unsigned)(m >> 32);
    at = 32;
  }
#pragma unroll
  for (int h = 16; h > 0; h >>= 1) {
    c = __popc(w & ((1u << h) - 1u));
    if (k >= c) {
      k -= c;
      w >>= h;
      at += h;
    }
  }
  return at;
}
__device__ __forceinline__ unsigned from_lane(int lane, unsigned v) { return (unsigned)__builtin_amdgcn_ds_bpermute(4 * lane, (int)v); }

template <class CN, bool kExt>
__device__ __forceinline__ void sm_waves(const KParams& P, CN& C, const Shells& s_cmp, int* s_spec,
                                         unsigned long long* s_mat, const LaneSlots& L, volatile K_LDS long long* wq, HitQueue hq,
                                         int wave = 0, int first = 0)
{
  constexpr int kPhases = kExt ? LS_N : LS_CPZ + 1;
  if (__lane_id() == 0) {
    // the wave's own first chunk, where chunks are given out that way
    // (dealt thinly: the first share; the waves of one workgroup take shares far apart, so that the
    // longest streams run on different CUs)
    if (first && P.shares) {
      const int share = (wave % (int)(blockDim.x >> 6)) * (int)gridDim.x + (int)blockIdx.x;
      wq[0] = share < P.shares ? (long long)share : 1ll << 62;
      wq[1] = P.lanes;
    } else {
      wq[0] = first ? (long long)wave * P.chunk0 : 0;
      wq[1] = first ? P.chunk0 : 0;
    }
    wq[2] = 0;
    wq[3] = 0;
  }
  __builtin_amdgcn_wave_barrier();
  char* const stage = kExt ? stage_of(P) : nullptr;
  const bool singles = kExt && P.mode == MCPET_TALLY_SINGLES;
  Stream st;
  Photon ph;
  bool have = false;
  bool prompt = false;           // the current decay still has its prompt gamma to emit
  int photon_no = 1;
  int trials = 0;                // of the current GCOa loop
  int state = (int)__lane_id() < P.lanes ? LS_DECAY : LS_DONE;
  NextStream next;                    // of lane i: a stream that waits if bit i of `ready` is set
  unsigned long long ready = 0ull;
  bool spent = false;                 // the queue has no streams left
  for (;;) {
    int best = -1;
    if (P.sm_policy == 0) {
      int bestc = 0;
#pragma unroll
      for (int sidx = 0; sidx < kPhases; sidx++) {
        const int c = __popcll(__ballot(state == sidx));
        if (c > bestc) {
          bestc = c;
          best = sidx;
        }
      }
    } else {
      int bestw = 0x7fffffff;
#pragma unroll
      for (int sidx = 0; sidx < kPhases; sidx++) {
        const int c = __popcll(__ballot(state == sidx));
        const int w = (64 - c) * P.sm_cost[sidx];
        if (c > 0 && w < bestw) {
          bestw = w;
          best = sidx;
        }
      }
    }
    best = __builtin_amdgcn_readfirstlane(best);
    if (stage) {   // the whole wave is here: 64 records at a time, all of them at the end
      for (;;) {
        const int c = __builtin_amdgcn_readfirstlane((int)wq[2]);
        if (c < (best < 0 ? 1 : 64)) break;
        stage_flush(P, stage, wq, c, min(c, 64));
      }
    }
    if (best < 0) break;
#if MCPET_SM_STATS
    const long long t_phase = clock64();
    {
      const int lanes = __popcll(__ballot(state == best));
      if (__lane_id() == 0) {
        C.add(KC_PHASE_EXEC + best, 1u);
        C.add(KC_PHASE_LANES + best, (unsigned)lanes);
      }
    }
#endif
    // The phases as blocks, each run for the lanes in its state when the wave selected it. With
    // chaining (MCPET_CHAIN) a block also runs right after the block that feeds it, for every
    // lane then in its state (the lanes that just arrived and those already waiting): a
    // Compton event's trials and the photon's next Woodcock steps follow its interaction
    // without a phase selection in between. The block order (a chained block comes after its
    // feeder) is the one with the fewest spilled registers among those measured.
    const bool run_int = best == LS_INTERACT;
    if (run_int && state == LS_INTERACT) {
      ComptonState cs;
      ph.prob = L[CS_PROB];
      ph.mfp_density = L[CS_MFPD];
      ph.randno = L[CS_RANDNO];
      const int o = interaction_begin(P, ph, st.r, C, s_cmp, cs, s_mat);
      if (o == IA_COMPTON) {
        cs_store(L, cs);
        trials = 0;
        state = LS_CTAU;
      } else if (o == IA_ABSORBED) {
        state = after_photon<kExt>(P, singles, photon_no, prompt, ph, L);
      } else {
        state = LS_STEP;
      }
    }
    const bool run_tau = best == LS_CTAU || ((MCPET_CHAIN & 1) && run_int);
    if (run_tau && state == LS_CTAU) {
      ComptonState cs;
      cs_load(L, cs);
      cs.trials = trials;
      bool ok;
      int k = 0;
      do {
        ok = gcoa_tau_trial(ph.E, ph.mat0, st.r, C, s_cmp, cs);
      } while (!ok && ++k < MCPET_TRIALS_PER_PHASE);
      trials = cs.trials;
      if (ok) {
        trials = 0;
        state = LS_CPZ;
      }
      cs_store(L, cs);
    }
    const bool run_pz = best == LS_CPZ || ((MCPET_CHAIN & 2) && run_tau);
    if (run_pz && state == LS_CPZ) {
      ComptonState cs;
      cs_load(L, cs);
      cs.trials = trials;
      bool ok;
      int k = 0;
      do {
        ok = gcoa_pz_trial(ph.E, ph.mat0, st.r, C, s_cmp, cs);
      } while (!ok && ++k < MCPET_TRIALS_PER_PHASE);
      if (ok) {
        // (the photon is where its last step found it inside the box)
        if (!compton_end(P, ph, st.r, C, cs, s_mat)) state = after_photon<kExt>(P, singles, photon_no, prompt, ph, L);
        else state = LS_STEP;
      } else {
        trials = cs.trials;
      }
    }
    const bool run_tally = best == LS_TALLY;
    if (run_tally && state == LS_TALLY) {
      Pair pr;
      pair_load<kExt>(L, pr);
      tally_pair<CN, kExt>(P, ph, pr, st, C, s_spec, stage, wq, kExt ? nullptr : hq);
      state = prompt ? LS_SOURCE3 : LS_DECAY;
    }
    if (!kExt && run_tally && __builtin_amdgcn_readfirstlane((int)wq[3]) >= HIT_FULL) hits_take(P, hq, wq, C, s_spec);
    const bool run_decay = best == LS_DECAY || ((MCPET_CHAIN & 16) && run_tally);
    if (run_decay) {   // the whole wave is here
      bool go = false;
      if (state == LS_DECAY && have) {
        go = decay_time(P, st, C);
        if (!go) {
          stream_finish(P, st);
          have = false;
        }
      }
      for (;;) {
        const bool want = state == LS_DECAY && !have;
        const unsigned long long need = __ballot(want);
        if (!need) break;
        if (!ready) {
          if (spent) {
            if (want) state = LS_DONE;
            break;
          }
          next = next_streams(&P, wq, first);
          if (next.flags & 1) {
            C.inc(KC_STREAMS);
            C.inc(KC_RNDRAWS);
          }
          if (next.flags & 2) C.inc(KC_DECAYS);
          spent = !__any(next.flags & 1);
          ready = __ballot(next.flags & 2);
          continue;
        }
        const int rank = __popcll(need & ((1ull << __lane_id()) - 1ull));
        const int n = min(__popcll(need), __popcll(ready));
        const bool mine = want && rank < n;
        const int src = nth_bit(ready, min(rank, n - 1));
        const unsigned w[8] = {from_lane(src, (unsigned)next.x), from_lane(src, (unsigned)next.y), from_lane(src, next.remaining[0]),
                               from_lane(src, next.remaining[1]), from_lane(src, next.inv_act[0]), from_lane(src, next.inv_act[1]),
                               from_lane(src, next.tid), from_lane(src, (unsigned)next.absvox)};
        if (mine) {
          st.r.x = (int)w[0];
          st.r.y = (int)w[1];
          st.remaining = (unsigned long long)w[3] << 32 | w[2];
          st.inv_act = __longlong_as_double((long long)((unsigned long long)w[5] << 32 | w[4]));
          st.event = ((unsigned long long)w[6] << 32) + 1ull;   // at its first decay
          st.absvox = (int)w[7];
          have = go = true;
        }
        for (int k = 0; k < n; k++) ready &= ready - 1ull;
      }
      if (go) {
        // decay branches (no draws for a pure positron emitter without prompt gamma)
        bool pair = true;
        if (P.positron_frac < 1.0f) pair = rn(st.r, C) < P.positron_frac;
        prompt = false;
        if (P.prompt_frac > 0.0f) prompt = rn(st.r, C) < P.prompt_frac;
        Pair pr;
        source_first(P, st, C, pr.p1, pr.d1);
        pr.EF = -10.0f;
        pair_store_source(L, pr);
        if (prompt) C.inc(KC_EMIT_PROMPT);
        if (pair) {
          C.inc(KC_EMIT_PAIR);
          for (int k = 0; k < 3; k++) {
            ph.pos[k] = pr.p1[k];
            ph.dir[k] = pr.d1[k];
          }
          photon_start(P, ph);
          photon_no = 1;
          state = (locate(P, ph.pos) < 0) ? after_photon<kExt>(P, singles, 1, prompt, ph, L) : LS_STEP;
        } else {
          state = prompt ? LS_SOURCE3 : LS_DECAY;
        }
      }
    }
    const bool run_src2 = best == LS_SOURCE2;
    if (run_src2 && state == LS_SOURCE2) {
      float p1[3], d1[3];
      for (int k = 0; k < 3; k++) {
        p1[k] = L[PS_P1 + k];
        d1[k] = L[PS_D1_LATER + k];
      }
      source_second(P, st, C, d1, ph.dir);
      for (int k = 0; k < 3; k++) ph.pos[k] = p1[k];
      photon_start(P, ph);
      photon_no = 2;
      state = (locate(P, ph.pos) < 0) ? after_photon<kExt>(P, singles, 2, prompt, ph, L) : LS_STEP;
    }
    const bool run_det = kExt && best == LS_DETECT;
    if (run_det && state == LS_DETECT) {
      if (ph.index > -1) record_single(P, ph.pos, ph.dir, ph.E, ph.travel, ph.ss, photon_no - 1, st, C, s_spec, stage, wq);
      state = (photon_no == 1) ? LS_SOURCE2 : (photon_no == 2 && prompt) ? LS_SOURCE3 : LS_DECAY;
    }
    const bool run_src3 = kExt && best == LS_SOURCE3;
    if (run_src3 && state == LS_SOURCE3) {
      for (int k = 0; k < 3; k++) ph.pos[k] = L[PS_P1 + k];
      isotropic_dir(st, C, ph.dir);
      photon_start(P, ph, P.prompt_energy);
      photon_no = 3;
      prompt = false;
      state = (locate(P, ph.pos) < 0) ? after_photon<kExt>(P, singles, 3, false, ph, L) : LS_STEP;
    }
    const bool run_step = best == LS_STEP || ((MCPET_CHAIN & 4) && run_pz) ||
                          ((MCPET_CHAIN & 8) && (run_decay || run_src2 || run_src3));
    if (run_step && state == LS_STEP) {
      const StepParams S = P;   // one block of scalar loads
      int o, k = 0;
      do {
        o = woodcock_step(S, s_cmp.pal, ph, st.r, C);
      } while (o == STEP_VIRTUAL && ++k < MCPET_STEPS_PER_PHASE);
      if (o == STEP_ESCAPED) {
        state = after_photon<kExt>(P, singles, photon_no, prompt, ph, L);
      } else if (o == STEP_REAL) {
        // the interaction's inputs wait in LDS (Compton slots, free until GCOa starts)
        L[CS_PROB] = ph.prob;
        L[CS_MFPD] = ph.mfp_density;
        L[CS_RANDNO] = ph.randno;
        state = LS_INTERACT;
      }
    }
#if MCPET_SM_STATS
    if (__lane_id() == 0) C.add(KC_PHASE_CYCLES + best, (unsigned)(clock64() - t_phase));
#endif
  }
  if (!kExt) hits_take(P, hq, wq, C, s_spec);   // the last ones
}

// Persistent kernel over one phantom.
template <class CN, bool kExt>
// Parameters are read through a pointer to device memory: only the fields a phase uses are
// loaded (as scalars), instead of a by-value block that would be kept in scalar registers
// (and spilled) or copied to private memory.
__global__ __launch_bounds__(K_BLOCK) K_OCCUPANCY void k_transport_sm(const KParams* __restrict__ Pd)
{
  const KParams& P = *Pd;
  K_PROLOGUE(CN)
  __shared__ float s_slots[kExt ? LANE_SLOTS_EXT : LANE_SLOTS][K_BLOCK];
  __shared__ long long s_wq[K_BLOCK / 64][4];
  __shared__ float s_hits[K_BLOCK / 64][kExt ? 1 : HIT_WORDS * HIT_LEN];
  const LaneSlots L{&s_slots[0][threadIdx.x]};
  const int waves = (int)(blockDim.x >> 6), wave = (int)(threadIdx.x >> 6);
  sm_waves<CN, kExt>(P, C, s_cmp, s_spec, s_mat, L, (volatile K_LDS long long*)s_wq[wave], (HitQueue)s_hits[wave], (int)blockIdx.x * waves + wave,
                     P.chunk0 ? (int)gridDim.x * waves : 0);
  K_EPILOGUE
}

// Batched persistent kernel over n phantoms that share their interaction tables and
// scanner (params Ps[0..n-1], one per phantom, each with its own stream queue, voxels and
// tallies). Every workgroup works on one phantom at a time, so all parameters stay uniform and
// the spectrum is a sum in LDS as in the single-phantom kernel (added up in global memory its few
// hot bins took a fifth of the time: 16 phantoms, 2.3e8 decays, 62.7 -> 50.5 ms): its waves pull streams from that phantom's queue, and
// when the queue is empty and their lanes are done, they flush counters and material dose (per-wave
// LDS slices) and the workgroup the spectrum to that phantom and move to the next one. Workgroups
// start at different phantoms and visit every phantom once, so the phantoms' queues drain
// concurrently and no phantom waits for a launch of its own. The palette is read from global
// memory. Per phantom, streams and random numbers are those of a single-phantom run, so each
// phantom's tallies equal its own run's bit for bit.
template <class CN, bool kExt>
__global__ __launch_bounds__(K_BLOCK) K_OCCUPANCY void k_transport_batch(const KParams* __restrict__ Ps, int n, int n_spec)
{
  __shared__ unsigned s_shell_of[K_MAXMAT];
  extern __shared__ v4f s_dyn[];                          // the shells, n_spec spectrum bins
  int* const s_spec = (int*)(s_dyn + Ps[0].n_shells);
  __shared__ unsigned long long s_matw[K_BLOCK / 64][2 * K_MAXMAT];
  __shared__ unsigned s_cntw[K_BLOCK / 64][KC_N];
  __shared__ float s_slots[kExt ? LANE_SLOTS_EXT : LANE_SLOTS][K_BLOCK];
  __shared__ long long s_wq[K_BLOCK / 64][4];
  __shared__ float s_hits[K_BLOCK / 64][kExt ? 1 : HIT_WORDS * HIT_LEN];
  {
    for (int i = threadIdx.x; i < Ps[0].n_shells; i += blockDim.x) {
      const float4 v = gld(Ps[0].shells, i);
      s_dyn[i] = v4f{v.x, v.y, v.z, v.w};
    }
    if (threadIdx.x < K_MAXMAT) s_shell_of[threadIdx.x] = Ps[0].shell_of[threadIdx.x];
    for (int i = threadIdx.x; i < (K_BLOCK / 64) * 2 * K_MAXMAT; i += blockDim.x) (&s_matw[0][0])[i] = 0ull;
    for (int i = threadIdx.x; i < (K_BLOCK / 64) * KC_N; i += blockDim.x) (&s_cntw[0][0])[i] = 0u;
    load_tot511(Ps[0]);   // the phantoms of a batch share their interaction tables
    for (int i = threadIdx.x; i < n_spec; i += blockDim.x) s_spec[i] = 0;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const LaneSlots L{&s_slots[0][threadIdx.x]};
  const Shells s_cmp{(const K_LDS v4f*)s_dyn, (const K_LDS unsigned*)s_shell_of, nullptr};
  const int first = (int)blockIdx.x % n;
  for (int j = 0; j < n; j++) {
    const int k = __builtin_amdgcn_readfirstlane((first + j) % n);
    const KParams& P = Ps[k];
    CN C;
    C.init(s_cntw[wave]);
    sm_waves<CN, kExt>(P, C, s_cmp, s_spec, s_matw[wave], L, (volatile K_LDS long long*)s_wq[wave], (HitQueue)s_hits[wave]);
    C.flush(P, s_cntw[wave]);
    __builtin_amdgcn_wave_barrier();
    if (lane < KC_N && s_cntw[wave][lane]) {
      gatomic_add(&P.counters[lane], (unsigned long long)s_cntw[wave][lane]);
      s_cntw[wave][lane] = 0u;
    }
    if (lane < 2 * K_MAXMAT && s_matw[wave][lane]) {
      gatomic_add(&P.mat_edep[lane], s_matw[wave][lane]);
      s_matw[wave][lane] = 0ull;
    }
    __builtin_amdgcn_wave_barrier();
    if (P.lds_spectrum) {   // uniform: every wave of the workgroup is at this phantom
      __syncthreads();
      for (int i = threadIdx.x; i < P.ne; i += blockDim.x)
        if (s_spec[i]) {
          gatomic_add(&P.spectrum[i], s_spec[i]);
          s_spec[i] = 0;
        }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------------- self tests

__global__ void k_selftest_ranecu(int seed, const long long* ids, int nstreams, int n, float* out, double* out_d, int as_double,
                                  const uint32_t* j1, const uint32_t* j2)
{
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nstreams) return;
  int sx, sy;
  init_stream_seeds(ids[i], seed, j1, j2, &sx, &sy);
  for (int k = 0; k < n; k++) {
    if (as_double) out_d[(size_t)i * n + k] = mcr_ranecu_double(&sx, &sy);
    else out[(size_t)i * n + k] = mcr_ranecu(&sx, &sy);
  }
}

__global__ void k_selftest_fmath(const double* x, const double* y, int n, double* od, float* of)
{
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double a = x[i], b = y[i];
  double s, c;
  mcf_sincos(a, &s, &c);
  od[0 * (size_t)n + i] = mcf_log(fabs(a) + 1e-300);
  od[1 * (size_t)n + i] = mcf_exp(a);
  od[2 * (size_t)n + i] = s;
  od[3 * (size_t)n + i] = c;
  od[4 * (size_t)n + i] = mcf_atan2(a, b);
  od[5 * (size_t)n + i] = mcf_acos(fmin(fmax(b, -1.0), 1.0));
  od[6 * (size_t)n + i] = sqrt(fabs(a));
  float af = (float)a, bf = (float)b, sf, cf;
  mcf_sincosf(af, &sf, &cf);
  of[0 * (size_t)n + i] = mcf_logf(fabsf(af) + 1e-30f);
  of[1 * (size_t)n + i] = mcf_expf(af);
  of[2 * (size_t)n + i] = mcf_powf(fminf(fabsf(bf), 1.0f), fabsf(af));
  of[3 * (size_t)n + i] = sf;
  of[4 * (size_t)n + i] = cf;
  of[5 * (size_t)n + i] = mcf_atan2f(af, bf);
  of[6 * (size_t)n + i] = sqrtf(fabsf(af)) / (bf + 3.0f);
  of[7 * (size_t)n + i] = mcf_acosf(fminf(fmaxf(bf, -1.0f), 1.0f));
}

// Differences between the functions of fastmath.h (and mcr_step) and the general ones (fmath.h, f2i_rd, IEEE
// division and root, 64-bit remainders) over n arguments of the stated ranges: every float from bit
// pattern `first` on where a range is a set of floats (every state of both generators for mcr_step), else drawn from the
// argument's number, in part next to the values where a rounding, an exponent or a quadrant changes.
// res[0]: the differences, res[1]: the smallest argument number with one, res[2]: the arguments in range.
enum FastFn {
  FF_FLOOR, FF_FLOOR_NAN, FF_SQRT, FF_LOG, FF_EXP, FF_SINCOS, FF_DIV_1000, FF_RANECU,   // argument: first + i
  FF_DIV, FF_DIV_R, FF_DDIV, FF_DSQRT, FF_DLOG, FF_DEXP, FF_DSINCOS,                             // drawn
  FF_N
};
__device__ __forceinline__ unsigned long long ff_draw(unsigned long long& z)   // splitmix64
{
  z += 0x9E3779B97F4A7C15ull;
  unsigned long long x = z;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
// a float with exponent in [-e, e]; of its mantissas one in four has only its first or last bits set or cleared
__device__ __forceinline__ float ff_float(unsigned long long& z, int e)
{
  const unsigned long long h = ff_draw(z);
  unsigned m = (unsigned)h & 0x7fffffu;
  if ((h >> 60) == 0) m &= 7u;
  if ((h >> 60) == 1) m |= 0x7ffff8u;
  if ((h >> 60) == 2) m &= 0x700000u;
  if ((h >> 60) == 3) m |= 0x0fffffu;
  return mcf_ffrom((unsigned)(127 + (int)((h >> 32) % (2 * e + 1)) - e) << 23 | m | ((unsigned)(h >> 59) & 1u) << 31);
}
__device__ __forceinline__ double ff_double(unsigned long long& z, int e)
{
  const unsigned long long h = ff_draw(z), k = ff_draw(z);
  unsigned long long m = h & 0xfffffffffffffull;
  if ((k >> 60) == 0) m &= 7ull;
  if ((k >> 60) == 1) m |= 0xffffffffffff8ull;
  if ((k >> 60) == 2) m &= 0xe000000000000ull;
  if ((k >> 60) == 3) m |= 0x1ffffffffffffull;
  return mcf_from_bits((unsigned long long)(1023 + (int)((unsigned)(k >> 32) % (unsigned)(2 * e + 1)) - e) << 52 | m | (k & 1ull) << 63);
}
// x moved by -2 .. 2 of its last places
__device__ __forceinline__ float ff_near(float x, unsigned long long& z) { return mcf_ffrom(mcf_fbits(x) + (unsigned)(ff_draw(z) % 5) - 2u); }
__device__ __forceinline__ double ff_near(double x, unsigned long long& z) { return mcf_from_bits(mcf_bits(x) + ff_draw(z) % 5 - 2ull); }
// equal bits; a NaN equals any
__device__ __forceinline__ bool ff_same(float a, float b) { return mcf_fbits(a) == mcf_fbits(b) || (a != a && b != b); }
__device__ __forceinline__ bool ff_same(double a, double b) { return mcf_bits(a) == mcf_bits(b) || (a != a && b != b); }

// 1: they differ on argument i, 0: they do not, -1: it is outside the function's range
template <int FN>
__device__ __forceinline__ int ff_compare(unsigned long long first, unsigned long long i)
{
  const float x = mcf_ffrom((unsigned)(first + i));
  const int state = (int)(first + i);
  unsigned long long z = (first + i) * 0xD1342543DE82EF95ull;
  if (FN == FF_FLOOR) return x != x ? -1 : floor_i32(x) != f2i_rd(x);
  if (FN == FF_FLOOR_NAN) return floor_i32_nan(x) != f2i_rd(x);
  if (FN == FF_SQRT) return !(x == 0.0f || (x > 0x1p-100f && x < MCF_INFF)) ? -1 : !ff_same(sqrt_nz(x), sqrtf(x));
  if (FN == FF_LOG) return !(x >= 0x1p-126f && x < MCF_INFF) ? -1 : !ff_same(log_n(x), mcf_logf(x));
  if (FN == FF_EXP) return x > 88.0f ? -1 : !ff_same(exp_n(x), mcf_expf(x));   // NaN stays NaN
  if (FN == FF_SINCOS) {
    if (!(fabsf(x) < 8192.0f)) return -1;
    float s, c, ms, mc;
    sincos_n(x, &s, &c);
    mcf_sincosf(x, &ms, &mc);
    return !ff_same(s, ms) || !ff_same(c, mc) || !ff_same(cos_n(x), mc);
  }
  if (FN == FF_DIV_1000) {   // (tallied energies over 1000: quotients from 2^-80 up, and floors of positive ones anywhere)
    const bool normal = fabsf(x) >= 0x1p-80f;
    if (!(fabsf(x) < MCF_INFF) || !(normal || x >= 0.0f)) return -1;
    const float q = div_r(x, 1000.0f, 1.0f / 1000.0f);
    return (normal && !ff_same(q, x / 1000.0f)) || floor_i32_nan(q) != f2i_rd(x / 1000.0f);
  }
  if (FN == FF_RANECU) {
    if (state < 1 || state >= MCR_M1) return -1;
    const int y0 = state < MCR_M2 ? state : 1;
    int sx = state, sy = y0;
    const int out = mcr_step(&sx, &sy);
    const int x1 = (int)(40014ull * (unsigned)state % (unsigned)MCR_M1), y1 = (int)(40692ull * (unsigned)y0 % (unsigned)MCR_M2);
    return sx != x1 || sy != y1 || out != (x1 - y1 < 1 ? x1 - y1 + (MCR_M1 - 1) : x1 - y1);
  }
  if (FN == FF_DIV || FN == FF_DIV_R) {   // half of the quotients next to a float, some of these next to an integer
    const float b = ff_float(z, 30);
    float a = ff_float(z, 30);
    const unsigned long long how = ff_draw(z) & 3;
    if (how < 2) a = ff_near((how ? rintf(ff_float(z, 12)) : ff_float(z, 30)) * b, z);
    if (!(fabsf(a) >= 0x1p-62f && fabsf(a) < 0x1p62f)) return -1;
    return !ff_same(FN == FF_DIV ? div_n(a, b) : div_r(a, b, 1.0f / b), a / b);
  }
  if (FN == FF_DDIV) {
    const double b = ff_double(z, 200);
    double a = ff_double(z, 200);
    const unsigned long long how = ff_draw(z) & 3;
    if (how < 2) a = ff_near((how ? rint(ff_double(z, 20)) : ff_double(z, 200)) * b, z);
    if (!(fabs(a) >= 0x1p-402 && fabs(a) < 0x1p402)) return -1;
    return !ff_same(div_n(a, b), a / b);
  }
  if (FN == FF_DSQRT) {   // half of them next to a square
    double a = fabs(ff_double(z, 200));
    if (ff_draw(z) & 1) {
      const double r = ff_double(z, 100);
      a = ff_near(r * r, z);
    }
    return !ff_same(sqrt_n(a), sqrt(a));
  }
  if (FN == FF_DLOG) {   // all exponents, the generator's outputs, and next to 1 and sqrt(2)
    const unsigned long long how = ff_draw(z) & 3;
    double a = fabs(ff_double(z, 1021));
    if (how == 1) a = (double)(1 + ff_draw(z) % 2147483561ull) * (1.0 / 2147483562.0);
    if (how == 2) a = 1.0 + ff_double(z, 52) * 0x1p-53;
    if (how == 3) a = ff_near((ff_draw(z) & 1 ? 1.0 : 0x1.6a09e667f3bcdp+0) * mcf_pow2i((int)(ff_draw(z) % 101) - 50), z);
    return !(a >= 0x1p-1022) ? -1 : !ff_same(log_n(a), mcf_log(a));
  }
  if (FN == FF_DEXP) {   // every exponent below 2^10, next to where the power of two changes, and the ends
    const unsigned long long how = ff_draw(z) & 3;
    double a = (double)(ff_draw(z) >> 11) * 0x1p-53 * 712.0;
    if (how == 1) a = fabs(ff_double(z, 1000)) * 0x1p-991;
    if (how == 2) a = ff_near(((double)(ff_draw(z) % 1026) + 0.5) * 0x1.62e42fefa39efp-1, z);
    if (how == 3) a = (ff_draw(z) & 7) ? ff_near(0x1.62e42fefa39efp+9, z) : (ff_draw(z) & 1) ? 0.0 : MCF_INF;
    return !ff_same(exp_nonneg(a), mcf_exp(a));
  }
  // angles of up to 2^30 either way, and next to where the quadrant changes
  const unsigned long long how = ff_draw(z) & 3;
  double a = ((double)(ff_draw(z) >> 11) * 0x1p-52 - 1.0) * (how == 0 ? 0x1p30 : 7.0);
  if (how == 2) a = ff_near(((double)(int)(ff_draw(z) % 2000001) - 1000000.0) * 0x1.921fb54442d18p-1, z);
  if (how == 3) a = ff_double(z, 29);
  if (!(fabs(a) < 0x1p30)) return -1;
  double s, c, ms, mc;
  sincos_n(a, &s, &c);
  mcf_sincos(a, &ms, &mc);
  return !ff_same(s, ms) || !ff_same(c, mc);
}
template <int FN>
__global__ __launch_bounds__(256) void k_selftest_fastmath(unsigned long long first, unsigned long long n, unsigned long long* res)
{
  unsigned long long count = 0, least = ~0ull, compared = 0;
  for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (unsigned long long)gridDim.x * 256) {
    const int d = ff_compare<FN>(first, i);
    if (d >= 0) compared++;
    if (d > 0) {
      count++;
      least = min(least, i);
    }
  }
  atomicAdd(&res[2], compared);
  if (count) {
    atomicAdd(&res[0], count);
    atomicMin(&res[1], least);
  }
}

// Clear n words (a memset that a captured graph may hold).
__global__ void k_fill_u32(unsigned* __restrict__ p, size_t n)
{
  const size_t base = (size_t)blockIdx.x * 256 * 16 + threadIdx.x;
#pragma unroll
  for (int k = 0; k < 16; k++)
    if (base + (size_t)k * 256 < n) p[base + (size_t)k * 256] = 0u;
}

// Zero up to K_FILL_MAX regions of 4-byte words in one launch: block row y clears region y,
// its blocks grid-striding over the region's words (16-byte stores where the region allows).
struct FillRegions {
  unsigned* p[K_FILL_MAX];
  unsigned long long n[K_FILL_MAX];   // words
};
__global__ __launch_bounds__(256) void k_fill_regions(FillRegions r)
{
  unsigned* p = r.p[blockIdx.y];
  const size_t n = r.n[blockIdx.y];
  const size_t stride = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (((uintptr_t)p & 15) == 0) {
    uint4* q = (uint4*)p;
    const size_t n4 = n / 4;
    for (size_t k = i; k < n4; k += stride) q[k] = uint4{0u, 0u, 0u, 0u};
    for (size_t k = n4 * 4 + i; k < n; k += stride) p[k] = 0u;
  } else {
    for (size_t k = i; k < n; k += stride) p[k] = 0u;
  }
}

__global__ void k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n16)
{
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n16; i += stride) dst[i] = src[i];
}

}  // namespace

size_t mcpet_transport_dyn_lds(const KParams& P)
{
  return 16 * (size_t)P.n_shells + (P.vox_fmt == 1 && P.lds_palette ? 8 * (size_t)P.n_palette : 0) +
         (P.lds_spectrum ? 4 * (size_t)P.ne : 0);
}

// Workgroups of the persistent kernel that a CU holds at once.
int mcpet_transport_resident(const KParams& P, int count_events, int block_size)
{
  const bool ext = P.mode != 2 || P.prompt_frac > 0.0f;
  const void* f = count_events ? (ext ? (const void*)k_transport_sm<FullCounters, true> : (const void*)k_transport_sm<FullCounters, false>)
                               : (ext ? (const void*)k_transport_sm<LiteCounters, true> : (const void*)k_transport_sm<LiteCounters, false>);
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, block_size, mcpet_transport_dyn_lds(P)) != hipSuccess || n < 1) return 1;
  return n;
}

hipError_t mcpet_launch_transport(const KParams& P, const KParams* d_P, int kind, int count_events, int blocks, int block_size,
                                  hipStream_t stream)
{
  if (block_size > K_BLOCK || block_size % 64 != 0) return hipErrorInvalidValue;
  const size_t lds = mcpet_transport_dyn_lds(P);
  const bool ext = P.mode != 2 || P.prompt_frac > 0.0f;   // lists or prompt gammas
  if (kind == MCPET_KERNEL_PERSISTENT && count_events && ext)
    hipLaunchKernelGGL((k_transport_sm<FullCounters, true>), dim3(blocks), dim3(block_size), lds, stream, d_P);
  else if (kind == MCPET_KERNEL_PERSISTENT && count_events)
    hipLaunchKernelGGL((k_transport_sm<FullCounters, false>), dim3(blocks), dim3(block_size), lds, stream, d_P);
  else if (kind == MCPET_KERNEL_PERSISTENT && ext)
    hipLaunchKernelGGL((k_transport_sm<LiteCounters, true>), dim3(blocks), dim3(block_size), lds, stream, d_P);
  else if (kind == MCPET_KERNEL_PERSISTENT)
    hipLaunchKernelGGL((k_transport_sm<LiteCounters, false>), dim3(blocks), dim3(block_size), lds, stream, d_P);
  else
    hipLaunchKernelGGL(k_transport_plain, dim3(blocks), dim3(block_size), lds, stream, P);
  return hipGetLastError();
}

hipError_t mcpet_launch_transport_batch(const KParams* d_params, int n, int n_shells, int n_spec, bool ext, int count_events, int blocks,
                                        int block_size, hipStream_t stream)
{
  const size_t lds = 16 * (size_t)n_shells + 4 * (size_t)n_spec;
  if (block_size > K_BLOCK || block_size % 64 != 0 || n < 1) return hipErrorInvalidValue;
  if (count_events && ext)
    hipLaunchKernelGGL((k_transport_batch<FullCounters, true>), dim3(blocks), dim3(block_size), lds, stream, d_params, n, n_spec);
  else if (count_events)
    hipLaunchKernelGGL((k_transport_batch<FullCounters, false>), dim3(blocks), dim3(block_size), lds, stream, d_params, n, n_spec);
  else if (ext)
    hipLaunchKernelGGL((k_transport_batch<LiteCounters, true>), dim3(blocks), dim3(block_size), lds, stream, d_params, n, n_spec);
  else
    hipLaunchKernelGGL((k_transport_batch<LiteCounters, false>), dim3(blocks), dim3(block_size), lds, stream, d_params, n, n_spec);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------- projections

// Dense per-voxel map for the projections: .y = mu(511 keV) = density x (a + E b) of the
// voxel's material total-cross-section line (every voxel), .x = 0 (activity added next).
__global__ void k_dense_mu(const KParams* __restrict__ Pd, float2* __restrict__ out, long long nvox)
{
  const KParams& P = *Pd;
  const int idx = f2i_rd((K_E511 - P.e0) * P.ide);
  for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long long)gridDim.x * blockDim.x) {
    // the palette lives in global memory here (LDS holds it only inside the transport)
    const float2 md = P.vox_fmt == 1 ? P.palette[P.vox8[v]] : P.vox_fmt == 2 ? P.palette[P.vox16[v]] : P.vox[v];
    const float2 tb = P.tot[idx * K_MAXMAT + (__float_as_int(md.y) & 0xff)];
    out[v] = make_float2(0.0f, md.x * (tb.x + K_E511 * tb.y));
  }
}

// Activity of the emitting-voxel list into the map's .x.
__global__ void k_dense_activity(const int* __restrict__ vox, const float* __restrict__ act, long long n, float2* __restrict__ out)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[vox[i]].x = act[i];
}

// Line integrals through the phantom along the lines of response of a rebinned sinogram grid
// (the scatter surrogate's phantom inputs). Workgroup (h, w) owns the crystal pairs
// lors[off[h W + w] .. off[h W + w + 1]) of its transaxial bins; item i = d nl + l of the group
// is pair l in plane group d (plane-major: a wave's lanes share a plane, whose lines all lie in
// or all outside the phantom's axial extent), whose line runs in the plane z of the group's central ring sum
// between the two crystal centres (angle 2 pi (k + 1/2) / N - pi at radius R around the
// scanner axis) and is sampled at t0 + (j + 1/2) step < t1 inside the phantom's box [t0, t1]:
// act_out = mean over the pairs of the activity integral (Bq cm), att_out = mean of
// exp(-integral of mu(511 keV)) (map: the (activity, mu) of every voxel). One lane per item;
// the per-plane sums run over the pairs in order (deterministic).
__global__ __launch_bounds__(256) void k_project(const KParams* __restrict__ Pd, const float2* __restrict__ map,
                                                 const int2* __restrict__ lors, const int* __restrict__ off, int D, int H,
                                                 int W, int gz, float step, float* __restrict__ act_out,
                                                 float* __restrict__ att_out)
{
  const KParams& P = *Pd;
  __shared__ float s_act[256], s_att[256];
  const int g = blockIdx.x, h = g / W, w = g - h * W;
  const int l0 = off[g], nl = off[g + 1] - l0, n_items = nl * D;
  const float twopi_n = 2.0f * (float)K_PI / (float)P.ncrystals;
  float acc_a = 0.0f, acc_t = 0.0f;   // plane group threadIdx.x (< D)
  for (int base = 0; base < n_items; base += 256) {
    const int i = base + (int)threadIdx.x;
    float ia = 0.0f, im = 0.0f;
    if (i < n_items) {
      const int d = i / nl, l = i - d * nl;
      const float sc = fminf((float)(d * gz) + 0.5f * (float)(gz - 1), (float)(P.nzs - 1));
      const float z = P.cz + ((0.5f * sc + 0.5f) / (float)P.nrows - 0.5f) * P.fovz;
      const int2 pr = lors[l0 + l];
      const float f1 = twopi_n * ((float)pr.x + 0.5f) - (float)K_PI, f2 = twopi_n * ((float)pr.y + 0.5f) - (float)K_PI;
      const float ax = P.cx + P.radius * cosf(f1), ay = P.cy + P.radius * sinf(f1);
      float dx = P.cx + P.radius * cosf(f2) - ax, dy = P.cy + P.radius * sinf(f2) - ay;
      const float len = sqrtf(dx * dx + dy * dy);
      if (len > 0.0f && z > 0.0f && z < P.bz) {
        dx /= len;
        dy /= len;
        // clip to the box [0, bx] x [0, by]
        float t0 = 0.0f, t1 = len;
        const float o[2] = {ax, ay}, v[2] = {dx, dy}, hi[2] = {P.bx, P.by};
        for (int k = 0; k < 2; k++) {
          if (fabsf(v[k]) < 1e-12f) {
            if (o[k] <= 0.0f || o[k] >= hi[k]) t1 = -1.0f;
          } else {
            const float ta = (0.0f - o[k]) / v[k], tb = (hi[k] - o[k]) / v[k];
            t0 = fmaxf(t0, fminf(ta, tb));
            t1 = fminf(t1, fmaxf(ta, tb));
          }
        }
        // four samples per pass, their loads issued together
        for (int j = 0; t0 + ((float)j + 0.5f) * step < t1; j += 4) {
          float2 m[4];
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const float t = t0 + ((float)(j + u) + 0.5f) * step;
            const float p[3] = {ax + t * dx, ay + t * dy, z};
            const int v0 = t < t1 ? locate(P, p) : -1;
            m[u] = v0 >= 0 ? map[v0] : make_float2(0.0f, 0.0f);
          }
#pragma unroll
          for (int u = 0; u < 4; u++) {
            ia += m[u].x;
            im += m[u].y;
          }
        }
      }
    }
    s_act[threadIdx.x] = ia * step;
    s_att[threadIdx.x] = expf(-im * step);
    __syncthreads();
    if ((int)threadIdx.x < D) {
      // items of plane d in this chunk: i = d nl + l, in increasing l
      const int d = threadIdx.x, lo = max(base, d * nl), hi = min(base + 256, (d + 1) * nl);
      for (int i = lo; i < hi; i++) {
        acc_a += s_act[i - base];
        acc_t += s_att[i - base];
      }
    }
    __syncthreads();
  }
  if ((int)threadIdx.x < D) {
    const size_t oi = ((size_t)threadIdx.x * H + h) * W + w;
    act_out[oi] = nl > 0 ? acc_a / (float)nl : 0.0f;
    att_out[oi] = nl > 0 ? acc_t / (float)nl : 1.0f;
  }
}

// a[0..n) times float32(1 / max(a)) (a >= 0; unchanged when the maximum is 0), in two launches:
// k_max_bits folds the block maxima into *mx (float bits, which order as unsigned integers for
// a >= 0; *mx starts at 0), k_scale_by reads it. The maximum is order-independent, so the
// result is exact and reproducible.
__global__ __launch_bounds__(256) void k_max_bits(const float* __restrict__ a, int n, unsigned* __restrict__ mx)
{
  __shared__ float s[256];
  float m = 0.0f;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) m = fmaxf(m, a[i]);
  s[threadIdx.x] = m;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) s[threadIdx.x] = fmaxf(s[threadIdx.x], s[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(mx, __float_as_uint(s[0]));
}

__global__ __launch_bounds__(256) void k_scale_by(float* __restrict__ a, int n, const unsigned* __restrict__ mx)
{
  const float m = __uint_as_float(*mx);
  if (!(m > 0.0f)) return;
  const float sc = (float)(1.0 / (double)m);
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) a[i] = a[i] * sc;
}

hipError_t mcpet_launch_project(const KParams* d_params, const int* active_vox, const float* active_act, long long n_active,
                                float2* map, size_t nvox, const int2* lors, const int* off, int D, int H, int W, int gz,
                                float step, float* act_out, float* att_out, hipStream_t stream)
{
  if (D < 1 || D > 256 || H < 1 || W < 1) return hipErrorInvalidValue;
  const size_t nb = (nvox + 255) / 256;
  const unsigned mb = nb < 1 ? 1u : nb > 8192 ? 8192u : (unsigned)nb;
  hipLaunchKernelGGL(k_dense_mu, dim3(mb), dim3(256), 0, stream, d_params, map, (long long)nvox);
  if (n_active > 0)
    hipLaunchKernelGGL(k_dense_activity, dim3((unsigned)((n_active + 255) / 256)), dim3(256), 0, stream, active_vox, active_act,
                       n_active, map);
  hipLaunchKernelGGL(k_project, dim3(H * W), dim3(256), 0, stream, d_params, map, lors, off, D, H, W, gz, step, act_out,
                     att_out);
  return hipGetLastError();
}

hipError_t mcpet_launch_scale_by_max(float* a, int n, unsigned* mx, hipStream_t stream)
{
  hipError_t e = hipMemsetAsync(mx, 0, sizeof(unsigned), stream);
  if (e != hipSuccess) return e;
  const int nb = n < 1 ? 1 : (n + 255) / 256 > 256 ? 256 : (n + 255) / 256;
  hipLaunchKernelGGL(k_max_bits, dim3(nb), dim3(256), 0, stream, a, n, mx);
  hipLaunchKernelGGL(k_scale_by, dim3(nb), dim3(256), 0, stream, a, n, mx);
  return hipGetLastError();
}

hipError_t mcpet_launch_fill_regions(void* const* p, const size_t* n_words, int n, hipStream_t stream)
{
  for (int i0 = 0; i0 < n; i0 += K_FILL_MAX) {
    FillRegions r{};
    const int m = std::min(K_FILL_MAX, n - i0);
    size_t most = 0;
    for (int k = 0; k < m; k++) {
      r.p[k] = (unsigned*)p[i0 + k];
      r.n[k] = n_words[i0 + k];
      most = std::max(most, n_words[i0 + k]);
    }
    if (most == 0) continue;
    const unsigned bx = (unsigned)std::min<size_t>(2048, (most / 4 + 255) / 256 + 1);
    hipLaunchKernelGGL(k_fill_regions, dim3(bx, m), dim3(256), 0, stream, r);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t mcpet_launch_fill_u32(void* p, size_t n_words, hipStream_t stream)
{
  if (n_words == 0) return hipSuccess;
  const size_t per = 256 * 16;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n_words + per - 1) / per)), dim3(256), 0, stream, (unsigned*)p, n_words);
  return hipGetLastError();
}

hipError_t mcpet_launch_selftest_ranecu(int seed, const long long* d_ids, int nstreams, int n, float* d_out, double* d_out_d,
                                        int as_double, const uint32_t* j1, const uint32_t* j2, hipStream_t stream)
{
  int blocks = (nstreams + 255) / 256;
  hipLaunchKernelGGL(k_selftest_ranecu, dim3(blocks), dim3(256), 0, stream, seed, d_ids, nstreams, n, d_out, d_out_d, as_double,
                     j1, j2);
  return hipGetLastError();
}

template <int FN>
static hipError_t launch_selftest_fastmath(int fn, unsigned long long first, unsigned long long n, unsigned long long* d_res, hipStream_t stream)
{
  if constexpr (FN < FF_N) {
    if (fn != FN) return launch_selftest_fastmath<FN + 1>(fn, first, n, d_res, stream);
    const unsigned blocks = (unsigned)std::min<unsigned long long>(8192, (n + 255) / 256);
    hipLaunchKernelGGL(k_selftest_fastmath<FN>, dim3(blocks), dim3(256), 0, stream, first, n, d_res);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
hipError_t mcpet_launch_selftest_fastmath(int fn, unsigned long long first, unsigned long long n, unsigned long long* d_res, hipStream_t stream)
{
  return launch_selftest_fastmath<0>(fn, first, n, d_res, stream);
}

hipError_t mcpet_launch_selftest_fmath(const double* d_x, const double* d_y, int n, double* d_od, float* d_of, hipStream_t stream)
{
  hipLaunchKernelGGL(k_selftest_fmath, dim3((n + 255) / 256), dim3(256), 0, stream, d_x, d_y, n, d_od, d_of);
  return hipGetLastError();
}

hipError_t mcpet_launch_copy(const uint4* src, uint4* dst, size_t n16, hipStream_t stream)
{
  hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, stream, src, dst, n16);
  return hipGetLastError();
}
