// mcd_step.h — what the transport kernels share: LDS staging of a
// configuration's tables, the DS energy loss and polar angle of a step, record
// and scatter-row output, counter reductions.
#pragma once

#include <hip/hip_runtime.h>

#include "mcd_device.h"
#include "mcd_internal.h"

namespace mcd {

// Kernel arguments read anew where a rare path uses them.  The compiler cannot
// tell these loads from others, so it neither hoists what the path computes
// from them out of a loop nor keeps their values for it: in the inline-guard
// kernel the FP64 pick's constants took 40 SGPRs and VGPRs of every step.
template <class T>
using Const4 = const __attribute__((address_space(4))) T;
// The arguments of a kernel that takes (DevCfg, RunArgs, ..).
struct KernelArgs {
  DevCfg c;
  RunArgs R;
};
__device__ __forceinline__ const KernelArgs& args_anew() {
  Const4<KernelArgs>* p = (Const4<KernelArgs>*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return (const KernelArgs&)*p;
}
// The same for an object in the constant address space (a batch item's).
template <class T>
__device__ __forceinline__ const T& anew(const T& x) {
  Const4<T>* p = (Const4<T>*)&x;
  asm volatile("" : "+s"(p));
  return (const T&)*p;
}

// LDS of the one-configuration kernels: the pick table (nf floats), then the
// two loss-table descriptors at a 16-byte aligned offset.
__host__ __device__ constexpr int tab_offset_floats(int nf) { return (nf + 3) & ~3; }
inline size_t single_lds_bytes(const DevCfg& c) {
  return (size_t)tab_offset_floats(c.pick.n_nodes * c.pick.stride) * sizeof(float) + 2 * sizeof(DevTable);
}

// Stage the pick table and the two loss-table descriptors (Moller,
// Gryzinski) that a lane selects by its channel.
__device__ __forceinline__ DevTable* stage_single(const DevCfg& c, float* lds) {
  const int nf = c.pick.n_nodes * c.pick.stride;
  for (int i = threadIdx.x; i < nf; i += blockDim.x) lds[i] = c.pick.nodes[i];
  DevTable* tabs = reinterpret_cast<DevTable*>(lds + tab_offset_floats(nf));
  if (threadIdx.x == 0) {
    tabs[0] = c.tm;
    tabs[1] = c.tg;
  }
  return tabs;
}

// An LDS copy of the pick table in the wide record
// (pick_stride_wide): each node's record, then its differences to the next
// node, each the same float subtraction the compact record's interpolation
// does at every step, so the interpolated values are the same bit for bit.
template <int NCH>
__device__ __forceinline__ DevTable* stage_single_wide(const DevCfg& c, float* lds) {
  constexpr int S = pick_stride(NCH), SW = pick_stride_wide(NCH), NB = NCH - 1, D = NB + 3;
  const int n = c.pick.n_nodes;
  const float* __restrict__ g = c.pick.nodes;
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const float* a = g + (size_t)k * S;
    float* o = lds + (size_t)k * SW;
    for (int i = 0; i < D; ++i) o[i] = a[i];
    for (int i = 0; i <= NB; ++i) o[D + i] = k + 1 < n ? a[S + i] - a[i] : 0.f;
  }
  DevTable* tabs = reinterpret_cast<DevTable*>(lds + tab_offset_floats(n * SW));
  if (threadIdx.x == 0) {
    tabs[0] = c.tm;
    tabs[1] = c.tg;
  }
  return tabs;
}

// The record is written once, when the trajectory ends, as nine dword
// stores marked non-temporal: records of one wavefront land in different
// cache lines at different times, and streaming them past L2 keeps them from
// evicting the loss tables and from being read back to merge partial lines.
__device__ __forceinline__ void write_rec(mcd_electron_rec* rec, float E, const float* d, const float* p, uint32_t nsc,
                                          int o1, int o2, uint32_t flags) {
  uint32_t* w = reinterpret_cast<uint32_t*>(rec);
  __builtin_nontemporal_store(__float_as_uint(E), w + 0);
  __builtin_nontemporal_store(__float_as_uint(d[0]), w + 1);
  __builtin_nontemporal_store(__float_as_uint(d[1]), w + 2);
  __builtin_nontemporal_store(__float_as_uint(d[2]), w + 3);
  __builtin_nontemporal_store(__float_as_uint(p[0]), w + 4);
  __builtin_nontemporal_store(__float_as_uint(p[1]), w + 5);
  __builtin_nontemporal_store(__float_as_uint(p[2]), w + 6);
  __builtin_nontemporal_store(nsc, w + 7);
  // outcome, outcome2, flags, pad (bytes 32..35, little endian)
  __builtin_nontemporal_store((uint32_t)(o1 & 0xFF) | ((uint32_t)(o2 & 0xFF) << 8) | ((flags & 0xFFu) << 16), w + 8);
}

// wave-level append of scatter rows; returns the slot or ~0 when full
__device__ __forceinline__ uint64_t append_slot(bool want, unsigned long long* cursor, uint64_t cap, int lane) {
  uint64_t m = __ballot(want);
  if (!m) return ~0ull;
  int leader = __ffsll((unsigned long long)m) - 1;
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(cursor, (unsigned long long)__popcll(m));
  base = lane_u64(base, leader);
  uint64_t slot = base + __popcll(m & ((1ull << lane) - 1ull));
  return (want && slot < cap) ? slot : ~0ull;
}

__device__ __forceinline__ void wave_add_counters(unsigned long long* cnt, const uint64_t* v, int nv, int lane) {
  for (int i = 0; i < nv; ++i) {
    uint64_t x = v[i];
    for (int off = 32; off > 0; off >>= 1) {
      uint32_t lo = __shfl_xor((uint32_t)x, off), hi = __shfl_xor((uint32_t)(x >> 32), off);
      x += ((uint64_t)hi << 32) | lo;
    }
    if (lane == 0 && x) atomicAdd(&cnt[i], (unsigned long long)x);
  }
}

// The channel order d_pick_ordered expects: a crossing cell's swap was
// applied to pe.perm by the interpolation; undo it so the FP64 pick sees node
// k's order and decides the pair exactly.
template <int NCH>
__device__ __forceinline__ void guard_perm(const PickEval<NCH>& pe, uint32_t& plo, uint32_t& phi) {
  plo = pe.perm_lo;
  phi = pe.perm_hi;
  if (pe.swap != (int)kMetaNoSwap && pe.pB > pe.pA) {
    uint64_t pm = ((uint64_t)phi << 32) | plo;
    const uint64_t la = (pm >> (4 * pe.swap)) & 15u, lb = (pm >> (4 * (pe.swap + 1))) & 15u;
    pm &= ~((uint64_t)0xFFu << (4 * pe.swap));
    pm |= (lb << (4 * pe.swap)) | (la << (4 * (pe.swap + 1)));
    plo = (uint32_t)pm;
    phi = (uint32_t)(pm >> 32);
  }
}

// Energy loss (Wh + Wl, Wl only for the plasmon) and polar angle (c2 =
// cos^2(theta/2), s2 = sin^2(theta/2)) of a DS step on channel ch; flags
// raised by the step are added to sflags.  tabs: the two loss-table
// descriptors (Moller, Gryzinski) in LDS.
__device__ __forceinline__ void ds_loss_angles(const DevCfg& c, const DevTable* __restrict__ tabs, F2 E, int ch,
                                               float u2, float& Wh, float& Wl, float& c2, float& s2,
                                               uint32_t& sflags) {
  // 1/E for both the screening parameter and the loss fraction: one
  // reciprocal for the wavefront instead of one in each channel branch
  const float rE = __builtin_amdgcn_rcpf(E.hi);
  Wl = 0.f;
  if (ch == MCD_CH_RUTH) {  // Rutherford_halfPol, scattering.py:125-152
    Wh = 0.f;
    const float a = c.c_alpha_f * rE;
    const float om = 1.f - u2;
    const float inv = __builtin_amdgcn_rcpf(om + a);
    s2 = a * u2 * inv;
    c2 = om * (1.f + a) * inv;
  } else if (ch == MCD_CH_QUINN) {  // scattering.py:643-656
    Wh = c.Epl_hi; Wl = c.Epl_lo;
    c2 = 1.f; s2 = 0.f;
  } else {  // Moller table, or the outer-shell Gryzinski table for all shells (:602-640)
    const DevTable& t = tabs[ch == MCD_CH_MOLLER ? 0 : 1];  // LDS: no per-lane kernel-argument loads
    const F2 Ec = E;
    int row;
    const int col = table_lookup(t, E.hi, [Ec](float v) { return f_lt_f2(v, Ec); }, u2, row);
    Wh = ldg(t.Ws + col);
    if (!f_lt_f2(Wh, E)) sflags |= MCD_FLAG_LOSS_GE_E;
    // binaryCollModel (:156-179): W <= (E - E_F)/2
    const F2 D = f2_sub(E, c.Ef2_hi, c.Ef2_lo);
    const float w2 = 2.f * Wh;
    const bool ok = !(D.hi < w2 || (D.hi == w2 && D.lo < 0.f));
    if (ok) {
      const float x = Wh * rE;
      const float sq = __builtin_amdgcn_sqrtf(1.f - x);
      c2 = 0.5f * (1.f + sq);
      s2 = 0.5f * x * __builtin_amdgcn_rcpf(1.f + sq);
    } else {
      c2 = s2 = __builtin_nanf("");
      sflags |= MCD_FLAG_NAN_DIR;
    }
  }
}

// Free path l, loss Wh + Wl and Joy's screening parameter a (the polar angle's)
// of a continuous-mode step; ln_u0 = ln of the path's random number.  EXPL:
// the explicit Bethe law, evaluated in FP64.  NIGRAM: the screening, where the
// caller has branched on it.
enum { kScreenAny = -1 };
template <bool EXPL, int NIGRAM = kScreenAny>
__device__ __forceinline__ void cont_path_loss(const DevCfg& c, F2 E, float ln_u0, float& a, float& l, float& Wh,
                                               float& Wl, uint32_t& sflags) {
  Wl = 0.f;
  // Rutherford-only mean free path (scattering.py:780-797)
  // Joy's screening: the polar angle (Rutherford_halfPol) in every model
  a = c.c_alpha_f * __builtin_amdgcn_rcpf(E.hi);
  float sig;
  if (NIGRAM == kScreenAny ? c.elastic >= MCD_ELASTIC_NIGRAM : NIGRAM) {  // ruther_N_sigma(_wDefl), crossSections.py:91-147
    const float b = 0.48f * (c.nig_zp_f * __builtin_amdgcn_rcpf(E.hi));
    sig = c.nig_num_f * __builtin_amdgcn_rcpf(4.f * b * (1.f + b) * (E.hi * E.hi));
  } else {
    const float Ek = E.hi * 1e-3f;
    const float rr = (Ek + 511.f) * __builtin_amdgcn_rcpf(Ek + 1024.f);
    sig = c.ruth_k_f * rr * rr * __builtin_amdgcn_rcpf(Ek * Ek * a * (1.f + a));
  }
  const float mfp = c.mfp_k_f * __builtin_amdgcn_rcpf(sig);
  l = -mfp * ln_u0;
  if (!(l < 1e4f)) sflags |= MCD_FLAG_LONG_PATH;
  // Bethe stopping power at the pre-step energy (stoppingPowers.py:112-215)
  if constexpr (EXPL) {
    // explicit law (:177-215), its shell sum folded to Z_eff (ln E - ln E*),
    // in FP64: near Emin ln E and ln E* are close, and their FP32
    // difference would lose most of its bits; the loss l*S is kept as a pair
    const double Ed = (double)E.hi + (double)E.lo;
    const double Wd = (double)l * (c.expl_k * (log(Ed) - c.lnEstar) / Ed);
    Wh = (float)Wd;
    Wl = (float)(Wd - (double)Wh);
  } else {
    float S;
    const float iE = __builtin_amdgcn_rcpf(E.hi);
    if (c.bethe == MCD_BETHE_CLASSICAL) S = c.bethe_k1_f * iE * ln_f(c.bethe_c1_f * E.hi);
    else S = c.bethe_k1_f * iE * ln_f(c.bethe_c1_f * (E.hi + c.bethe_kJ_f));
    Wh = l * S;
  }
  if (!f_lt_f2(Wh, E)) sflags |= MCD_FLAG_LOSS_GE_E;
}

// FP64 step: every quantity in double and the exact pick.  Arithmetic is not
// contracted into FMAs so the operation order matches the reference expressions.
struct DStep {
  double l, W, c2, hp;
  int ch;
  uint32_t sflags;
};

#pragma clang fp contract(off)
// One step's physics in FP64; tm, tg: the two loss tables (NCH channels, DS).
template <int MODE, int NCH>
__device__ __forceinline__ DStep d_step_physics(const DevCfg& c, const DevTable& tm, const DevTable& tg, double E,
                                                const U4 r) {
  DStep o;
  o.sflags = 0;
  o.ch = MCD_CH_RUTH;
  if (MODE == MCD_MODE_DS) {
    const double u0 = u01d(r.x), u1 = u01d(r.y), u2 = u01d(r.z), u3 = u01d(r.w);
    double mfp;
    o.ch = d_pick<NCH>(E, u0, c, &mfp);          // det_type, scattering.py:530-549
    o.l = -mfp * log(u1);                   // compute_pathl, :551-565
    if (o.ch == MCD_CH_RUTH) {              // :575-586
      o.W = 0.;
      const double a = c.c_alpha / E;
      o.c2 = 1. - (a * u2 / (1. + a - u2));
    } else if (o.ch == MCD_CH_QUINN) {      // :643-656
      o.W = c.Epl;
      o.c2 = 1.;
    } else {                                // :602-640
      const DevTable& t = (o.ch == MCD_CH_MOLLER) ? tm : tg;
      const double Ec = E;
      int row;
      const int col = table_lookup(t, (float)E, [Ec](float v) { return (double)v < Ec; }, (float)u2, row);
      o.W = (double)ldg(t.Ws + col);
      if (!(o.W < E)) o.sflags |= MCD_FLAG_LOSS_GE_E;
      if (o.W <= (E - c.Ef) * 0.5) o.c2 = 0.5 * (sqrt(1 - (o.W / E)) + 1);
      else { o.c2 = __builtin_nan(""); o.sflags |= MCD_FLAG_NAN_DIR; }
    }
    o.hp = kPi * u3;
  } else {
    const double u0 = u01d(r.x), u1 = u01d(r.y), u2 = u01d(r.z);
    const double sr = d_sigma_ruth(E, c);
    const double mfp = 1. / (c.atnd * sr) * 1e14;  // scattering.py:792
    o.l = -mfp * log(u0);                          // :802-813
    if (!(o.l < 1e4)) o.sflags |= MCD_FLAG_LONG_PATH;
    double S;                                      // stoppingPowers.py:112-215
    if (c.bethe == MCD_BETHE_CLASSICAL) S = 2. * kPiEFour * c.atnd * ((double)c.Z / E) * log(1.166 * (E) / c.J) * 1e-14;
    else if (c.bethe == MCD_BETHE_JL)
      S = 2. * kPiEFour * c.atnd * ((double)c.Z / E) * log(1.166 * (E + c.bethe_kk * c.J) / c.J) * 1e-14;
    else {
      const double pref = (2. * kPiEFour * c.atnd / E) * 1e-14;
      double sumi = c.n_val * log(E * 1. / c.E_val);
      for (int i = 0; i < c.n_shells; ++i) sumi = sumi + c.ns[i] * log(E * 1. / c.Eb[i]);
      S = pref * sumi;
    }
    o.W = o.l * S;                                 // compute_Eloss, :815-826
    if (!(o.W < E)) o.sflags |= MCD_FLAG_LOSS_GE_E;
    const double a = c.c_alpha / E;                // compute_sAngles, :828-840
    o.c2 = 1. - (a * u1 / (1. + a - u1));
    o.hp = kPi * u2;
  }
  return o;
}

__device__ __forceinline__ void d_advance(const double* p, double l, const double* d, double* np_) {
  for (int i = 0; i < 3; ++i) np_[i] = p[i] + l * d[i];
}
#pragma clang fp contract(on)

// ---------------------------------------------------------------------------
// Service guard (DS, FP32, one kernel).  Wavefront 0 of a workgroup is a
// service wavefront: a transport wavefront posts the guard-band picks of a step
// to its LDS mailbox and waits; the service wavefront settles them in FP64, one
// of its lanes per posted lane, and posts the channels back.  The FP64 code is
// on a path no transport wavefront executes, so the kernel keeps the register
// budget of an FP64-free step without a second kernel or a park buffer.
struct GuardSlot {
  float Ehi, Elo, u;
  uint32_t perm_lo, perm_hi;
  int meta;  // posted: swap position | exact << 8; replied: the channel
};
struct GuardBox {
  unsigned long long mask;  // posted lanes
  uint32_t state;           // kBoxPosted, then kBoxReplied
  uint32_t bit;             // this mailbox's bit in the workgroup's pending word
  GuardSlot lane[64];
};
constexpr uint32_t kBoxPosted = 1u, kBoxReplied = 2u;
// A transport wavefront waits at most R.guard_spins s_sleep(2) polls for a
// reply (kGuardSpinCap by default); past it the step takes the Rutherford
// channel and is flagged MCD_FLAG_GUARD_TIMEOUT (counted as an error).

__device__ __forceinline__ uint32_t box_load(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void box_store(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Post the picks with ch < 0 and wait for the channels (called by the active
// lanes of a wavefront together).  sflags tells how a lane's pick was settled.
template <int NCH>
__device__ __forceinline__ void served_pick(GuardBox* box, uint32_t* pending, uint32_t max_spins, F2 E, float u0,
                                            const PickEval<NCH>& pe, int& ch, uint32_t& sflags) {
  const int lane = threadIdx.x & 63;
  if (ch < 0) {
    GuardSlot& g = box->lane[lane];
    uint32_t plo, phi;
    guard_perm<NCH>(pe, plo, phi);
    g.Ehi = E.hi; g.Elo = E.lo; g.u = u0;
    g.perm_lo = plo; g.perm_hi = phi;
    g.meta = (pe.swap & 0xFF) | (pe.exact ? 0x100 : 0);
  }
  const uint64_t m = __ballot(ch < 0);
  const int leader = __ffsll((unsigned long long)__ballot(true)) - 1;
  if (lane == leader) {
    box->mask = m;
    box_store(&box->state, kBoxPosted);
    __hip_atomic_fetch_or(pending, box->bit, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  uint32_t spins = 0;
  while (box_load(&box->state) != kBoxReplied && ++spins < max_spins) __builtin_amdgcn_s_sleep(2);
  if (ch < 0) {
    ch = spins < max_spins ? box->lane[lane].meta : MCD_CH_RUTH;
    sflags |= spins < max_spins ? MCD_FLAG_FP64_PICK : MCD_FLAG_GUARD_TIMEOUT;
  }
}

}  // namespace mcd
