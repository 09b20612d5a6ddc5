// mcd_window.h — transport with several lanes per electron (device code).
//
// A launch of few electrons cannot fill the chip with one electron per lane;
// it takes the longest trajectory (10^3 steps) times the latency of a step on
// a lone wavefront (FP32 1.1 to 1.4 us, 2.9 us with 11 channels: ~400
// instructions issued one after the other, two LDS and three L2 round trips;
// FP64 18 us).  Here G lanes (4 to 64) share an electron and take a window of
// its next G steps at a time:
//   1. Random words: lane j draws step s+j's Philox words and everything that
//      depends on them alone (path-length logarithm, azimuth).
//   2. Energy chain: channel, loss and angle of a step depend on the energy at
//      its start and on its random words, not on position or direction.
//      DS: every lane evaluates its step at a guessed energy, first the
//      window's start energy; the losses found give each lane the energy the
//      chain of subtractions leads to; the steps are evaluated again there.  A
//      step whose loss did not change was evaluated at its exact energy, so the
//      window is final when no loss changes (two evaluations as a rule, 2.2 on
//      average: a channel or table column seldom changes over the few hundred
//      eV of a window).  The energies are the same subtractions in the same
//      order as one step after the other gives.
//      Continuous mode: every loss depends on the energy, so the chain runs
//      step after step, without anything that does not feed it.
//   3. Geometry: path, position, exit test and rotation step after step, all
//      electrons of the wavefront at once, the three components of each vector
//      in three lanes of a quad.  Steps past the electron's end are dropped.
// Every formula is the one of transport_loop and k_transport_f64, so records,
// scatter rows and counters are the same bit for bit.
// Cycles of a 64-lane window (Cu 20 keV, FP32; clock readings in a copy of the
// kernel, a few electrons): random words 660, energy chain 9900, geometry 14100 (220 a step), the rest 1150; 64 steps of one lane on its
// own take 160000.
#pragma once

#include <hip/hip_runtime.h>

#include "mcd_device.h"
#include "mcd_internal.h"
#include "mcd_step.h"

namespace mcd {

// Lane of a quad permutation (sel: source lane of quad lanes 0..3).
template <int S0, int S1, int S2, int S3>
__device__ __forceinline__ float quad_perm(float x) {
  constexpr int ctrl = S0 | (S1 << 2) | (S2 << 4) | (S3 << 6);
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), ctrl, 0xF, 0xF, true));
}
template <int S0, int S1, int S2, int S3>
__device__ __forceinline__ double quad_perm(double x) {
  constexpr int ctrl = S0 | (S1 << 2) | (S2 << 4) | (S3 << 6);
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), ctrl, 0xF, 0xF, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(x), ctrl, 0xF, 0xF, true));
}
// The value of quad lane I in every lane of the quad.
template <int I, class T>
__device__ __forceinline__ T quad_lane(T x) {
  return quad_perm<I, I, I, I>(x);
}
// The value of the lane before, within a row of 16 lanes.
__device__ __forceinline__ float row_prev(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x111, 0xF, 0xF, true));
}
__device__ __forceinline__ double row_prev(double x) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), 0x111, 0xF, 0xF, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(x), 0x111, 0xF, 0xF, true));
}
__device__ __forceinline__ F2 row_prev(F2 x) { return {row_prev(x.hi), row_prev(x.lo)}; }
// The value of a lane, the same lane for the whole wavefront.
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}
__device__ __forceinline__ double lane_value(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}
__device__ __forceinline__ F2 lane_value(F2 x, int lane) { return {lane_value(x.hi, lane), lane_value(x.lo, lane)}; }
// The value of any lane.
__device__ __forceinline__ uint64_t shfl_any(uint64_t v, int src) {
  const uint32_t lo = __shfl((uint32_t)v, src), hi = __shfl((uint32_t)(v >> 32), src);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint32_t shfl_any(uint32_t v, int src) { return __shfl(v, src); }
__device__ __forceinline__ float shfl_any(float v, int src) { return __shfl(v, src); }
__device__ __forceinline__ double shfl_any(double v, int src) { return __shfl(v, src); }
__device__ __forceinline__ F2 shfl_any(F2 v, int src) { return {__shfl(v.hi, src), __shfl(v.lo, src)}; }
__device__ __forceinline__ F2 select(bool c, F2 a, F2 b) { return {c ? a.hi : b.hi, c ? a.lo : b.lo}; }
__device__ __forceinline__ double select(bool c, double a, double b) { return c ? a : b; }

// A window's place in the wavefront: group of G = 2^lg lanes from lane base on,
// lane j of it; gmask: G ones.
struct Group {
  int lg, G, lane, j, base;
  uint64_t gmask;
  __device__ __forceinline__ Group(int lg_, int lane_)
      : lg(lg_), G(1 << lg_), lane(lane_), j(lane_ & ((1 << lg_) - 1)), base(lane_ & ~((1 << lg_) - 1)),
        gmask(lg_ == 6 ? ~0ull : (1ull << (1 << lg_)) - 1ull) {}
  // bits of the group's lanes
  __device__ __forceinline__ uint64_t ballot(bool b) const { return (__ballot(b) >> base) & gmask; }
};

// Energies at the start of each step of the window: lane j of a group gets
// E0 - W_0 - .. - W_(j-1) (E0 and the losses: the group's), one subtraction
// after the other.  P::Energy is a float pair or a double.
template <class P>
__device__ __forceinline__ typename P::Energy chain_energies(typename P::Energy E0, typename P::Energy W,
                                                             const Group& g) {
  typename P::Energy cur = E0;
  if (g.lg <= 4) {
    // lane by lane within the row: after t rounds lanes up to t are final
    const typename P::Energy prev = row_prev(W);
    for (int t = 1; t < g.G; ++t) cur = select(g.j != 0, P::minus(row_prev(cur), prev), E0);
    return cur;
  }
  // one or two electrons per wavefront: only the steps that lose energy (the
  // subtraction of zero leaves an energy as it is)
  uint64_t m = __ballot(P::any(W));
  if (g.lg == 5) m = (m | (m >> 32)) & 0xFFFFFFFFull;
  while (m) {
    const int k = __builtin_ctzll(m);
    m &= m - 1ull;
    typename P::Energy w = lane_value(W, k);
    if (g.lg == 5) w = select(g.lane >= 32, lane_value(W, k + 32), w);
    cur = select(g.j > k, P::minus(cur, w), cur);
  }
  return cur;
}

// DS: evaluate the window's steps until every one has seen its exact energy.
// todo: this lane's step is one of the window's.
template <class P>
__device__ __forceinline__ void ds_energies(const DevCfg& c, const float* __restrict__ lds,
                                            const DevTable* __restrict__ tabs, typename P::Energy E0,
                                            const typename P::Draw& r, bool todo, const Group& g,
                                            typename P::Energy& Ej, typename P::Step& s) {
  Ej = E0;
  while (true) {
    const typename P::Energy old = s.W;
    if (todo && !P::absorbed(Ej, c)) P::step(c, lds, tabs, Ej, r, s);
    // the first step of the group whose loss is not the one its energies were
    // formed with: it and the steps before it are final
    const uint64_t changed = g.ballot(todo && P::differ(s.W, old));
    todo = todo && changed != 0ull && g.j > __builtin_ctzll(changed | (1ull << 63));
    if (!__any(todo)) break;
    const typename P::Energy Ec = chain_energies<P>(E0, s.W, g);
    Ej = select(todo, Ec, Ej);
  }
}

// ---------------------------------------------------------------------------
// FP32, energies as float pairs.  A staged step: path, cos and sin of the polar
// angle, cos and |sin| of the azimuth.
struct Fp32Base {
  static constexpr int kWaves = 2;  // wavefronts per SIMD of k_window, at least
  typedef float Real;
  typedef F2 Energy;
  struct alignas(8) Staged {
    float l, ct, st, cp, sp, pad;
  };
  struct Step {
    float l, c2, s2;
    F2 W;
    int ch;
    uint32_t flags;
  };
  static __device__ __forceinline__ Step no_step() { return {0.f, 1.f, 0.f, {0.f, 0.f}, MCD_CH_RUTH, 0u}; }
  static __device__ __forceinline__ F2 start(const DevCfg& c) { return {c.E0_hi, c.E0_lo}; }
  static __device__ __forceinline__ float dir0(const DevCfg& c, int i) {
    return i == 0 ? c.dir0_f[0] : (i == 1 ? c.dir0_f[1] : c.dir0_f[2]);
  }
  static __device__ __forceinline__ float thickness(const DevCfg& c) { return c.thickness_f; }
  static __device__ __forceinline__ F2 minus(F2 a, F2 b) { return f2_sub(a, b.hi, b.lo); }
  static __device__ __forceinline__ bool any(F2 w) { return w.hi != 0.f; }
  static __device__ __forceinline__ bool differ(F2 a, F2 b) { return a.hi != b.hi || a.lo != b.lo; }
  static __device__ __forceinline__ bool absorbed(F2 e, const DevCfg& c) { return f2_le(e, c.Emin_hi, c.Emin_lo); }
  static __device__ __forceinline__ float value(F2 e) { return e.hi; }
  static __device__ __forceinline__ float loss(F2 w) { return w.hi + w.lo; }
  static __device__ __forceinline__ void stage(Staged& w, const Step& s, float u_az) {
    float cp, sp;
    cos_abs_sin_2pi(u_az, cp, sp);
    w.l = s.l;
    w.ct = s.c2 - s.s2;
    w.st = 2.f * __builtin_amdgcn_sqrtf(s.c2 * s.s2);
    w.cp = cp;
    w.sp = sp;
  }
  // Kahan-compensated flight: position t and compensation npc after it
  static __device__ __forceinline__ void fly(const Staged& w, float p, float pc, float d, float& t, float& npc) {
    const float v = w.l * d - pc;
    t = p + v;
    npc = (t - p) - v;
  }
  // f_rotate on vectors spread over a quad: the same products and sums per
  // component, the two norms from all three components
  static __device__ __forceinline__ void rotate(const Staged& r, int, float& d, float& y) {
    const float ct = r.ct, st = r.st, cp = r.cp, sp = r.sp;
    const float y1 = quad_perm<1, 2, 0, 1>(y), y2 = quad_perm<2, 0, 1, 2>(y);
    const float d1 = quad_perm<1, 2, 0, 1>(d), d2 = quad_perm<2, 0, 1, 2>(d);
    const float w = y1 * d2 - y2 * d1;
    const float nd = ct * d + st * (cp * w + sp * y);
    const float ny = cp * y - sp * w;
    const float nd0 = quad_lane<0>(nd), nd1 = quad_lane<1>(nd), nd2 = quad_lane<2>(nd);
    const float ny0 = quad_lane<0>(ny), ny1 = quad_lane<1>(ny), ny2 = quad_lane<2>(ny);
    d = nd * __builtin_amdgcn_rsqf(nd0 * nd0 + nd1 * nd1 + nd2 * nd2);
    y = ny * __builtin_amdgcn_rsqf(ny0 * ny0 + ny1 * ny1 + ny2 * ny2);
  }
};

template <int NCH>
struct Fp32Ds : Fp32Base {
  static constexpr bool kPickTable = true;
  static constexpr bool kServed = false;
  static constexpr int kTurns = 1;
  struct Draw {
    float u0, lg1, u2, az;
  };
  static __device__ __forceinline__ Draw draw(const U4 r) {
    return {u01f(r.x), log2_f(u01f(r.y)), u01f(r.z), u01f(r.w)};
  }
  static __device__ __forceinline__ float half_azimuth(const Draw& r) { return kPiF * r.az; }
  static __device__ __forceinline__ void stage(Staged& w, const Step& s, const Draw& r) {
    Fp32Base::stage(w, s, r.az);
  }
  static __device__ __forceinline__ void step(const DevCfg& c, const float* __restrict__ lds,
                                              const DevTable* __restrict__ tabs, F2 E, const Draw& r, Step& s) {
    step_of<false>(c, lds, tabs, E, r, s);
  }
  // ITEM: as in transport_loop
  template <bool ITEM>
  static __device__ __forceinline__ void step_of(const DevCfg& c, const float* __restrict__ lds,
                                                 const DevTable* __restrict__ tabs, F2 E, const Draw& r, Step& s) {
    float mfp_ln2;
    PickEval<NCH> pe;
    s.flags = 0;
    s.ch = f_pick_table<NCH>(lds, c.pick, E.hi, r.u0, mfp_ln2, pe);
    if (s.ch < 0) {  // guard band: settle the pick in FP64
      uint32_t plo, phi;
      guard_perm<NCH>(pe, plo, phi);
      const DevCfg& ca = ITEM ? anew(c) : args_anew().c;
      s.ch = d_pick_ordered<NCH>((double)E.hi + (double)E.lo, (double)r.u0, ca, plo, phi, pe.swap, pe.exact);
      s.flags |= MCD_FLAG_FP64_PICK;
    }
    s.l = -mfp_ln2 * r.lg1;
    ds_loss_angles(c, tabs, E, s.ch, r.u2, s.W.hi, s.W.lo, s.c2, s.s2, s.flags);
  }
  static __device__ __forceinline__ void energies(const DevCfg& c, const float* __restrict__ lds,
                                                  const DevTable* __restrict__ tabs, Staged*, F2 E0,
                                                  const Draw (&r)[1], const bool (&todo)[1], const Group& g, int,
                                                  F2 (&Ej)[1], Step (&s)[1]) {
    ds_energies<Fp32Ds<NCH>>(c, lds, tabs, E0, r[0], todo[0], g, Ej[0], s[0]);
  }
};

// A batch item's.
template <int NCH>
struct Fp32DsItem : Fp32Ds<NCH> {
  typedef typename Fp32Ds<NCH>::Draw Draw;
  typedef typename Fp32Ds<NCH>::Step Step;
  typedef typename Fp32Ds<NCH>::Staged Staged;
  static __device__ __forceinline__ void step(const DevCfg& c, const float* __restrict__ lds,
                                              const DevTable* __restrict__ tabs, F2 E, const Draw& r, Step& s) {
    Fp32Ds<NCH>::template step_of<true>(c, lds, tabs, E, r, s);
  }
  static __device__ __forceinline__ void energies(const DevCfg& c, const float* __restrict__ lds,
                                                  const DevTable* __restrict__ tabs, Staged*, F2 E0,
                                                  const Draw (&r)[1], const bool (&todo)[1], const Group& g, int,
                                                  F2 (&Ej)[1], Step (&s)[1]) {
    ds_energies<Fp32DsItem<NCH>>(c, lds, tabs, E0, r[0], todo[0], g, Ej[0], s[0]);
  }
};

// In the served-guard kernel: wide pick records, guard picks through the
// wavefront's mailbox (at the start of the workgroup's LDS).
template <int NCH>
struct Fp32DsServed : Fp32Ds<NCH> {
  static constexpr bool kServed = true;
  typedef typename Fp32Ds<NCH>::Draw Draw;
  typedef typename Fp32Ds<NCH>::Step Step;
  typedef typename Fp32Ds<NCH>::Staged Staged;
  static_assert(sizeof(Staged) == sizeof(GuardSlot), "a window takes the place of a mailbox's slots");
  static __device__ __forceinline__ void step(const DevCfg& c, const float* __restrict__ lds,
                                              const DevTable* __restrict__ tabs, F2 E, const Draw& r, Step& s) {
    float mfp_ln2;
    PickEval<NCH> pe;
    s.flags = 0;
    s.ch = f_pick_table<NCH, true>(lds, c.pick, E.hi, r.u0, mfp_ln2, pe);
    if (__any(s.ch < 0)) {
      extern __shared__ float lds0[];
      const int n_boxes = (int)(blockDim.x >> 6) - 1;
      GuardBox* boxes = reinterpret_cast<GuardBox*>(lds0);
      served_pick<NCH>(boxes + (__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) - 1),
                       reinterpret_cast<uint32_t*>(boxes + n_boxes) + 1, args_anew().R.guard_spins, E, r.u0, pe, s.ch,
                       s.flags);
    }
    s.l = -mfp_ln2 * r.lg1;
    ds_loss_angles(c, tabs, E, s.ch, r.u2, s.W.hi, s.W.lo, s.c2, s.s2, s.flags);
  }
  static __device__ __forceinline__ void energies(const DevCfg& c, const float* __restrict__ lds,
                                                  const DevTable* __restrict__ tabs, Staged*, F2 E0,
                                                  const Draw (&r)[1], const bool (&todo)[1], const Group& g, int,
                                                  F2 (&Ej)[1], Step (&s)[1]) {
    ds_energies<Fp32DsServed<NCH>>(c, lds, tabs, E0, r[0], todo[0], g, Ej[0], s[0]);
    // the staged steps that follow overwrite the slots the picks were read from
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
};

template <bool EXPL>
struct Fp32Cont : Fp32Base {
  static constexpr bool kPickTable = false;
  static constexpr bool kServed = false;
  static constexpr int kTurns = 4;
  struct Draw {
    float ln0, u1, az;
  };
  static __device__ __forceinline__ Draw draw(const U4 r) { return {ln_f(u01f(r.x)), u01f(r.y), u01f(r.z)}; }
  static __device__ __forceinline__ float half_azimuth(const Draw& r) { return kPiF * r.az; }
  static __device__ __forceinline__ void stage(Staged& w, const Step& s, const Draw& r) {
    Fp32Base::stage(w, s, r.az);
  }
  template <int M, int NIGRAM>
  static __device__ __forceinline__ void chain(const DevCfg& c, const Staged* wp, F2 E0, const Group& g, int turns,
                                               F2 (&Ej)[M]) {
    F2 cur = E0;
    float a, l, ln0 = wp[0].l;
    uint32_t flags = 0;
    int k = 0;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      Ej[i] = cur;
      if (i < turns) {
        for (int kk = 0; kk < g.G; ++kk) {
          Ej[i] = select(g.j == kk, cur, Ej[i]);
          const float next = wp[++k].l;
          F2 W;
          cont_path_loss<EXPL, NIGRAM>(c, cur, ln0, a, l, W.hi, W.lo, flags);
          cur = minus(cur, W);
          ln0 = next;
        }
      }
    }
  }
  // Step after step: all lanes of a group form step k's loss from its staged
  // logarithm, the lane of step k keeps the energy it starts from; then every
  // lane its own steps' paths, losses and angles.
  template <int M>
  static __device__ __forceinline__ void energies(const DevCfg& c, const float* __restrict__,
                                                  const DevTable* __restrict__, Staged* win, F2 E0, const Draw (&r)[M],
                                                  const bool (&todo)[M], const Group& g, int turns, F2 (&Ej)[M],
                                                  Step (&s)[M]) {
    Staged* wp = win + g.base * turns;
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (i < turns) wp[i * g.G + g.j].l = r[i].ln0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // one loop per screening: a branch in it costs six instructions a step
    if (c.elastic >= MCD_ELASTIC_NIGRAM) chain<M, 1>(c, wp, E0, g, turns, Ej);
    else chain<M, 0>(c, wp, E0, g, turns, Ej);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < M; ++i) {
      if (!todo[i]) continue;
      float a;
      s[i].flags = 0;
      cont_path_loss<EXPL>(c, Ej[i], r[i].ln0, a, s[i].l, s[i].W.hi, s[i].W.lo, s[i].flags);
      const float om = 1.f - r[i].u1;
      const float inv = __builtin_amdgcn_rcpf(om + a);
      s[i].s2 = a * r[i].u1 * inv;
      s[i].c2 = om * (1.f + a) * inv;
    }
  }
};

// ---------------------------------------------------------------------------
// FP64 (DS).  A staged step: path and the half angles' cosines and sines.
#pragma clang fp contract(off)
template <int NCH>
struct Fp64Ds {
  // 65000 electrons, us at 2 and 3: Cu, 7 channels 11020 and 9860, Si, 6 channels
  // 4770 and 4560; Au with 11 channels 12500 and, with spills, 12870
  static constexpr int kWaves = NCH <= 7 ? 3 : 2;
  typedef double Real;
  typedef double Energy;
  static constexpr bool kServed = false;
  static constexpr bool kPickTable = false;
  static constexpr int kTurns = 1;
  struct alignas(16) Staged {
    double l, c_ht, s_ht, c_hp, s_hp, pad;
  };
  struct Step {
    double l, c2, W;
    int ch;
    uint32_t flags;
  };
  typedef U4 Draw;
  static __device__ __forceinline__ Step no_step() { return {0., 1., 0., MCD_CH_RUTH, 0u}; }
  static __device__ __forceinline__ double start(const DevCfg& c) { return c.E0; }
  static __device__ __forceinline__ double dir0(const DevCfg& c, int i) {
    return i == 0 ? c.dir0[0] : (i == 1 ? c.dir0[1] : c.dir0[2]);
  }
  static __device__ __forceinline__ double thickness(const DevCfg& c) { return c.thickness; }
  static __device__ __forceinline__ double minus(double a, double b) { return a - b; }
  static __device__ __forceinline__ bool any(double w) { return w != 0.; }
  static __device__ __forceinline__ bool differ(double a, double b) { return a != b; }
  static __device__ __forceinline__ bool absorbed(double e, const DevCfg& c) { return e <= c.Emin; }
  static __device__ __forceinline__ float value(double e) { return (float)e; }
  static __device__ __forceinline__ float loss(double w) { return (float)w; }
  static __device__ __forceinline__ Draw draw(const U4 r) { return r; }
  static __device__ __forceinline__ float half_azimuth(const Draw& r) { return (float)(kPi * u01d(r.w)); }
  static __device__ __forceinline__ void stage(Staged& w, const Step& s, const Draw& r) {
    double c_ht, s_ht, c_hp, s_hp;
    d_half_angles(s.c2, kPi * u01d(r.w), c_ht, s_ht, c_hp, s_hp);
    w.l = s.l;
    w.c_ht = c_ht;
    w.s_ht = s_ht;
    w.c_hp = c_hp;
    w.s_hp = s_hp;
  }
  static __device__ __forceinline__ void step(const DevCfg& c, const float* __restrict__,
                                              const DevTable* __restrict__ tabs, double E, const Draw& r, Step& s) {
    const DStep o = d_step_physics<MCD_MODE_DS, NCH>(c, tabs[0], tabs[1], E, r);
    s.l = o.l;
    s.c2 = o.c2;
    s.W = o.W;
    s.ch = o.ch;
    s.flags = o.sflags | (o.c2 != o.c2 ? MCD_FLAG_NAN_DIR : 0u);
  }
  static __device__ __forceinline__ void energies(const DevCfg& c, const float* __restrict__ lds,
                                                  const DevTable* __restrict__ tabs, Staged*, double E0,
                                                  const Draw (&r)[1], const bool (&todo)[1], const Group& g, int,
                                                  double (&Ej)[1], Step (&s)[1]) {
    ds_energies<Fp64Ds<NCH>>(c, lds, tabs, E0, r[0], todo[0], g, Ej[0], s[0]);
  }
  static __device__ __forceinline__ void fly(const Staged& w, double p, double, double d, double& t, double& npc) {
    t = p + w.l * d;
    npc = 0.;
  }
  // d_rotate: quaternion and |q|^2 in every lane, then each lane the row of the
  // rotation matrix that gives its component (i), summed in index order
  static __device__ __forceinline__ void rotate(const Staged& r, int i, double& d, double& y) {
    const double d0 = quad_lane<0>(d), d1 = quad_lane<1>(d), d2 = quad_lane<2>(d);
    const double y0 = quad_lane<0>(y), y1 = quad_lane<1>(y), y2 = quad_lane<2>(y);
    const double a1 = r.c_hp, b1 = d0 * r.s_hp, c1 = d1 * r.s_hp, e1 = d2 * r.s_hp;
    const double a2 = r.c_ht, b2 = y0 * r.s_ht, c2 = y1 * r.s_ht, e2 = y2 * r.s_ht;
    const double w = a1 * a2 - b1 * b2 - c1 * c2 - e1 * e2;
    const double x = a1 * b2 + b1 * a2 + c1 * e2 - e1 * c2;
    const double v = a1 * c2 - b1 * e2 + c1 * a2 + e1 * b2;
    const double z = a1 * e2 + b1 * c2 - c1 * b2 + e1 * a2;
    const double n = w * w + x * x + v * v + z * z;
    // (x, v, z) turned so that p is component i and q, s the next two
    const double p = i == 0 ? x : (i == 1 ? v : z);
    const double q = i == 0 ? v : (i == 1 ? z : x);
    const double s = i == 0 ? z : (i == 1 ? x : v);
    const double m0 = 1.0 - 2 * (q * q + s * s) / n, m1 = 2 * (p * q - s * w) / n, m2 = 2 * (p * s + q * w) / n;
    const double e0_ = i == 0 ? m0 : (i == 1 ? m2 : m1);
    const double e1_ = i == 0 ? m1 : (i == 1 ? m0 : m2);
    const double e2_ = i == 0 ? m2 : (i == 1 ? m1 : m0);
    const double nd = e0_ * d0 + e1_ * d1 + e2_ * d2;
    const double ny = e0_ * y0 + e1_ * y1 + e2_ * y2;
    const double nd0 = quad_lane<0>(nd), nd1 = quad_lane<1>(nd), nd2 = quad_lane<2>(nd);
    const double ny0 = quad_lane<0>(ny), ny1 = quad_lane<1>(ny), ny2 = quad_lane<2>(ny);
    d = nd / sqrt(nd0 * nd0 + nd1 * nd1 + nd2 * nd2);
    y = ny / sqrt(ny0 * ny0 + ny1 * ny1 + ny2 * ny2);
  }
};
#pragma clang fp contract(on)

// The record of an electron (write_rec), spread over its group's first quad.
__device__ __forceinline__ void write_rec_quad(mcd_electron_rec* rec, int j, float E, float d, float p, uint32_t nsc,
                                               int o1, int o2, uint32_t flags) {
  uint32_t* w = reinterpret_cast<uint32_t*>(rec);
  if (j < 3) {
    __builtin_nontemporal_store(__float_as_uint(d), w + 1 + j);
    __builtin_nontemporal_store(__float_as_uint(p), w + 4 + j);
  }
  if (j == 0) {
    __builtin_nontemporal_store(__float_as_uint(E), w + 0);
    __builtin_nontemporal_store(nsc, w + 7);
    __builtin_nontemporal_store((uint32_t)(o1 & 0xFF) | ((uint32_t)(o2 & 0xFF) << 8) | ((flags & 0xFFu) << 16), w + 8);
  }
}

// Direction and position of one electron, component (lane & 3) of each vector
// (lanes 3 of a quad repeat component 0), and its energy and counters.
template <class P>
struct WinEl {
  typename P::Real p, pc, d, y;
  typename P::Energy E;
  uint64_t e;
  uint32_t ctr1, step, flags;
};

// The start of electron e, component comp of each vector.
template <class P>
__device__ __forceinline__ WinEl<P> win_start(const DevCfg& c, uint64_t e, int comp) {
  WinEl<P> s;
  s.p = s.pc = 0;
  s.d = P::dir0(c, comp);
  s.y = comp == 1 ? 1 : 0;
  s.E = P::start(c);
  s.e = e;
  s.ctr1 = c.config_id | (uint32_t)(e >> 32) << 16;
  s.step = s.flags = 0;
  return s;
}

// A window is G steps; in continuous mode at least 16, up to 4 (kTurns) a lane:
// its chain gains nothing from the lanes, and the work of a window beside its
// steps (1100 cycles) is spread over more of them.
template <class P, bool ROWS>
constexpr int win_turns() { return ROWS ? 1 : P::kTurns; }
__device__ __forceinline__ int win_turns_of(int most, int lg) { return min(most, lg < 4 ? 16 >> lg : 1); }

// LDS: the pick table (kPickTable), the two loss-table descriptors (DS), one
// window of staged steps per wavefront: one a lane and turn, two more for the
// reads ahead.
__host__ __device__ constexpr int win_stage(int turns) { return 64 * turns + 2; }
template <class P>
__host__ __device__ inline size_t win_stage_offset(const DevCfg& c) {
  const int nf = P::kPickTable ? c.pick.n_nodes * c.pick.stride : 0;
  return ((size_t)tab_offset_floats(nf) * sizeof(float) + 2 * sizeof(DevTable) + 15) & ~(size_t)15;
}

// A wavefront's electrons (those of the active lanes, 2^lg lanes each) to their
// end; lg grows as fewer are left.
template <class P, bool ROWS, int M>
__device__ __forceinline__ void window_loop(const DevCfg& c, const RunArgs& R, const float* __restrict__ lds,
                                            const DevTable* __restrict__ tabs, typename P::Staged* win, int lg,
                                            WinEl<P> s, bool active, uint32_t& n_events, uint32_t& n_fp64) {
  typedef typename P::Real Real;
  const int lane = threadIdx.x & 63;
  uint32_t k0 = (uint32_t)R.seed, k1 = (uint32_t)(R.seed >> 32);
  const int comp = (lane & 3) == 3 ? 0 : (lane & 3);

  while (true) {
    // the key words stay loop-carried SGPR values (see transport_loop)
    asm volatile("" : "+s"(k0), "+s"(k1));
    Group g(lg, lane);
    const uint64_t live = __ballot(active && g.j == 0);
    if (!live) break;
    if (lg < 6 && 2 * __popcll(live) * g.G <= 64) {
      // fewer electrons than half the groups: wider groups, longer windows
      const int n = __popcll(live);
      while (lg < 6 && (n << (lg + 1)) <= 64) ++lg;
      g = Group(lg, lane);
      const int mine = lane >> lg;
      int src = 0;
      uint64_t m = live;
      for (int i = 0; i < n; ++i) {
        const int b = __builtin_ctzll(m);
        m &= m - 1ull;
        src = i == mine ? b : src;
      }
      src += lane & 3;
      s.p = shfl_any(s.p, src); s.pc = shfl_any(s.pc, src); s.d = shfl_any(s.d, src); s.y = shfl_any(s.y, src);
      s.E = shfl_any(s.E, src);
      s.e = shfl_any(s.e, src);
      s.ctr1 = shfl_any(s.ctr1, src); s.step = shfl_any(s.step, src); s.flags = shfl_any(s.flags, src);
      active = mine < n;
    }

    const int turns = win_turns_of(M, lg), N = g.G * turns;  // the window's steps

    // steps of the window before maxScatt ends the trajectory ('long')
    const int64_t left = active ? c.max_scatt - (int64_t)s.step : 0;
    if (active && left <= 0) {
      write_rec_quad(&R.els[s.e - R.first], g.j, P::value(s.E), (float)s.d, (float)(s.p - s.pc), s.step, MCD_OUT_LONG, 0,
                     s.flags);
      active = false;
    }
    const int nw = (int)(left < N ? (left > 0 ? left : 0) : N);

    // ---- 1. random words of steps s + j, s + j + G, .. ----
    typename P::Draw r[M];
    bool todo[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int k = g.j + i * g.G;
      todo[i] = active && i < turns && k < nw;
      if (i < turns) r[i] = P::draw(philox10((uint32_t)s.e, s.ctr1, s.step + (uint32_t)k, 0u, k0, k1));
    }

    // ---- 2. energy chain ----
    typename P::Energy Ej[M], Eaft[M];  // at the start and the end of a step
    typename P::Step st[M];
#pragma unroll
    for (int i = 0; i < M; ++i) st[i] = P::no_step();
    P::energies(c, lds, tabs, win, s.E, r, todo, g, turns, Ej, st);
    constexpr int kNever = 1 << 16;
    int ka = kNever;  // the step that absorbs the electron: the window ends with it
    typename P::Staged* wp = win + g.base * turns;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      Eaft[i] = P::minus(Ej[i], st[i].W);
      const uint64_t am = g.ballot(todo[i] && P::absorbed(Eaft[i], c));
      if (am && ka == kNever) ka = i * g.G + __builtin_ctzll(am);
      if (i < turns) P::stage(wp[i * g.G + g.j], st[i], r[i]);
    }
    const int m = ka < nw ? ka + 1 : nw;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // ---- 3. geometry, step after step ----
    const bool rec_row = ROWS && active && s.e < R.row_max_electron;
    const Real thick = P::thickness(c);
    int ran = 0;  // steps executed
    // depth after the last executed step (an exit ends the window); NaN, neither
    // in front nor behind, for a window that passes whole inside the film
    Real tz = (Real)__builtin_nan("");
    bool go = active && m > 0;
    Real rx = 0, ry = 0, rz = 0, rdx = 0, rdy = 0, rdz = 0;  // ROWS: lane j's step
    // selects instead of branches: no lane leaves the loop before the last
    auto advance = [&](const typename P::Staged& w, int k) {
      Real t, npc;
      P::fly(w, s.p, s.pc, s.d, t, npc);
      const Real depth = quad_lane<2>(t);
      if constexpr (ROWS) {
        const Real p0 = quad_lane<0>(s.p), p1 = quad_lane<1>(s.p), p2 = quad_lane<2>(s.p);
        rx = k == g.j ? p0 : rx; ry = k == g.j ? p1 : ry; rz = k == g.j ? p2 : rz;
      }
      const bool stay = go && !(depth <= 0) && !(depth >= thick);
      tz = go ? depth : tz;
      ran += go ? 1 : 0;
      s.pc = stay ? npc : s.pc;
      s.p = stay ? t : s.p;
      Real nd = s.d, ny = s.y;
      P::rotate(w, comp, nd, ny);
      if constexpr (ROWS) {
        const Real d0 = quad_lane<0>(nd), d1 = quad_lane<1>(nd), d2 = quad_lane<2>(nd);
        rdx = k == g.j ? d0 : rdx; rdy = k == g.j ? d1 : rdy; rdz = k == g.j ? d2 : rdz;
      }
      go = stay && k != ka;
      s.d = go ? nd : s.d;
      s.y = go ? ny : s.y;
      go = go && k + 1 < m;
    };
    typename P::Staged wa = wp[0], wb;
    if constexpr (!ROWS) {
      // Most windows run whole, without an exit: every electron through all its
      // steps with no test but the smallest and largest depth; the electrons
      // that end in this window start it again below.
      const Real p_ = s.p, pc_ = s.pc, d_ = s.d, y_ = s.y;
      Real lo = 1, hi = 0;
      auto pass = [&](const typename P::Staged& w) {
        Real t;
        P::fly(w, s.p, s.pc, s.d, t, s.pc);
        s.p = t;
        lo = fmin(lo, t);
        hi = fmax(hi, t);
        P::rotate(w, comp, s.d, s.y);
      };
      for (int k = 0; k < N; k += 2) {  // each step's values are read one step ahead
        wb = wp[k + 1];
        __builtin_amdgcn_sched_barrier(0);
        pass(wa);
        wa = wp[k + 2];
        __builtin_amdgcn_sched_barrier(0);
        pass(wb);
      }
      const bool in = quad_lane<2>(lo) > 0 && quad_lane<2>(hi) < thick;
      if (active && m == N && ka == kNever && in) {
        ran = N;
        go = false;
      } else {
        s.p = p_; s.pc = pc_; s.d = d_; s.y = y_;
        wa = wp[0];
      }
    }
    for (int k = 0; __any(go); k += 2) {
      wb = wp[k + 1];
      advance(wa, k);
      wa = wp[k + 2];
      advance(wb, k + 1);
    }
    int o1 = MCD_OUT_NONE, o2 = MCD_OUT_NONE;
    if (tz <= 0) o1 = MCD_OUT_BKS;
    else if (tz >= thick) o1 = MCD_OUT_TRSM;
    if (ran == ka + 1) {
      if (o1 == MCD_OUT_NONE) o1 = MCD_OUT_ABS; else o2 = MCD_OUT_ABS;
    }
    __builtin_amdgcn_wave_barrier();

    // ---- outputs of the executed steps ----
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const bool mine = active && g.j + i * g.G < ran;
      n_events += mine ? 1u : 0u;
      n_fp64 += mine && (st[i].flags & MCD_FLAG_FP64_PICK) ? 1u : 0u;
      if (__any(mine && st[i].flags)) {
#pragma unroll
        for (uint32_t bit = 1u; bit <= (P::kServed ? 16u : 8u); bit <<= 1)
          if (g.ballot(mine && (st[i].flags & bit))) s.flags |= bit;
        if (P::kServed && mine && (st[i].flags & MCD_FLAG_GUARD_TIMEOUT))
          atomicAdd(R.counters + MCD_CNT_GUARD_TIMEOUTS, 1ull);
      }
    }
    if constexpr (ROWS) {
      const uint64_t slot = append_slot(rec_row && g.j < ran, R.row_cursor, R.row_cap, lane);
      if (slot != ~0ull) {
        mcd_scatter_rec* w = &R.rows[slot];
        const bool last = g.j == ran - 1;
        w->electron = (uint32_t)s.e; w->step = s.step + (uint32_t)g.j; w->config = (uint16_t)c.config_id;
        w->channel = (uint8_t)st[0].ch; w->outcome = last ? (uint8_t)(o2 ? o2 : o1) : (uint8_t)MCD_OUT_NONE;
        w->E = P::value(Ej[0]); w->E_loss = P::loss(st[0].W); w->pol = (float)st[0].c2; w->az = P::half_azimuth(r[0]);
        w->pathl = (float)st[0].l;
        w->x = (float)rx; w->y = (float)ry; w->z = (float)rz;
        w->energy = P::value(Eaft[0]);
        w->dx = (float)rdx; w->dy = (float)rdy; w->dz = (float)rdz;
        w->step_flags = st[0].flags;
      }
    }
    const int last = ran > 0 ? ran - 1 : 0, turn = last >> lg, from = g.base + (last & (g.G - 1));
    typename P::Energy Epre = shfl_any(Ej[0], from), Enext = shfl_any(Eaft[0], from);
#pragma unroll
    for (int i = 1; i < M; ++i) {
      Epre = select(turn == i, shfl_any(Ej[i], from), Epre);
      Enext = select(turn == i, shfl_any(Eaft[i], from), Enext);
    }
    if (active) {
      s.step += (uint32_t)ran;
      s.E = Enext;
      if (o1 != MCD_OUT_NONE) {
        write_rec_quad(&R.els[s.e - R.first], g.j, P::value(Epre), (float)s.d, (float)(s.p - s.pc), s.step, o1, o2,
                       s.flags);
        active = false;
      }
    }
  }
}

// One electron per lane, mid-flight: what transport_loop hands over.
struct LaneEl {
  bool active;
  uint64_t e;
  uint32_t step, flags;
  F2 E;
  float p[3], pc[3], d[3], y[3];
};

// The last electrons of a wavefront (at most 16), one per lane so far, to
// their end with 4 to 64 lanes each.
template <class P>
__device__ __forceinline__ void window_drain(const DevCfg& c, const RunArgs& R, const float* __restrict__ lds,
                                             const DevTable* __restrict__ tabs, typename P::Staged* win,
                                             const LaneEl& q, uint32_t& n_events, uint32_t& n_fp64) {
  uint64_t m = __ballot(q.active);
  const int n = __popcll(m);
  if (!n) return;
  int lg = 2;
  while (lg < 6 && (n << (lg + 1)) <= 64) ++lg;
  const int lane = threadIdx.x & 63, mine = lane >> lg;
  const int comp = (lane & 3) == 3 ? 0 : (lane & 3);
  int src = 0;
  for (int i = 0; i < n; ++i) {
    const int b = __builtin_ctzll(m);
    m &= m - 1ull;
    src = i == mine ? b : src;
  }
  auto pick = [&](const float* v) {
    const float a0 = shfl_any(v[0], src), a1 = shfl_any(v[1], src), a2 = shfl_any(v[2], src);
    return comp == 0 ? a0 : (comp == 1 ? a1 : a2);
  };
  WinEl<P> s;
  s.p = pick(q.p);
  s.pc = pick(q.pc);
  s.d = pick(q.d);
  s.y = pick(q.y);
  s.E = shfl_any(q.E, src);
  s.e = shfl_any(q.e, src);
  s.ctr1 = c.config_id | (uint32_t)(s.e >> 32) << 16;
  s.step = shfl_any(q.step, src);
  s.flags = shfl_any(q.flags, src);
  window_loop<P, false, 1>(c, R, lds, tabs, win, lg, s, mine < n, n_events, n_fp64);
}

}  // namespace mcd
