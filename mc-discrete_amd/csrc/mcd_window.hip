// mcd_window.hip — transport of small launches: several lanes per electron.
//
// A launch of few electrons cannot fill the chip with one electron per lane;
// it takes the longest trajectory (10^3 steps) times the latency of a step on
// a lone wavefront (1.1 to 1.4 us: ~400 instructions issued one after the
// other, two LDS and three L2 round trips).  Here G lanes (4 to 64) share an
// electron and take a window of its next G steps at a time:
//   1. Random words: lane j draws step s+j's Philox words and everything that
//      depends on them alone (path-length logarithm, azimuth).
//   2. Energy chain (DS): channel, loss and angle of a step depend on the
//      energy at its start and on its random words, not on position or
//      direction.  Every lane evaluates its step at a guessed energy, first the
//      window's start energy; the losses found give each lane the energy the
//      chain of subtractions leads to; the steps are evaluated again there.  A
//      step whose loss did not change was evaluated at its exact energy, so the
//      window is final when no loss changes (two evaluations as a rule: a
//      channel or table column seldom changes over the few hundred eV of a
//      window).  The energies are the same float-pair subtractions in the same
//      order as one step after the other gives.
//   3. Geometry: path, position, exit test and rotation step after step, all
//      electrons of the wavefront at once, the three components of each vector
//      in three lanes of a quad.  Steps past the electron's end are dropped.
// Every formula is the one of transport_loop, so records, scatter rows and
// counters are the same bit for bit.
#include <hip/hip_runtime.h>

#include "mcd_device.h"
#include "mcd_internal.h"
#include "mcd_step.h"

namespace mcd {

// Lane of a quad permutation of a float (sel: source lane of quad lanes 0..3).
template <int S0, int S1, int S2, int S3>
__device__ __forceinline__ float quad_perm(float x) {
  constexpr int ctrl = S0 | (S1 << 2) | (S2 << 4) | (S3 << 6);
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), ctrl, 0xF, 0xF, true));
}
// The value of the lane before, within a row of 16 lanes.
__device__ __forceinline__ float row_prev(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x111, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_f(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// One staged step of the geometry pass: path, cos and sin of the polar angle,
// cos and |sin| of the azimuth.
struct alignas(16) WinStep {
  float l, ct, st, cp, sp, pad[3];
};
constexpr int kWinStage = 66;  // staged steps per wavefront: one a lane, two more for the reads ahead
static_assert(sizeof(WinStep) == 32, "a staged step is two 16-byte reads");

// Direction and position of one electron, component (lane & 3) of each vector
// (lanes 3 of a quad repeat component 0), and its energy and counters.
struct WinEl {
  float p, pc, d, y;
  F2 E;
  uint64_t e;
  uint32_t ctr1, step, flags;
};

__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src) {
  const uint32_t lo = __shfl((uint32_t)v, src), hi = __shfl((uint32_t)(v >> 32), src);
  return ((uint64_t)hi << 32) | lo;
}

// f_rotate (mcd_device.h) on vectors spread over a quad: the same products and
// sums per component, the two norms from all three components.
__device__ __forceinline__ void rotate_quad(float ct, float st, float cp, float sp, float& d, float& y) {
  const float y1 = quad_perm<1, 2, 0, 1>(y), y2 = quad_perm<2, 0, 1, 2>(y);
  const float d1 = quad_perm<1, 2, 0, 1>(d), d2 = quad_perm<2, 0, 1, 2>(d);
  const float w = y1 * d2 - y2 * d1;
  const float nd = ct * d + st * (cp * w + sp * y);
  const float ny = cp * y - sp * w;
  const float nd0 = quad_perm<0, 0, 0, 0>(nd), nd1 = quad_perm<1, 1, 1, 1>(nd), nd2 = quad_perm<2, 2, 2, 2>(nd);
  const float ny0 = quad_perm<0, 0, 0, 0>(ny), ny1 = quad_perm<1, 1, 1, 1>(ny), ny2 = quad_perm<2, 2, 2, 2>(ny);
  d = nd * __builtin_amdgcn_rsqf(nd0 * nd0 + nd1 * nd1 + nd2 * nd2);
  y = ny * __builtin_amdgcn_rsqf(ny0 * ny0 + ny1 * ny1 + ny2 * ny2);
}

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

// Energies at the start of each step of the window: lane j of a group gets
// E0 - W_0 - .. - W_(j-1) (E0 and the losses: the group's), one float-pair
// subtraction after the other.  lg: log2 of the group size, j = lane & (G - 1).
__device__ __forceinline__ F2 chain_energies(F2 E0, float Wh, float Wl, int lg, int lane, int j) {
  F2 cur = E0;
  if (lg <= 4) {
    // lane by lane within the row: after t rounds lanes up to t are final
    const float ph = row_prev(Wh), pl = row_prev(Wl);
    const int G = 1 << lg;
    for (int t = 1; t < G; ++t) {
      const F2 in = {row_prev(cur.hi), row_prev(cur.lo)};
      const F2 nx = f2_sub(in, ph, pl);
      cur.hi = j ? nx.hi : E0.hi;
      cur.lo = j ? nx.lo : E0.lo;
    }
    return cur;
  }
  // one or two electrons per wavefront: only the steps that lose energy (the
  // subtraction of zero leaves a normalised pair as it is)
  uint64_t m = __ballot(Wh != 0.f);
  const bool upper = lg == 5 && lane >= 32;
  if (lg == 5) m = (m | (m >> 32)) & 0xFFFFFFFFull;
  while (m) {
    const int k = __builtin_ctzll(m);
    m &= m - 1ull;
    float wh = lane_f(Wh, k), wl = lane_f(Wl, k);
    if (lg == 5) {
      const float uh = lane_f(Wh, k + 32), ul = lane_f(Wl, k + 32);
      wh = upper ? uh : wh;
      wl = upper ? ul : wl;
    }
    const F2 nx = f2_sub(cur, wh, wl);
    if (j > k) cur = nx;
  }
  return cur;
}

// Channel, free path, loss and polar angle of one DS step at energy E.
template <int NCH>
__device__ __forceinline__ void ds_step_at(const DevCfg& c, const float* __restrict__ lds,
                                           const DevTable* __restrict__ tabs, F2 E, float u0, float lg1, float u2,
                                           int& ch, float& l, float& Wh, float& Wl, float& c2, float& s2,
                                           uint32_t& sf) {
  float mfp_ln2;
  PickEval<NCH> pe;
  sf = 0;
  ch = f_pick_table<NCH>(lds, c.pick, E.hi, u0, mfp_ln2, pe);
  if (ch < 0) {  // guard band: settle the pick in FP64
    uint32_t plo, phi;
    guard_perm<NCH>(pe, plo, phi);
    ch = d_pick_ordered<NCH>((double)E.hi + (double)E.lo, (double)u0, c, plo, phi, pe.swap, pe.exact);
    sf |= MCD_FLAG_FP64_PICK;
  }
  l = -mfp_ln2 * lg1;
  ds_loss_angles(c, tabs, E, ch, u2, Wh, Wl, c2, s2, sf);
}

// LDS: the pick table, the two loss-table descriptors, one window of staged
// steps per wavefront.
__host__ __device__ inline size_t win_stage_offset(const DevCfg& c) {
  return ((size_t)tab_offset_floats(c.pick.n_nodes * c.pick.stride) * sizeof(float) + 2 * sizeof(DevTable) + 15) &
         ~(size_t)15;
}

template <int NCH, bool ROWS>
__global__ __launch_bounds__(256, 2) void k_window_ds(DevCfg c, RunArgs R, int lg) {
  extern __shared__ float lds[];
  const DevTable* tabs = stage_single(c, lds);
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  WinStep* win = reinterpret_cast<WinStep*>(reinterpret_cast<char*>(lds) + win_stage_offset(c)) + kWinStage * wib;
  __syncthreads();
  uint32_t k0 = (uint32_t)R.seed, k1 = (uint32_t)(R.seed >> 32);
  const int comp = (lane & 3) == 3 ? 0 : (lane & 3);
  const float dir0 = comp == 0 ? c.dir0_f[0] : (comp == 1 ? c.dir0_f[1] : c.dir0_f[2]);
  uint32_t n_events = 0, n_fp64 = 0;
  WinEl s = {};
  bool active = false, open = true;
  // the first electrons by position, later ones from the work counter
  const uint64_t slots = (uint64_t)gridDim.x * (blockDim.x >> lg);
  uint64_t next = (((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> lg);
  bool first = true;

  while (true) {
    // the key words stay loop-carried SGPR values (see transport_loop)
    asm volatile("" : "+s"(k0), "+s"(k1));
    int G = 1 << lg, j = lane & (G - 1), base = lane & ~(G - 1);
    if (open) {
      const uint64_t idle = __ballot(!active && j == 0);
      if (idle) {
        if (!first) {
          const int leader = __ffsll((unsigned long long)idle) - 1;
          unsigned long long b = 0;
          if (lane == leader) b = atomicAdd(R.queue, (unsigned long long)__popcll(idle));
          next = slots + lane_u64(b, leader) + __popcll(idle & ((1ull << base) - 1ull));
        }
        first = false;
        if (!active && next < R.n) {
          active = true;
          s.e = R.first + next;
          s.ctr1 = c.config_id | (uint32_t)(s.e >> 32) << 16;
          s.step = 0;
          s.flags = 0;
          s.E = {c.E0_hi, c.E0_lo};
          s.p = s.pc = 0.f;
          s.d = dir0;
          s.y = comp == 1 ? 1.f : 0.f;
        }
        // an index past the end: every later one is past it too
        open = slots < R.n && !__any(!active);
      }
    }
    const uint64_t live = __ballot(active && j == 0);
    if (!live) break;
    if (!open && lg < 6 && 2 * __popcll(live) * G <= 64) {
      // fewer electrons than half the groups: wider groups, longer windows
      const int n = __popcll(live);
      while (lg < 6 && (n << (lg + 1)) <= 64) ++lg;
      G = 1 << lg;
      j = lane & (G - 1);
      base = lane & ~(G - 1);
      const int g = lane >> lg;
      int src = 0;
      uint64_t m = live;
      for (int i = 0; i < n; ++i) {
        const int b = __builtin_ctzll(m);
        m &= m - 1ull;
        src = i == g ? b : src;
      }
      src += lane & 3;
      s.p = __shfl(s.p, src); s.pc = __shfl(s.pc, src); s.d = __shfl(s.d, src); s.y = __shfl(s.y, src);
      s.E.hi = __shfl(s.E.hi, src); s.E.lo = __shfl(s.E.lo, src);
      s.e = shfl_u64(s.e, src);
      s.ctr1 = __shfl(s.ctr1, src); s.step = __shfl(s.step, src); s.flags = __shfl(s.flags, src);
      active = g < n;
    }
    const uint64_t gmask = (G == 64 ? ~0ull : (1ull << G) - 1ull);

    // steps of the window before maxScatt ends the trajectory ('long')
    int64_t left = active ? c.max_scatt - (int64_t)s.step : 0;
    if (active && left <= 0) {
      write_rec_quad(&R.els[s.e - R.first], j, s.E.hi, s.d, s.p - s.pc, s.step, MCD_OUT_LONG, 0, s.flags);
      active = false;
    }
    const int nw = (int)(left < G ? (left > 0 ? left : 0) : G);

    // ---- 1. random words of step s + j ----
    const U4 r = philox10((uint32_t)s.e, s.ctr1, s.step + (uint32_t)j, 0u, k0, k1);
    const float u0 = u01f(r.x), u2 = u01f(r.z), u_az = u01f(r.w);
    const float lg1 = log2_f(u01f(r.y));

    // ---- 2. energy chain ----
    F2 Ej = s.E;
    float l = 0.f, Wh = 0.f, Wl = 0.f, c2 = 1.f, s2 = 0.f;
    int ch = MCD_CH_RUTH;
    uint32_t sf = 0;
    bool todo = active && j < nw;  // this lane's step is not final
    while (true) {
      const float oh = Wh, ol = Wl;
      if (todo && !f2_le(Ej, c.Emin_hi, c.Emin_lo))
        ds_step_at<NCH>(c, lds, tabs, Ej, u0, lg1, u2, ch, l, Wh, Wl, c2, s2, sf);
      // the first step of the group whose loss is not the one its energies
      // were formed with: it and the steps before it are final
      const uint64_t changed = (__ballot(todo && (Wh != oh || Wl != ol)) >> base) & gmask;
      todo = todo && changed != 0ull && j > __builtin_ctzll(changed | (1ull << 63));
      if (!__any(todo)) break;
      const F2 Ec = chain_energies(s.E, Wh, Wl, lg, lane, j);
      if (todo) Ej = Ec;
    }
    const F2 Eaft = f2_sub(Ej, Wh, Wl);  // the step's end energy
    const bool absorbed = f2_le(Eaft, c.Emin_hi, c.Emin_lo);
    // the window ends with the step that absorbs the electron
    const uint64_t am = (__ballot(active && j < nw && absorbed) >> base) & gmask;
    const int ka = am ? __builtin_ctzll(am) : 64;  // step that absorbs
    const int m = ka < nw ? ka + 1 : nw;
    {
      float cp, sp;
      cos_abs_sin_2pi(u_az, cp, sp);
      win[lane].l = l;
      win[lane].ct = c2 - s2;
      win[lane].st = 2.f * __builtin_amdgcn_sqrtf(c2 * s2);
      win[lane].cp = cp;
      win[lane].sp = sp;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // ---- 3. geometry, step after step ----
    const bool rec_row = ROWS && active && s.e < R.row_max_electron;
    int ran = 0;     // steps executed
    float tz = 1.f;  // depth after the last executed step (an exit ends the window)
    bool go = active && m > 0;
    float rx = 0.f, ry = 0.f, rz = 0.f, rdx = 0.f, rdy = 0.f, rdz = 0.f;  // ROWS: lane j's step
    // selects instead of branches: no lane leaves the loop before the last
    auto advance = [&](const WinStep& w, int k) {
      const float v = w.l * s.d - s.pc;
      const float t = s.p + v;
      const float depth = quad_perm<2, 2, 2, 2>(t);
      if constexpr (ROWS) {
        const float p0 = quad_perm<0, 0, 0, 0>(s.p), p1 = quad_perm<1, 1, 1, 1>(s.p), p2 = quad_perm<2, 2, 2, 2>(s.p);
        rx = k == j ? p0 : rx; ry = k == j ? p1 : ry; rz = k == j ? p2 : rz;
      }
      const bool stay = go && !(depth <= 0.f) && !(depth >= c.thickness_f);
      const float npc = (t - s.p) - v;
      tz = go ? depth : tz;
      ran += go ? 1 : 0;
      s.pc = stay ? npc : s.pc;
      s.p = stay ? t : s.p;
      float nd = s.d, ny = s.y;
      rotate_quad(w.ct, w.st, w.cp, w.sp, nd, ny);
      if constexpr (ROWS) {
        const float d0 = quad_perm<0, 0, 0, 0>(nd), d1 = quad_perm<1, 1, 1, 1>(nd), d2 = quad_perm<2, 2, 2, 2>(nd);
        rdx = k == j ? d0 : rdx; rdy = k == j ? d1 : rdy; rdz = k == j ? d2 : rdz;
      }
      go = stay && k != ka;
      s.d = go ? nd : s.d;
      s.y = go ? ny : s.y;
      go = go && k + 1 < m;
    };
    const WinStep* wp = win + base;
    WinStep wa = wp[0], wb;
    if constexpr (!ROWS) {
      // Most windows run whole, without an exit: every electron through all G
      // steps with no test but the smallest and largest depth; the electrons
      // that end in this window start it again below.
      const float p_ = s.p, pc_ = s.pc, d_ = s.d, y_ = s.y;
      float lo = 1.f, hi = 0.f;
      auto pass = [&](const WinStep& w) {
        const float v = w.l * s.d - s.pc;
        const float t = s.p + v;
        s.pc = (t - s.p) - v;
        s.p = t;
        lo = fminf(lo, t);
        hi = fmaxf(hi, t);
        rotate_quad(w.ct, w.st, w.cp, w.sp, s.d, s.y);
      };
      for (int k = 0; k < G; k += 2) {  // each step's values are read one step ahead
        wb = wp[k + 1];
        __builtin_amdgcn_sched_barrier(0);
        pass(wa);
        wa = wp[k + 2];
        __builtin_amdgcn_sched_barrier(0);
        pass(wb);
      }
      const bool in = quad_perm<2, 2, 2, 2>(lo) > 0.f && quad_perm<2, 2, 2, 2>(hi) < c.thickness_f;
      if (active && m == G && ka == 64 && in) {
        ran = G;
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
    if (tz <= 0.f) o1 = MCD_OUT_BKS;
    else if (tz >= c.thickness_f) o1 = MCD_OUT_TRSM;
    if (ran == ka + 1) {
      if (o1 == MCD_OUT_NONE) o1 = MCD_OUT_ABS; else o2 = MCD_OUT_ABS;
    }
    __builtin_amdgcn_wave_barrier();

    // ---- outputs of the executed steps ----
    const bool mine = active && j < ran;
    n_events += mine ? 1u : 0u;
    n_fp64 += mine && (sf & MCD_FLAG_FP64_PICK) ? 1u : 0u;
    if (__any(mine && sf)) {
#pragma unroll
      for (uint32_t bit = 1u; bit <= 8u; bit <<= 1)
        if ((__ballot(mine && (sf & bit)) >> base) & gmask) s.flags |= bit;
    }
    if constexpr (ROWS) {
      const uint64_t slot = append_slot(rec_row && mine, R.row_cursor, R.row_cap, lane);
      if (slot != ~0ull) {
        mcd_scatter_rec* w = &R.rows[slot];
        const bool last = j == ran - 1;
        w->electron = (uint32_t)s.e; w->step = s.step + (uint32_t)j; w->config = (uint16_t)c.config_id;
        w->channel = (uint8_t)ch; w->outcome = last ? (uint8_t)(o2 ? o2 : o1) : (uint8_t)MCD_OUT_NONE;
        w->E = Ej.hi; w->E_loss = Wh + Wl; w->pol = c2; w->az = kPiF * u_az; w->pathl = l;
        w->x = rx; w->y = ry; w->z = rz;
        w->energy = Eaft.hi;
        w->dx = rdx; w->dy = rdy; w->dz = rdz;
        w->step_flags = sf;
      }
    }
    const int lastl = base + (ran > 0 ? ran - 1 : 0);
    const float Epre = __shfl(Ej.hi, lastl);
    const float nh = __shfl(Eaft.hi, lastl), nl = __shfl(Eaft.lo, lastl);
    if (active) {
      s.step += (uint32_t)ran;
      s.E = {nh, nl};
      if (o1 != MCD_OUT_NONE) {
        write_rec_quad(&R.els[s.e - R.first], j, Epre, s.d, s.p - s.pc, s.step, o1, o2, s.flags);
        active = false;
      }
    }
  }
  const uint64_t cnt[2] = {n_events, n_fp64};
  wave_add_counters(R.counters + MCD_CNT_EVENTS, cnt, 1, lane);
  wave_add_counters(R.counters + MCD_CNT_FP64_PICKS, cnt + 1, 1, lane);
}

// ---------------------------------------------------------------------------
// host-side launchers
constexpr int kWinBlock = 256;

static size_t window_lds_bytes(const DevCfg& c) {
  return win_stage_offset(c) + (kWinBlock / 64) * kWinStage * sizeof(WinStep);
}

// log2 of the lanes per electron for a launch of n electrons, 0 where one lane
// per electron is the faster form.  The kernel's registers allow 4 wavefronts
// per SIMD; the widest group whose lanes fit in 15/16 of those is taken (wider
// groups take turns on the SIMDs, narrower ones leave it waiting: Cu 20 keV
// 70 deg, 2000 electrons 313 us at 64 lanes, 356 at 32; 4000: 448 at 64, 409
// at 32, 471 at 16; 10007: 655 at 32, 636 at 16, 741 at 8; 30000: 1201 at 16,
// 981 at 8, 1211 at 4).  Quads go on to 1.5 times those lanes: 90000
// electrons take 2.09 ms (Au 30 keV 5.0 ms), one lane each 2.50 ms (7.7 ms);
// at 131072 both take 2.6 ms on Cu.  Pick tables beyond 64 KB of LDS with the
// staged steps (512 nodes: 27 KB with 7 channels) take the other kernels.
int window_log2_lanes(const DevCfg& c, uint64_t n, int n_cu) {
  if (window_lds_bytes(c) > 64 * 1024) return 0;
  const uint64_t resident = (uint64_t)n_cu * 4 * 4 * 64;
  for (int lg = 6; lg > 2; --lg)
    if (n <= (resident - resident / 16) >> lg) return lg;
  return n <= (resident + resident / 2) >> 2 ? 2 : 0;
}

template <int NCH>
static hipError_t window_ds(const DevCfg& c, const RunArgs& R, int lg, hipStream_t s) {
  const size_t lds = window_lds_bytes(c);
  const uint64_t per = kWinBlock >> lg;
  const uint64_t grid = (R.n + per - 1) / per;
  const void* k = R.rows ? reinterpret_cast<const void*>(&k_window_ds<NCH, true>)
                         : reinterpret_cast<const void*>(&k_window_ds<NCH, false>);
  void* args[] = {(void*)&c, (void*)&R, (void*)&lg};
  return hipLaunchKernel(k, dim3((unsigned)grid), dim3(kWinBlock), args, lds, s);
}

hipError_t launch_window_ds(const DevCfg& c, const RunArgs& R, int lg, hipStream_t s) {
  if (lg < 2 || lg > 6) return hipErrorInvalidValue;
  switch (c.n_shells + 3) {
    case 4: return window_ds<4>(c, R, lg, s);
    case 5: return window_ds<5>(c, R, lg, s);
    case 6: return window_ds<6>(c, R, lg, s);
    case 7: return window_ds<7>(c, R, lg, s);
    case 8: return window_ds<8>(c, R, lg, s);
    case 9: return window_ds<9>(c, R, lg, s);
    case 10: return window_ds<10>(c, R, lg, s);
    case 11: return window_ds<11>(c, R, lg, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mcd
