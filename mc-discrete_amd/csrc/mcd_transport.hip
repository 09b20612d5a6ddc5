// mcd_transport.hip — persistent electron-transport kernels for gfx950.
//
// One electron per lane.  Each wavefront refills its idle lanes from a device
// work counter (ballot + popcount prefix, one atomic per refill), so lanes
// whose electron was absorbed or backscattered pick up the next electron
// immediately instead of idling until the wavefront's longest trajectory ends.
// The step follows trajectory_DS (MC/tools/singleScatter.py:10-41) and
// trajectory_cont_cl (singleScatter.py:205-239); see mcd_device.h for the
// numerics.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mcd_device.h"
#include "mcd_internal.h"
#include "mcd_step.h"
#include "mcd_window.h"

namespace mcd {

// Counts of records i0, i0 + step, ... < n: each thread reads only the
// records' outcome dword (byte 32: outcome, outcome2, flags), the wavefronts
// reduce by shuffles, the block sums its wavefronts in `part` (one row of 5
// per wavefront, blockDim.x <= 256) and adds once per counter to out[0..4]
// (electrons, bks, abs, trsm, long).
static_assert(sizeof(mcd_electron_rec) == 36 && offsetof(mcd_electron_rec, outcome) == 32 &&
                  offsetof(mcd_electron_rec, outcome2) == 33,
              "count_outcome_words reads the outcome bytes as dword 8 of a 9-dword record");
__device__ __forceinline__ void count_outcome_words(const mcd_electron_rec* __restrict__ els, uint64_t n, uint64_t i0,
                                                    uint64_t step, uint32_t (*part)[5], unsigned long long* out) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(els) + 8;
  uint32_t v[5] = {0u, 0u, 0u, 0u, 0u};
  for (uint64_t i = i0; i < n; i += step) {
    const uint32_t x = __builtin_nontemporal_load(w + 9 * i);
    const uint32_t o1 = x & 0xFFu, o2 = (x >> 8) & 0xFFu;
    v[0] += 1u;
    v[1] += o1 == MCD_OUT_BKS;
    v[2] += (uint32_t)(o1 == MCD_OUT_ABS) + (uint32_t)(o2 == MCD_OUT_ABS);
    v[3] += o1 == MCD_OUT_TRSM;
    v[4] += o1 == MCD_OUT_LONG;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    uint32_t x = v[k];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if (lane == 0) part[wv][k] = x;
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    unsigned long long t = 0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += part[q][threadIdx.x];
    if (t) atomicAdd(out + threadIdx.x, t);
  }
}

// ---------------------------------------------------------------------------
// Electrons a wavefront goes on with in the window form once the work counter is
// spent: 16, the most that groups of 4 lanes hold.  Their last 1000 to 5000 steps
// cost 1.4 to 1.9 us each with one lane per electron.  us without it, at 8 and at
// 16: inline, 2^20 electrons, Cu 6090, 5520 and 5420, Au 14060, 11870 and 11530,
// Al 8410, 7960 and 7860; continuous JL 4210, 4000 and 3980, explicit law 6510,
// 6200 and 6270; served, 2^22 electrons, Cu 14750, 14280 and 14150, Au 34280,
// 31390 and 30880.
constexpr int kDrain = 16;

// ---------------------------------------------------------------------------
// The service wavefront's loop: answer posted mailboxes until every transport
// wavefront of the workgroup has finished (each adds one to *done on exit;
// a wavefront exits only after its last reply, so none is left waiting).
// A posting wavefront sets its mailbox's bit in *pending, so an idle poll is
// one LDS read between sleeps of 512 clocks (the idle service wavefront takes
// few issue slots from the transport wavefronts on its SIMD).  The loop has
// no poll limit of its own, so a launch may run as long as its work needs:
// it ends because every transport wavefront ends (the work counter is finite,
// every trajectory is capped at kMaxStepsOff steps and every wait for a reply
// is bounded by R.guard_spins), and each of them adds to *done on exit.

template <int NCH>
__device__ void guard_service(const DevCfg& c, GuardBox* boxes, uint32_t* pending, uint32_t* done, int n_boxes) {
  const int lane = threadIdx.x & 63;
  const uint32_t nb = (uint32_t)__builtin_amdgcn_readfirstlane(n_boxes);
  // a waiting transport wavefront is blocked until the reply: serve first
  __builtin_amdgcn_s_setprio(3);
  while (true) {
    if (__builtin_amdgcn_readfirstlane(box_load(pending)) == 0u) {
      if (__builtin_amdgcn_readfirstlane(box_load(done)) == nb) break;
      __builtin_amdgcn_s_sleep(8);
      continue;
    }
    // all 64 lanes are active here: lane 0 takes the pending set for the wavefront
    uint32_t q = 0;
    if (lane == 0) q = __hip_atomic_exchange(pending, 0u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
    q = __builtin_amdgcn_readfirstlane(q);
    while (q) {
      GuardBox& b = boxes[__builtin_ctz(q)];
      q &= q - 1u;
      if (box_load(&b.state) != kBoxPosted) continue;
      if ((b.mask >> lane) & 1ull) {
        GuardSlot& g = b.lane[lane];
        const int meta = g.meta;
        g.meta = d_pick_ordered<NCH>((double)g.Ehi + (double)g.Elo, (double)g.u, c, g.perm_lo, g.perm_hi,
                                     meta & 0xFF, (meta >> 8) & 1);
      }
      box_store(&b.state, kBoxReplied);
    }
  }
}

// ---------------------------------------------------------------------------
// FP32 transport (DS and continuous).
// The persistent loop of one wavefront over the electrons of one
// configuration: refill idle lanes from the configuration's work counter,
// step every active lane, write the record when a trajectory ends; returns
// when the counter is exhausted and every lane is idle.
// PHASE 0: the FP64 guard pick inline.  PHASE 1 (DS): no FP64 code; a step
// whose pick falls in the guard band parks the electron (state at the start
// of the step) and the lane takes the next electron.  PHASE 2: refill from the
// parked electrons instead of new ones, guard inline.  Phases 1 + 2 give the
// same records as phase 0: a parked step is redone from the same state and
// Philox counter.  PHASE 3 (DS): guard-band picks go to the workgroup's
// service wavefront through `box`; same records as phase 0.
// EXPL (continuous mode): the explicit Bethe law, evaluated in FP64.
// ITEM: c is a batch item's configuration, not the kernel's argument.
// ROWS: the launch may store scatter rows.
// DRAIN: once the work counter is spent and at most R.drain lanes are left, the
// loop ends and hands them over in `rest`.
template <int MODE, int NCH, int PHASE = 0, bool PERIOD = false, bool EXPL = false, bool WIDE = false,
          bool DRAIN = false, bool ITEM = false, bool PRIO = PHASE == 3, int NIGRAM = kScreenAny,
          bool ROWS = true>
__device__ __forceinline__ void transport_loop(const DevCfg& c, const float* __restrict__ lds,
                                               const DevTable* __restrict__ tabs, const RunArgs& R,
                                               uint32_t& n_events, uint32_t& n_fp64, GuardBox* box = nullptr,
                                               uint32_t* pending = nullptr, LaneEl* rest = nullptr) {
  const int lane = threadIdx.x & 63;
  uint32_t k0 = (uint32_t)R.seed, k1 = (uint32_t)(R.seed >> 32);
  const uint32_t cap = (uint32_t)(c.max_scatt < 0xFFFFFFFFll ? c.max_scatt : 0xFFFFFFFFll);
  const uint64_t n_work = PHASE == 2 ? (uint64_t)__atomic_load_n(R.park_count, __ATOMIC_RELAXED) : R.n;

  bool active = false, open = true;
  WaveQueue wq;
  uint64_t e = 0;
  uint32_t ctr1 = 0;  // second Philox counter word of the lane's electron
  uint32_t step = 0, flags = 0;
  F2 E = {0.f, 0.f};
  float p[3] = {0.f, 0.f, 0.f}, pc[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 0.f}, y[3] = {0.f, 0.f, 0.f};

  uint32_t iter = 0;
  [[maybe_unused]] uint32_t piter = 0;
  const uint32_t refill_mask = PERIOD ? R.refill_mask : 0u;
  while (true) {
    // the key words stay loop-carried SGPR values (set where all lanes are
    // converged): otherwise the compiler hoists all twenty round keys out of
    // the loop and spills them to VGPR lanes, paying a v_readlane per round
    asm volatile("" : "+s"(k0), "+s"(k1));
    // compaction period (PERIOD kernels): idle lanes take new electrons every
    // (refill_mask + 1) steps, and at once when every lane is idle
    if (open && (!PERIOD || (iter++ & refill_mask) == 0u || !__any(active))) {
      uint64_t idle = __ballot(!active);
      if (idle) {
        const uint64_t idx = refill_index(wq, PHASE == 2 ? R.resume_queue : R.queue, idle, lane, n_work, open);
        if (!active) {
          if (idx < n_work) {
            active = true;
            if constexpr (PHASE == 2) {
              const ParkRec& q = R.park[idx];
              e = q.e;
              if (e - R.first >= R.n) {
                // not an electron of this launch: its record cannot be placed,
                // so the launch is reported invalid instead of writing out of range
                atomicAdd(R.counters + MCD_CNT_GUARD_TIMEOUTS, 1ull);
                active = false;
              } else {
                ctr1 = c.config_id | (uint32_t)(e >> 32) << 16;
                step = q.step;
                flags = q.flags;
                E.hi = q.Ehi; E.lo = q.Elo;
#pragma unroll
                for (int j = 0; j < 3; ++j) { p[j] = q.p[j]; pc[j] = q.pc[j]; d[j] = q.d[j]; y[j] = q.y[j]; }
              }
            } else {
              e = R.first + idx;
              ctr1 = c.config_id | (uint32_t)(e >> 32) << 16;
              step = 0;
              flags = 0;
              E.hi = c.E0_hi; E.lo = c.E0_lo;
              p[0] = p[1] = p[2] = 0.f;
              pc[0] = pc[1] = pc[2] = 0.f;
              d[0] = c.dir0_f[0]; d[1] = c.dir0_f[1]; d[2] = c.dir0_f[2];
              y[0] = 0.f; y[1] = 1.f; y[2] = 0.f;
            }
          }
        }
      }
    }
    if constexpr (DRAIN) {
      if (!open && __popcll(__ballot(active)) <= R.drain) {
        rest->active = active;
        rest->e = e;
        rest->step = step;
        rest->flags = flags;
        rest->E = E;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          rest->p[i] = p[i];
          rest->pc[i] = pc[i];
          rest->d[i] = d[i];
          rest->y[i] = y[i];
        }
        break;
      }
    }
    if (!__any(active)) break;
    // Wavefronts holding high-energy electrons (the longest remaining
    // trajectories) issue before the others on their SIMD, so the electrons
    // started last are not the ones left running alone after the work counter
    // is spent.  Served kernel, 2^22 electrons: 16.1 -> 15.4 ms (the same rule
    // applied only past the end of the counter gave 16.0 ms).
    if (PRIO && (PHASE == 3 || (piter++ & 7u) == 0u)) {
      const float span = c.E0_hi - c.Emin_hi;
      if (__any(active && E.hi > c.Emin_hi + 0.5f * span)) __builtin_amdgcn_s_setprio(3);
      else if (__any(active && E.hi > c.Emin_hi + 0.2f * span)) __builtin_amdgcn_s_setprio(2);
      else __builtin_amdgcn_s_setprio(1);
    }
    if (!active) continue;

    // ---- one loop iteration of trajectory_DS / trajectory_cont_cl ----
    if (step >= cap) {  // num_scatt > maxScatt -> 'long'
      const float sp[3] = {p[0] - pc[0], p[1] - pc[1], p[2] - pc[2]};  // compensated, as for other outcomes
      write_rec(&R.els[e - R.first], E.hi, d, sp, step, MCD_OUT_LONG, 0, flags);
      active = false;
      continue;
    }
    const U4 r = philox10((uint32_t)e, ctr1, step, 0u, k0, k1);
    const F2 Epre = E;
    float l, Wh, Wl = 0.f, c2, s2, u_az;
    int ch = MCD_CH_RUTH;
    uint32_t sflags = 0;
    if (MODE == MCD_MODE_DS) {
      const float u0 = u01f(r.x), u1 = u01f(r.y), u2 = u01f(r.z);
      u_az = u01f(r.w);
      float mfp_ln2;
      PickEval<NCH> pe;
      ch = f_pick_table<NCH, WIDE>(lds, c.pick, E.hi, u0, mfp_ln2, pe);
      if constexpr (PHASE == 1) {
        if (ch < 0) {  // guard band: park the electron for the resume kernel
          const uint64_t m = __ballot(true);
          const int leader = __ffsll((unsigned long long)m) - 1;
          unsigned long long base = 0;
          if (lane == leader) base = atomicAdd(R.park_count, (unsigned long long)__popcll(m));
          const uint64_t slot = lane_u64(base, leader) + __popcll(m & ((1ull << lane) - 1ull));
          ParkRec& q = R.park[slot];
          q.Ehi = E.hi; q.Elo = E.lo;
#pragma unroll
          for (int j = 0; j < 3; ++j) { q.p[j] = p[j]; q.pc[j] = pc[j]; q.d[j] = d[j]; q.y[j] = y[j]; }
          q.step = step;
          q.flags = flags;
          q.e = e;
          active = false;
          continue;
        }
      } else if constexpr (PHASE == 3) {
        if (__any(ch < 0)) {  // guard band: post to the service wavefront and wait
          served_pick<NCH>(box, pending, R.guard_spins, E, u0, pe, ch, sflags);
          if (sflags & MCD_FLAG_FP64_PICK) n_fp64++;
          if (sflags & MCD_FLAG_GUARD_TIMEOUT) atomicAdd(R.counters + MCD_CNT_GUARD_TIMEOUTS, 1ull);
        }
      } else {
        if (ch < 0) {  // guard band: settle the pick in FP64
          uint32_t plo, phi;
          guard_perm<NCH>(pe, plo, phi);
          const DevCfg& ca = ITEM ? anew(c) : args_anew().c;
          ch = d_pick_ordered<NCH>((double)E.hi + (double)E.lo, (double)u0, ca, plo, phi, pe.swap, pe.exact);
          sflags |= MCD_FLAG_FP64_PICK;
          n_fp64++;
        }
      }
      l = -mfp_ln2 * log2_f(u1);
      ds_loss_angles(c, tabs, E, ch, u2, Wh, Wl, c2, s2, sflags);
    } else {
      const float u0 = u01f(r.x), u1 = u01f(r.y);
      u_az = u01f(r.z);
      float a;
      cont_path_loss<EXPL, NIGRAM>(c, E, ln_f(u0), a, l, Wh, Wl, sflags);
      const float om = 1.f - u1;
      const float inv = __builtin_amdgcn_rcpf(om + a);
      s2 = a * u1 * inv;
      c2 = om * (1.f + a) * inv;
    }
    n_events++;

    // update_xyz (electron.py:64-84), Kahan-compensated position
    const float v0 = l * d[0] - pc[0], v1 = l * d[1] - pc[1], v2 = l * d[2] - pc[2];
    const float t0 = p[0] + v0, t1 = p[1] + v1, t2 = p[2] + v2;
    int o1 = MCD_OUT_NONE, o2 = MCD_OUT_NONE;
    const float pre0 = p[0], pre1 = p[1], pre2 = p[2];
    if (t2 <= 0.f) o1 = MCD_OUT_BKS;
    else if (t2 >= c.thickness_f) o1 = MCD_OUT_TRSM;
    else {
      pc[0] = (t0 - p[0]) - v0; pc[1] = (t1 - p[1]) - v1; pc[2] = (t2 - p[2]) - v2;
      p[0] = t0; p[1] = t1; p[2] = t2;
    }
    // update_energy (electron.py:44-59): absorbed when E - W <= Emin
    E = f2_sub(E, Wh, Wl);
    if (f2_le(E, c.Emin_hi, c.Emin_lo)) {
      if (o1 == MCD_OUT_NONE) o1 = MCD_OUT_ABS; else o2 = MCD_OUT_ABS;
    }
    flags |= sflags;
    const bool done = o1 != MCD_OUT_NONE;
    if (done) {
      // saveOutcomes: pre-loss energy, pre-rotation direction, last interior position
      const float sp[3] = {p[0] - pc[0], p[1] - pc[1], p[2] - pc[2]};
      write_rec(&R.els[e - R.first], Epre.hi, d, sp, step + 1, o1, o2, flags);
    }
    const bool rec_row = ROWS && R.rows != nullptr && e < R.row_max_electron;
    if (!done || rec_row) f_rotate(c2, s2, u_az, d, y);  // update_direction
    if (ROWS && R.rows != nullptr) {
      const uint64_t slot = append_slot(rec_row, R.row_cursor, R.row_cap, lane);
      if (slot != ~0ull) {
        mcd_scatter_rec* w = &R.rows[slot];
        w->electron = (uint32_t)e; w->step = step; w->config = (uint16_t)c.config_id;
        w->channel = (uint8_t)ch; w->outcome = (uint8_t)(o2 ? o2 : o1);
        w->E = Epre.hi; w->E_loss = Wh + Wl; w->pol = c2; w->az = kPiF * u_az; w->pathl = l;
        w->x = pre0; w->y = pre1; w->z = pre2;
        w->energy = E.hi;
        w->dx = d[0]; w->dy = d[1]; w->dz = d[2];
        w->step_flags = sflags;
      }
    }
    step++;
    if (done) active = false;
  }
}

// MINW: minimum resident wavefronts per SIMD the register allocation must
// allow (1 = compiler's choice, the default; others per launch).
// PRIO: issue priority by energy, every eighth step.  NIGRAM (continuous mode):
// the elastic screening, branched on at the launch instead of at every step.
template <int MODE, int NCH, int MINW, int PHASE = 0, bool EXPL = false, bool PRIO = false, int NIGRAM = kScreenAny,
          bool ROWS = true>
__global__ __launch_bounds__(256, MINW) void k_transport_f32(DevCfg c, RunArgs R) {
  extern __shared__ float lds[];
  DevTable* tabs = nullptr;
  if (MODE == MCD_MODE_DS) {
    tabs = stage_single(c, lds);
    __syncthreads();
  }
  uint32_t n_events = 0, n_fp64 = 0;
  constexpr bool drain = PHASE == 0 && MINW == 4 && !ROWS;
  LaneEl rest;
  transport_loop<MODE, NCH, PHASE, true, EXPL, false, drain, false, PRIO, NIGRAM, ROWS>(
      c, lds, tabs, R, n_events, n_fp64, nullptr, nullptr, &rest);
  if constexpr (drain) {
    typedef typename std::conditional<MODE == MCD_MODE_DS, Fp32Ds<NCH>, Fp32Cont<EXPL>>::type P;
    // The arguments read anew: shared with the loop above, the drain's uses
    // made the loop reload or spill its scalars at every step (5 % slower).
    const KernelArgs& A = args_anew();
    typename P::Staged* win = reinterpret_cast<typename P::Staged*>(reinterpret_cast<char*>(lds) + A.R.win_off) +
                              win_stage(1) * (threadIdx.x >> 6);
    if (A.R.drain) window_drain<P>(A.c, A.R, lds, tabs, win, rest, n_events, n_fp64);
  }
  const int lane = threadIdx.x & 63;
  const uint64_t cnt[2] = {n_events, n_fp64};
  wave_add_counters(R.counters + MCD_CNT_EVENTS, cnt, 1, lane);
  wave_add_counters(R.counters + MCD_CNT_FP64_PICKS, cnt + 1, 1, lane);
}

// Service-guard kernel (DS, FP32).  LDS: one GuardBox per transport wavefront,
// the finished-wavefront count and the pending-mailbox bits, the pick table
// (wide records), the two loss-table descriptors.  Wavefront 0 serves the guard
// picks, the others run the transport.
// MINW: resident wavefronts per SIMD the register allocation must allow.
__host__ __device__ inline int svc_pick_offset(int block) {
  return (int)(((block >> 6) - 1) * sizeof(GuardBox) + 16) / (int)sizeof(float);
}
static size_t svc_lds_bytes(const DevCfg& c, int block) {
  return svc_pick_offset(block) * sizeof(float) +
         (((size_t)tab_offset_floats(c.pick.n_nodes * pick_stride_wide(c.pick.n_ch)) * sizeof(float) +
           2 * sizeof(DevTable) + 15) & ~(size_t)15);
}

// Launches without scatter rows take a kernel without their tests in the step
// (us with and without, 2^22 electrons: Cu, 7 channels 14451 and 14166, Al 6780
// and 6633, Si 12988 and 12636; Au with 8 channels 20290 and 19910).  From 9
// channels on it spills more at 64 VGPRs (9 channels 20720 and 21000, 10 21060 and
// 21450, 11 21620 and 24070), and the one with the tests serves both.
template <int NCH>
constexpr bool kLean = NCH <= 8;

template <int NCH, int MINW, bool ROWS>
__global__ __launch_bounds__(1024, MINW) void k_transport_svc(DevCfg c, RunArgs R) {
  extern __shared__ float lds[];
  float* pick = lds + svc_pick_offset(blockDim.x);
  DevTable* tabs = stage_single_wide<NCH>(c, pick);
  const int n_boxes = (int)(blockDim.x >> 6) - 1;
  GuardBox* boxes = reinterpret_cast<GuardBox*>(lds);
  uint32_t* done = reinterpret_cast<uint32_t*>(boxes + n_boxes);
  uint32_t* pending = done + 1;
  if (threadIdx.x == 0) {
    *done = 0u;
    *pending = 0u;
  }
  if ((int)threadIdx.x < n_boxes) {
    boxes[threadIdx.x].state = 0u;
    boxes[threadIdx.x].bit = 1u << threadIdx.x;
  }
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (w == 0) {
    guard_service<NCH>(c, boxes, pending, done, n_boxes);
    return;
  }
  uint32_t n_events = 0, n_fp64 = 0;
  constexpr bool drain = !ROWS || !kLean<NCH>;  // launches with rows have none
  LaneEl rest;
  transport_loop<MCD_MODE_DS, NCH, 3, true, false, true, drain, false, true, kScreenAny, ROWS>(
      c, pick, tabs, R, n_events, n_fp64, boxes + (w - 1), pending, &rest);
  if constexpr (drain) {
    // The last electrons as in k_transport_f32; their windows take the place of
    // the mailbox's slots, which are free between two posts.
    typedef Fp32DsServed<NCH> P;
    const KernelArgs& A = args_anew();
    typename P::Staged* win = reinterpret_cast<typename P::Staged*>(boxes[w - 1].lane);
    if (A.R.drain) window_drain<P>(A.c, A.R, pick, tabs, win, rest, n_events, n_fp64);
  }
  const int lane = threadIdx.x & 63;
  // every lane is converged here; the service wavefront stops once all are counted
  if (lane == 0) __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  const uint64_t cnt[2] = {n_events, n_fp64};
  wave_add_counters(R.counters + MCD_CNT_EVENTS, cnt, 1, lane);
  wave_add_counters(R.counters + MCD_CNT_FP64_PICKS, cnt + 1, 1, lane);
}

// ---------------------------------------------------------------------------
// Batched launch: many configurations in one persistent grid.  A wavefront
// works on one configuration at a time (its constants and channel-pick table
// staged in the wavefront's own LDS slice), refills
// from that configuration's counter and, once the counter is exhausted and its
// lanes are idle, moves to the configuration with the most remaining work per
// active wavefront.  Initial placement spreads wavefronts over configurations
// in proportion to their estimated work.
// Work of an item in a phase: new electrons (phases 0, 1) or parked ones (2).
template <int PHASE>
__device__ __forceinline__ void item_work(const BatchItemDev& it, unsigned long long& done, unsigned long long& total) {
  if (PHASE == 2) {
    done = __atomic_load_n(it.R.resume_queue, __ATOMIC_RELAXED);
    total = __atomic_load_n(it.R.park_count, __ATOMIC_RELAXED);
  } else {
    done = __atomic_load_n(it.R.queue, __ATOMIC_RELAXED);
    total = it.R.n;
  }
}

// The item with the most estimated work left per wavefront already on it,
// among items [lo, hi); -1 when none has electrons left to claim.
template <int PHASE>
__device__ __forceinline__ int most_work_left(const BatchItemDev* __restrict__ items, int lo, int hi, int lane) {
  float best = 0.f;
  int bi = -1;
  for (int c = lo + lane; c < hi; c += 64) {
    unsigned long long q, n;
    item_work<PHASE>(items[c], q, n);
    if (q < n) {
      const unsigned long long act = __atomic_load_n(items[c].active, __ATOMIC_RELAXED);
      const float rem = (float)(n - q) * items[c].cost / (float)(act + 1);
      if (rem > best) { best = rem; bi = c; }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const float ob = __shfl_xor(best, off);
    const int oi = __shfl_xor(bi, off);
    if (ob > best || (ob == best && oi >= 0 && (bi < 0 || oi < bi))) { best = ob; bi = oi; }
  }
  return __builtin_amdgcn_readfirstlane(bi);
}

// The next item for a wavefront of XCD group [lo, hi): one of the group's
// items while any has electrons left to claim, so that the XCD's L2 holds the
// tables of its own group only; after that, help elsewhere.
template <int PHASE>
__device__ __forceinline__ int next_item(const BatchItemDev* __restrict__ items, int n_items, int lo, int hi,
                                         int lane) {
  const int ci = most_work_left<PHASE>(items, lo, hi, lane);
  return ci >= 0 ? ci : most_work_left<PHASE>(items, 0, n_items, lane);
}

// The XCD (accelerator complex die) the wavefront runs on: HW_REG_XCC_ID
// bits [3:0] (hardware register 20 of the gfx94x/gfx950 family).
__device__ __forceinline__ int xcc_id() {
  return (int)(__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 15u);
}

// The wavefront's LDS slice holds a copy of the configuration constants
// followed by the channel-pick table, so the step loop reads both from LDS.
constexpr int kCfgFloats = (int)((sizeof(DevCfg) + 15) / 16 * 4);

int batched_cfg_floats() { return kCfgFloats; }
// before them (DRAIN) the staged steps of its last electrons, which are read one past the end
constexpr int kItemWinFloats = (int)(64 * sizeof(Fp32Base::Staged) / sizeof(float));
constexpr int kItemTabFloats = (int)((2 * sizeof(DevTable) + 15) / 16 * 4);

// PERIOD: idle lanes take new electrons every refill_mask + 1 steps (the
// launch's compaction period), and at once when all are idle; otherwise every
// step.  A separate instantiation, so the every-step kernels keep their
// register budget.  c: the item's constants (scalar loads); cl: the
// wavefront's LDS copy, whose two table descriptors the lanes select from.
// DRAIN: the item's last electrons as in k_transport_f32, their staged steps at
// win (drain of them at most).
template <int MODE, int NCH, int PHASE, bool PERIOD, bool DRAIN, bool EXPL = false>
__device__ __forceinline__ void run_item(const DevCfg& c, const DevTable* tabs, const RunArgs& itR, const float* pick,
                                         Fp32Base::Staged* win, uint64_t seed, uint32_t refill_mask,
                                         unsigned long long* ic, uint32_t& ne, uint32_t& nf, GuardBox* box,
                                         uint32_t* pending) {
  RunArgs R = itR;
  R.seed = seed;
  R.refill_mask = refill_mask;
  // the item's counter block of this launch: phases 2 and 3 count errors in it
  if constexpr (PHASE >= 2) R.counters = ic;
  // the table descriptors from the LDS copy: the per-lane Moller / Gryzinski select reads LDS
  R.drain = DRAIN ? kDrain : 0;
  LaneEl rest;
  constexpr int kPhase = MODE == MCD_MODE_DS ? PHASE : 0;
  // items store no scatter rows
  transport_loop<MODE, NCH, kPhase, PERIOD, EXPL, false, DRAIN, true, kPhase == 3, kScreenAny, false>(
      c, pick, tabs, R, ne, nf, box, pending, &rest);
  if constexpr (DRAIN) {
    typedef typename std::conditional<MODE == MCD_MODE_DS, Fp32DsItem<NCH>, Fp32Cont<EXPL>>::type P;
    RunArgs D = anew(itR);
    D.seed = seed;
    window_drain<P>(anew(c), D, pick, tabs, win, rest, ne, nf);
  }
}

// The batched kernel's service wavefront: as guard_service, for mailboxes
// whose transport wavefronts may be on different configurations; the
// configuration of mailbox w is the LDS copy in wavefront w + 1's slice (that
// wavefront waits for the reply, so the copy stays in place).
__device__ void guard_service_batched(const float* lds, int slice_floats, GuardBox* boxes, uint32_t* pending,
                                      uint32_t* done, int n_boxes) {
  const int lane = threadIdx.x & 63;
  const uint32_t nb = (uint32_t)__builtin_amdgcn_readfirstlane(n_boxes);
  __builtin_amdgcn_s_setprio(3);
  while (true) {  // ends as guard_service does: every transport wavefront ends and adds to *done
    if (__builtin_amdgcn_readfirstlane(box_load(pending)) == 0u) {
      if (__builtin_amdgcn_readfirstlane(box_load(done)) == nb) break;
      __builtin_amdgcn_s_sleep(8);
      continue;
    }
    uint32_t q = 0;
    if (lane == 0) q = __hip_atomic_exchange(pending, 0u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
    q = __builtin_amdgcn_readfirstlane(q);
    while (q) {
      const int w = __builtin_ctz(q);
      GuardBox& b = boxes[w];
      q &= q - 1u;
      if (box_load(&b.state) != kBoxPosted) continue;
      const DevCfg& c = *reinterpret_cast<const DevCfg*>(lds + (size_t)(w + 1) * slice_floats);
      const int nch = __builtin_amdgcn_readfirstlane(c.n_shells + 3);
      if ((b.mask >> lane) & 1ull) {
        GuardSlot& g = b.lane[lane];
        const int meta = g.meta;
        const double E = (double)g.Ehi + (double)g.Elo, u = (double)g.u;
        const int sw = meta & 0xFF;
        const bool ex = (meta >> 8) & 1;
        int ch;
        switch (nch) {
          case 4: ch = d_pick_ordered<4>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 5: ch = d_pick_ordered<5>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 6: ch = d_pick_ordered<6>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 7: ch = d_pick_ordered<7>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 8: ch = d_pick_ordered<8>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 9: ch = d_pick_ordered<9>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          case 10: ch = d_pick_ordered<10>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
          default: ch = d_pick_ordered<11>(E, u, c, g.perm_lo, g.perm_hi, sw, ex); break;
        }
        g.meta = ch;
      }
      box_store(&b.state, kBoxReplied);
    }
  }
}

// LDS of the batched kernel: one slice per wavefront, then (served guard)
// one mailbox per transport wavefront and the finished count and pending bits.
__host__ __device__ inline size_t batched_box_offset(int block, int slice_floats) {
  return ((size_t)(block / 64) * slice_floats * sizeof(float) + 15) & ~(size_t)15;
}
static size_t batched_lds_bytes(int phase, int block, int slice_floats) {
  if (phase != 3) return (size_t)(block / 64) * slice_floats * sizeof(float);
  return batched_box_offset(block, slice_floats) + (size_t)(block / 64 - 1) * sizeof(GuardBox) + 16;
}

// PHASE 0: guard inline.  PHASE 1: DS items park guarded steps (no FP64 code
// in the kernel).  PHASE 2: DS items resume their parked electrons.  PHASE 3:
// wavefront 0 of each workgroup serves the guard picks of the others (no FP64
// code on the transport path, one phase).
// The items are read through the constant address space: they do not change
// during the launch, so the item's configuration constants, the same for the
// whole wavefront, are scalar loads into SGPRs (reloaded where needed) rather
// than per-lane LDS reads held in VGPRs.
// Register budgets measured on MI355X for the 64-configuration batch: 5
// resident wavefronts per SIMD for phases 0, 1 and 3 (phase 0 spills at its
// refill, FP64-guard and item-switch code and still beats 4 and 6
// wavefronts), 4 for phase 2.
// DRAIN (phase 0, short runs): every item's last electrons with several lanes
// each, 4 wavefronts per SIMD (119 VGPRs; 111 spills at 5).
template <int PHASE, bool PERIOD, bool DRAIN = false>
__global__ __launch_bounds__(PHASE == 3 ? 1024 : 256, PHASE == 2 || DRAIN ? 4 : 5) void k_transport_batched(
    const __attribute__((address_space(4))) BatchItemDev* __restrict__ citems, int n_items,
    const int* __restrict__ group_start, int n_groups, int slice_floats, uint64_t seed, uint32_t refill_mask,
    unsigned long long* __restrict__ counters) {
  const BatchItemDev* items = (const BatchItemDev*)citems;
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float* my = lds + (size_t)wib * slice_floats + (DRAIN ? kItemWinFloats : 0);
  float* pick = my + (DRAIN ? kItemTabFloats : kCfgFloats);
  const DevTable* tabs = DRAIN ? reinterpret_cast<const DevTable*>(my) : &reinterpret_cast<const DevCfg*>(my)->tm;
  Fp32Base::Staged* win = DRAIN ? reinterpret_cast<Fp32Base::Staged*>(my - kItemWinFloats) : nullptr;
  GuardBox* boxes = nullptr;
  uint32_t *done = nullptr, *pending = nullptr;
  if constexpr (PHASE == 3) {
    const int n_boxes = (int)(blockDim.x >> 6) - 1;
    boxes = reinterpret_cast<GuardBox*>(reinterpret_cast<char*>(lds) + batched_box_offset(blockDim.x, slice_floats));
    done = reinterpret_cast<uint32_t*>(boxes + n_boxes);
    pending = done + 1;
    if (threadIdx.x == 0) {
      *done = 0u;
      *pending = 0u;
    }
    if ((int)threadIdx.x < n_boxes) {
      boxes[threadIdx.x].state = 0u;
      boxes[threadIdx.x].bit = 1u << threadIdx.x;
    }
    __syncthreads();
    if (wib == 0) {
      guard_service_batched(lds, slice_floats, boxes, pending, done, n_boxes);
      return;
    }
  }
  GuardBox* box = PHASE == 3 ? boxes + (wib - 1) : nullptr;
  const int grp = xcc_id() % n_groups;
  const int glo = __builtin_amdgcn_readfirstlane(group_start[grp]);
  const int ghi = __builtin_amdgcn_readfirstlane(group_start[grp + 1]);
  int ci = -1;
  if (PHASE != 2) {
    // spread the group's wavefronts over its items in proportion to their
    // estimated work, so a wavefront mostly stays on one configuration
    // (blocks are placed on the XCDs round-robin: this XCD holds every
    // n_groups-th block)
    const int wpb = (int)(blockDim.x >> 6);
    const int local = (int)(blockIdx.x / n_groups) * wpb + wib;
    const int total = (int)((gridDim.x + n_groups - 1) / n_groups) * wpb;
    const float f = ((float)local + 0.5f) / (float)total;
    for (int c = glo; c < ghi; ++c)
      if (f >= items[c].cum_lo && f < items[c].cum_hi) ci = c;
    ci = __builtin_amdgcn_readfirstlane(ci);
  }
  if (ci < 0 || __atomic_load_n(items[ci].R.queue, __ATOMIC_RELAXED) >= items[ci].R.n)
    ci = next_item<PHASE>(items, n_items, glo, ghi, lane);
  while (ci >= 0) {
    const BatchItemDev& it = items[ci];
    if (lane == 0) atomicAdd(it.active, 1ull);
    // stage the configuration and its pick table in this wavefront's slice
    const float* src = DRAIN ? reinterpret_cast<const float*>(&it.c.tm) : reinterpret_cast<const float*>(&it.c);
    for (int i = lane; i < (int)((DRAIN ? 2 * sizeof(DevTable) : sizeof(DevCfg)) / 4); i += 64) my[i] = src[i];
    const int mode = it.c.mode;
    const int nch = it.c.n_shells + 3;
    if (mode == MCD_MODE_DS) {
      const int nfl = it.c.pick.n_nodes * it.c.pick.stride;
      for (int i = lane; i < nfl; i += 64) pick[i] = it.c.pick.nodes[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const DevCfg& c = *reinterpret_cast<const DevCfg*>(my);
    const DevCfg& cg = (const DevCfg&)citems[ci].c;  // the same constants as scalar loads
    const RunArgs& rg = (const RunArgs&)citems[ci].R;
    // set only where the loop uses it, so it is not live across the other phases' loops
    unsigned long long* icl = PHASE >= 2 ? counters + (size_t)it.slot * MCD_NCOUNTERS : nullptr;
    uint32_t ne = 0, nf = 0;
    if (mode == MCD_MODE_CONT) {
      if (PHASE != 2) {
        if ((DRAIN ? cg.bethe : c.bethe) == MCD_BETHE_EXPLICIT)
          run_item<MCD_MODE_CONT, 4, PHASE, PERIOD, DRAIN, true>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, nullptr, nullptr);
        else
          run_item<MCD_MODE_CONT, 4, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, nullptr, nullptr);
      }
    } else {
      switch (nch) {
        case 4: run_item<MCD_MODE_DS, 4, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 5: run_item<MCD_MODE_DS, 5, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 6: run_item<MCD_MODE_DS, 6, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 7: run_item<MCD_MODE_DS, 7, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 8: run_item<MCD_MODE_DS, 8, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 9: run_item<MCD_MODE_DS, 9, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        case 10: run_item<MCD_MODE_DS, 10, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
        default: run_item<MCD_MODE_DS, 11, PHASE, PERIOD, DRAIN>(cg, tabs, rg, pick, win, seed, refill_mask, icl, ne, nf, box, pending); break;
      }
    }
    const uint64_t cnt[2] = {ne, nf};
    unsigned long long* ic = counters + (size_t)it.slot * MCD_NCOUNTERS;
    wave_add_counters(ic + MCD_CNT_EVENTS, cnt, 1, lane);
    wave_add_counters(ic + MCD_CNT_FP64_PICKS, cnt + 1, 1, lane);
    if (lane == 0) atomicSub(it.active, 1ull);
    ci = next_item<PHASE>(items, n_items, glo, ghi, lane);
    __builtin_amdgcn_wave_barrier();
  }
  if constexpr (PHASE == 3) {
    // every lane is converged here; the service wavefront stops once all are counted
    if (lane == 0) __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
}

template <int PHASE, bool PERIOD, bool DRAIN = false>
static const void* batched_kernel() {
  return reinterpret_cast<const void*>(&k_transport_batched<PHASE, PERIOD, DRAIN>);
}

// The kernel of a phase; the phases that take new electrons (0, 1, 3) have a
// compaction-period form, the resume phase (2) refills every step.
static const void* batched_kernel(int phase, bool period, bool drain) {
  if (drain) return period ? batched_kernel<0, true, true>() : batched_kernel<0, false, true>();
  switch (phase) {
    case 1: return period ? batched_kernel<1, true>() : batched_kernel<1, false>();
    case 2: return batched_kernel<2, false>();
    case 3: return period ? batched_kernel<3, true>() : batched_kernel<3, false>();
    default: return period ? batched_kernel<0, true>() : batched_kernel<0, false>();
  }
}

// A slice (slice_floats without a drain) as the kernel lays it out.
static int batched_slice(int slice_floats, bool drain) {
  return drain ? slice_floats - kCfgFloats + kItemTabFloats + kItemWinFloats : slice_floats;
}
int batched_blocks_per_cu(int phase, int block, int slice_floats, bool period, bool drain) {
  int nb = 0;
  const size_t lds = batched_lds_bytes(phase, block, batched_slice(slice_floats, drain));
  const void* k = batched_kernel(phase, period, drain);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, block, lds) != hipSuccess) return 0;
  return nb;
}

hipError_t launch_batched(const BatchItemDev* items, int n_items, const int* group_start, int n_groups,
                          int slice_floats, uint64_t seed, uint32_t refill_mask, unsigned long long* counters,
                          int phase, int grid, int block, bool drain, hipStream_t s) {
  if (phase == 3 && (block < 128 || block > 1024)) return hipErrorInvalidValue;
  if (n_groups < 1 || n_groups > kMaxXcdGroups || (drain && phase)) return hipErrorInvalidValue;
  int slice = batched_slice(slice_floats, drain);
  const size_t lds = batched_lds_bytes(phase, block, slice);
  const void* k = batched_kernel(phase, refill_mask != 0u, drain);
  void* args[] = {(void*)&items, (void*)&n_items, (void*)&group_start, (void*)&n_groups, (void*)&slice,
                  (void*)&seed, (void*)&refill_mask, (void*)&counters};
  return hipLaunchKernel(k, dim3(grid), dim3(block), args, lds, s);
}

__global__ __launch_bounds__(256) void k_count_outcomes_batched(const BatchItemDev* __restrict__ items,
                                                                unsigned long long* counters) {
  __shared__ uint32_t part[4][5];
  const BatchItemDev& it = items[blockIdx.y];
  count_outcome_words(it.R.els, it.R.n, (uint64_t)blockIdx.x * blockDim.x + threadIdx.x,
                      (uint64_t)gridDim.x * blockDim.x, part,
                      counters + (size_t)it.slot * MCD_NCOUNTERS + MCD_CNT_ELECTRONS);
}

hipError_t launch_count_outcomes_batched(const BatchItemDev* items, int n_items, unsigned long long* counters,
                                         hipStream_t s) {
  hipLaunchKernelGGL(k_count_outcomes_batched, dim3(64, n_items), dim3(256), 0, s, items, counters);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP64 transport: the same loop with every quantity in double and the exact
// pick each step (the all-FP64 GPU run).  Arithmetic is not contracted into
// FMAs so the operation order matches the reference expressions.

template <int MODE, int NCH>
__global__ __launch_bounds__(256) void k_transport_f64(DevCfg c, RunArgs R) {
  const int lane = threadIdx.x & 63;
  const uint32_t k0 = (uint32_t)R.seed, k1 = (uint32_t)(R.seed >> 32);
  bool active = false, open = true;
  WaveQueue wq;
  uint64_t e = 0;
  uint32_t step = 0, flags = 0;
  double E = 0., p[3] = {0., 0., 0.}, d[3] = {0., 0., 0.}, y[3] = {0., 0., 0.};
  uint32_t n_events = 0;
  while (true) {
    if (open) {
      uint64_t idle = __ballot(!active);
      if (idle) {
        const uint64_t idx = refill_index(wq, R.queue, idle, lane, R.n, open);
        if (!active) {
          if (idx < R.n) {
            active = true;
            e = R.first + idx;
            step = 0; flags = 0;
            E = c.E0;
            p[0] = p[1] = p[2] = 0.;
            d[0] = c.dir0[0]; d[1] = c.dir0[1]; d[2] = c.dir0[2];
            y[0] = 0.; y[1] = 1.; y[2] = 0.;
          }
        }
      }
    }
    if (!__any(active)) break;
    if (!active) continue;
    if ((int64_t)step >= c.max_scatt) {
      const float df[3] = {(float)d[0], (float)d[1], (float)d[2]};
      const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
      write_rec(&R.els[e - R.first], (float)E, df, pf, step, MCD_OUT_LONG, 0, flags);
      active = false;
      continue;
    }
    const U4 r = philox10((uint32_t)e, c.config_id | (uint32_t)(e >> 32) << 16, step, 0u, k0, k1);
    const double Epre = E;
    const DStep o = d_step_physics<MODE, NCH>(c, c.tm, c.tg, E, r);
    n_events++;
    double np_[3];
    d_advance(p, o.l, d, np_);
    int o1 = MCD_OUT_NONE, o2 = MCD_OUT_NONE;
    const double pre0 = p[0], pre1 = p[1], pre2 = p[2];
    if (np_[2] <= 0.) o1 = MCD_OUT_BKS;
    else if (np_[2] >= c.thickness) o1 = MCD_OUT_TRSM;
    else { p[0] = np_[0]; p[1] = np_[1]; p[2] = np_[2]; }
    const double En = E - o.W;
    if (En <= c.Emin) { if (o1 == MCD_OUT_NONE) o1 = MCD_OUT_ABS; else o2 = MCD_OUT_ABS; }
    E = En;
    uint32_t sflags = o.sflags;
    if (o.c2 != o.c2) sflags |= MCD_FLAG_NAN_DIR;
    flags |= sflags;
    const bool done = o1 != MCD_OUT_NONE;
    if (done) {
      const float df[3] = {(float)d[0], (float)d[1], (float)d[2]};
      const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
      write_rec(&R.els[e - R.first], (float)Epre, df, pf, step + 1, o1, o2, flags);
    }
    const bool rec_row = R.rows != nullptr && e < R.row_max_electron;
    if (!done || rec_row) {
      double c_ht, s_ht, c_hp, s_hp;
      d_half_angles(o.c2, o.hp, c_ht, s_ht, c_hp, s_hp);
      d_rotate(c_ht, s_ht, c_hp, s_hp, d, y);
    }
    if (R.rows != nullptr) {
      const uint64_t slot = append_slot(rec_row, R.row_cursor, R.row_cap, lane);
      if (slot != ~0ull) {
        mcd_scatter_rec* w = &R.rows[slot];
        w->electron = (uint32_t)e; w->step = step; w->config = (uint16_t)c.config_id;
        w->channel = (uint8_t)o.ch; w->outcome = (uint8_t)(o2 ? o2 : o1);
        w->E = (float)Epre; w->E_loss = (float)o.W; w->pol = (float)o.c2; w->az = (float)o.hp;
        w->pathl = (float)o.l;
        w->x = (float)pre0; w->y = (float)pre1; w->z = (float)pre2;
        w->energy = (float)E;
        w->dx = (float)d[0]; w->dy = (float)d[1]; w->dz = (float)d[2];
        w->step_flags = sflags;
      }
    }
    step++;
    if (done) active = false;
  }
  const uint64_t cnt = n_events;
  wave_add_counters(R.counters + MCD_CNT_EVENTS, &cnt, 1, lane);
}

// ---------------------------------------------------------------------------
// Outcome counts from the electron records: electrons, bks, abs (both rows
// of an exit-then-absorb electron count), trsm, long.
__global__ __launch_bounds__(256) void k_count_outcomes(const mcd_electron_rec* __restrict__ els, uint64_t n,
                                                        unsigned long long* __restrict__ counters) {
  __shared__ uint32_t part[4][5];
  count_outcome_words(els, n, (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, (uint64_t)gridDim.x * blockDim.x,
                      part, counters + MCD_CNT_ELECTRONS);
}

hipError_t launch_count_outcomes(const mcd_electron_rec* els, uint64_t n, unsigned long long* counters,
                                 hipStream_t s) {
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(k_count_outcomes, dim3((unsigned)blocks), dim3(256), 0, s, els, n, counters);
  return hipGetLastError();
}

// Selected fields of scatter rows as packed columns: field f of row i goes to
// out + plan.dst[f] + i * plan.size[f].  One thread per row, grid-stride; a
// row is one 64-byte line, so its fields are read from one cache line and
// each column is written with consecutive addresses across the wavefront.
__global__ __launch_bounds__(256) void k_pack_scatter(const uint8_t* __restrict__ rows, uint64_t n, ScatPackPlan plan,
                                                      uint8_t* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint8_t* r = rows + i * sizeof(mcd_scatter_rec);
    for (int f = 0; f < plan.n; ++f) {
      const int sz = plan.size[f];
      const uint8_t* src = r + plan.src[f];
      uint8_t* dst = out + plan.dst[f] + i * (uint64_t)sz;
      if (sz == 4) *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(src);
      else if (sz == 2) *reinterpret_cast<uint16_t*>(dst) = *reinterpret_cast<const uint16_t*>(src);
      else *dst = *src;
    }
  }
}

hipError_t launch_pack_scatter(const mcd_scatter_rec* rows, uint64_t n, const ScatPackPlan& plan, void* out,
                               hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_pack_scatter, dim3((unsigned)blocks), dim3(256), 0, s,
                     reinterpret_cast<const uint8_t*>(rows), n, plan, reinterpret_cast<uint8_t*>(out));
  return hipGetLastError();
}

// First row of each electron in (electron, step) order: the exclusive prefix
// sum of the records' scatter counts (an electron has one row per event).  One
// workgroup: each thread adds a run of records, the workgroup scans its runs.
__global__ __launch_bounds__(1024) void k_row_starts(const mcd_electron_rec* __restrict__ els, uint64_t n,
                                                     uint64_t* __restrict__ starts) {
  __shared__ uint64_t part[1024];
  const uint64_t run = (n + blockDim.x - 1) / blockDim.x;
  const uint64_t a = run * threadIdx.x, b = a + run < n ? a + run : n;
  uint64_t sum = 0;
  for (uint64_t i = a; i < b; ++i) sum += els[i].n_scatt;
  part[threadIdx.x] = sum;
  __syncthreads();
  for (unsigned off = 1; off < blockDim.x; off <<= 1) {
    const uint64_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint64_t at = part[threadIdx.x] - sum;
  for (uint64_t i = a; i < b; ++i) {
    starts[i] = at;
    at += els[i].n_scatt;
  }
}

// Each row to its place in (electron, step) order.  One thread per row; the
// rows a wavefront appended lie side by side, mostly steps of one electron.
// Bound by the 64 bytes read and the packed bytes written per row.
__global__ __launch_bounds__(256) void k_order_scatter(const mcd_scatter_rec* __restrict__ rows, uint64_t n,
                                                       uint64_t n_els, uint32_t first, ScatPackPlan plan,
                                                       int row_bytes, const uint64_t* __restrict__ starts,
                                                       uint8_t* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const mcd_scatter_rec* r = rows + i;
    const uint32_t el = r->electron - first;
    if (el >= n_els) continue;
    const uint64_t place = starts[el] + r->step;
    if (place >= n) continue;
    uint8_t* dst = out + place * (uint64_t)row_bytes;
    const uint8_t* src = reinterpret_cast<const uint8_t*>(r);
    for (int f = 0; f < plan.n; ++f) {
      const uint8_t* v = src + plan.src[f];
      uint8_t* w = dst + plan.dst[f];  // packed rows: any alignment
      if (plan.size[f] == 4) __builtin_memcpy(w, v, 4);
      else if (plan.size[f] == 2) __builtin_memcpy(w, v, 2);
      else *w = *v;
    }
  }
}

hipError_t launch_order_scatter(const mcd_scatter_rec* rows, uint64_t n, const mcd_electron_rec* els, uint64_t n_els,
                                uint32_t first, const ScatPackPlan& plan, int row_bytes, void* out, uint64_t* starts,
                                hipStream_t s) {
  if (n == 0 || n_els == 0) return hipSuccess;
  hipLaunchKernelGGL(k_row_starts, dim3(1), dim3(1024), 0, s, els, n_els, starts);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_order_scatter, dim3((unsigned)blocks), dim3(256), 0, s, rows, n, n_els, first, plan, row_bytes,
                     starts, reinterpret_cast<uint8_t*>(out));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// host-side launchers

// LDS of a one-kernel launch that needs `used` bytes for its step, with the
// windows of its last electrons after them (D.win_off, D.drain); without them
// where they would take the place of resident wavefronts (16 per CU at 4 per
// SIMD, 160 KB of LDS).
static size_t with_drain(size_t used, int block, RunArgs& D) {
  const size_t at = (used + 15) & ~(size_t)15;
  const size_t all = at + (size_t)(block / 64) * win_stage(1) * sizeof(Fp32Base::Staged);
  const bool fits = all <= 64 * 1024 && all * (1024 / block) <= 160 * 1024;
  D.win_off = (int)at;
  D.drain = fits ? kDrain : 0;
  return fits ? all : used;
}

// The kernel of a launch.  Continuous mode at 4 wavefronts per SIMD: one per
// screening, and from three wavefronts per SIMD on, where they take turns, with
// issue priorities: in us without and with them, 50021 electrons (JL, less than
// one per SIMD) 1393 and 1405, 2^19 3776 and 3307, 2^22 11186 and 10624; explicit
// law 2^19 5764 and 5242, 2^22 27992 and 27475.  DS steps are longer and gain
// less than it costs them (2^18 Cu 2873 and 2771, but 2^20 Au 12019 and 12217).
// Launches without scatter rows take kernels without their tests in the step: us
// with and without, 131072 and 2^20 electrons, Cu 2242 and 2139, 5571 and 5393, Au
// 6058 and 5996, 11563 and 11405; explicit law 65536 1747 and 1635.
template <int MODE, int NCH, int MINW, bool EXPL>
static const void* f32_kernel(const DevCfg& c, int simd_waves, bool rows) {
  if constexpr (MINW == 4 && MODE == MCD_MODE_DS)
    if (!rows) return reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL, false, kScreenAny, false>);
  if constexpr (MODE == MCD_MODE_CONT && MINW == 4) {
    if (rows) return reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL>);
    if (c.elastic >= MCD_ELASTIC_NIGRAM)
      return simd_waves >= 3 ? reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL, true, 1, false>)
                             : reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL, false, 1, false>);
    return simd_waves >= 3 ? reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL, true, 0, false>)
                           : reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL, false, 0, false>);
  }
  return reinterpret_cast<const void*>(&k_transport_f32<MODE, NCH, MINW, 0, EXPL>);
}

template <int MODE, int NCH, int MINW, bool EXPL>
static hipError_t launch_f32(const DevCfg& c, const RunArgs& R, int grid, int block, size_t used, hipStream_t s) {
  RunArgs D = R;
  const size_t lds = MINW == 4 && !R.rows ? with_drain(used, block, D) : used;
  void* args[] = {(void*)&c, (void*)&D};
  return hipLaunchKernel(f32_kernel<MODE, NCH, MINW, EXPL>(c, R.simd_waves, R.rows != nullptr), dim3(grid), dim3(block), args, lds, s);
}

template <int MODE, int NCH, int MINW, bool EXPL>
static int occ_f32(const DevCfg& c, int block, size_t used) {
  int nb = 0;
  RunArgs D;
  const size_t lds = MINW == 4 ? with_drain(used, block, D) : used;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f32_kernel<MODE, NCH, MINW, EXPL>(c, 0, false), block, lds) !=
      hipSuccess)
    return 1;
  return nb < 1 ? 1 : nb;
}

// dispatch over (channel count, occupancy variant)
template <int MODE, int NCH, bool EXPL = false>
static hipError_t dispatch_w(int minw, const DevCfg& c, const RunArgs* R, int grid, int block, size_t lds,
                             hipStream_t s, int* occ) {
  switch (minw) {
#define MCD_W(W)                                                   \
  case W:                                                          \
    if (occ) { *occ = occ_f32<MODE, NCH, W, EXPL>(c, block, lds); return hipSuccess; } \
    return launch_f32<MODE, NCH, W, EXPL>(c, *R, grid, block, lds, s);
    MCD_W(1) MCD_W(4) MCD_W(5) MCD_W(6) MCD_W(8)
#undef MCD_W
    default: return hipErrorInvalidValue;
  }
}

static hipError_t dispatch_f32(int minw, const DevCfg& c, const RunArgs* R, int grid, int block, hipStream_t s,
                               int* occ) {
  if (c.mode == MCD_MODE_CONT) {
    if (c.bethe == MCD_BETHE_EXPLICIT) return dispatch_w<MCD_MODE_CONT, 4, true>(minw, c, R, grid, block, 0, s, occ);
    return dispatch_w<MCD_MODE_CONT, 4>(minw, c, R, grid, block, 0, s, occ);
  }
  const size_t lds = single_lds_bytes(c);
  switch (c.n_shells + 3) {
    case 4: return dispatch_w<MCD_MODE_DS, 4>(minw, c, R, grid, block, lds, s, occ);
    case 5: return dispatch_w<MCD_MODE_DS, 5>(minw, c, R, grid, block, lds, s, occ);
    case 6: return dispatch_w<MCD_MODE_DS, 6>(minw, c, R, grid, block, lds, s, occ);
    case 7: return dispatch_w<MCD_MODE_DS, 7>(minw, c, R, grid, block, lds, s, occ);
    case 8: return dispatch_w<MCD_MODE_DS, 8>(minw, c, R, grid, block, lds, s, occ);
    case 9: return dispatch_w<MCD_MODE_DS, 9>(minw, c, R, grid, block, lds, s, occ);
    case 10: return dispatch_w<MCD_MODE_DS, 10>(minw, c, R, grid, block, lds, s, occ);
    case 11: return dispatch_w<MCD_MODE_DS, 11>(minw, c, R, grid, block, lds, s, occ);
    default: return hipErrorInvalidValue;
  }
}

bool valid_minw(int w) { return w == 1 || w == 4 || w == 5 || w == 6 || w == 8; }

// the FP64 kernel of a configuration
static const void* f64_kernel(const DevCfg& c) {
  if (c.mode != MCD_MODE_DS) return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_CONT, 4>);
  switch (c.n_shells + 3) {
    case 4: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 4>);
    case 5: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 5>);
    case 6: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 6>);
    case 7: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 7>);
    case 8: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 8>);
    case 9: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 9>);
    case 10: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 10>);
    default: return reinterpret_cast<const void*>(&k_transport_f64<MCD_MODE_DS, 11>);
  }
}

hipError_t launch_transport(const DevCfg& c, const RunArgs& R, int precision, int minw, int grid, int block,
                            hipStream_t s) {
  if (precision == MCD_PREC_FP64) {
    void* args[] = {(void*)&c, (void*)&R};
    return hipLaunchKernel(f64_kernel(c), dim3(grid), dim3(block), args, 0, s);
  }
  return dispatch_f32(minw, c, &R, grid, block, s, nullptr);
}

// resident blocks per CU for the persistent grid
int max_blocks_per_cu(const DevCfg& c, int precision, int minw, int block) {
  int nb = 1;
  if (precision == MCD_PREC_FP64) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f64_kernel(c), block, 0) != hipSuccess || nb < 1) nb = 1;
    return nb;
  }
  if (dispatch_f32(minw, c, nullptr, 0, block, 0, &nb) != hipSuccess || nb < 1) nb = 1;
  return nb;
}

// ---------------------------------------------------------------------------
// Deferred guard (DS, FP32): phase 1 without FP64 code, phase 2 resumes.
template <int NCH, int PHASE>
static hipError_t deferred_nch(const DevCfg& c, const RunArgs* R, int grid, int block, size_t lds, hipStream_t s,
                               int* occ) {
  if (occ) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_transport_f32<MCD_MODE_DS, NCH, 1, PHASE>, block, lds) !=
        hipSuccess)
      nb = 1;
    *occ = nb < 1 ? 1 : nb;
    return hipSuccess;
  }
  hipLaunchKernelGGL((k_transport_f32<MCD_MODE_DS, NCH, 1, PHASE>), dim3(grid), dim3(block), lds, s, c, *R);
  return hipGetLastError();
}

template <int PHASE>
static hipError_t deferred_dispatch(const DevCfg& c, const RunArgs* R, int grid, int block, hipStream_t s, int* occ) {
  const size_t lds = single_lds_bytes(c);
  switch (c.n_shells + 3) {
    case 4: return deferred_nch<4, PHASE>(c, R, grid, block, lds, s, occ);
    case 5: return deferred_nch<5, PHASE>(c, R, grid, block, lds, s, occ);
    case 6: return deferred_nch<6, PHASE>(c, R, grid, block, lds, s, occ);
    case 7: return deferred_nch<7, PHASE>(c, R, grid, block, lds, s, occ);
    case 8: return deferred_nch<8, PHASE>(c, R, grid, block, lds, s, occ);
    case 9: return deferred_nch<9, PHASE>(c, R, grid, block, lds, s, occ);
    case 10: return deferred_nch<10, PHASE>(c, R, grid, block, lds, s, occ);
    case 11: return deferred_nch<11, PHASE>(c, R, grid, block, lds, s, occ);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_transport_deferred(const DevCfg& c, const RunArgs& R, int phase, int grid, int block,
                                     hipStream_t s) {
  if (c.mode != MCD_MODE_DS) return hipErrorInvalidValue;
  return phase == 1 ? deferred_dispatch<1>(c, &R, grid, block, s, nullptr)
                    : deferred_dispatch<2>(c, &R, grid, block, s, nullptr);
}

// ---------------------------------------------------------------------------
// Service guard (DS, FP32): one kernel, wavefront 0 of each workgroup settles
// the guard-band picks of the others.
template <int NCH, int MINW>
static hipError_t svc_nch(const DevCfg& c, const RunArgs* R, int grid, int block, size_t lds, hipStream_t s,
                          int* occ) {
  if (occ) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_transport_svc<NCH, MINW, !kLean<NCH>>, block, lds) !=
        hipSuccess)
      nb = 1;
    *occ = nb < 1 ? 1 : nb;
    return hipSuccess;
  }
  RunArgs D = *R;
  D.drain = R->rows ? 0 : kDrain;
  if (R->rows || !kLean<NCH>)
    hipLaunchKernelGGL((k_transport_svc<NCH, MINW, true>), dim3(grid), dim3(block), lds, s, c, D);
  else
    hipLaunchKernelGGL((k_transport_svc<NCH, MINW, !kLean<NCH>>), dim3(grid), dim3(block), lds, s, c, D);
  return hipGetLastError();
}

template <int MINW>
static hipError_t svc_dispatch(const DevCfg& c, const RunArgs* R, int grid, int block, hipStream_t s, int* occ) {
  const size_t lds = svc_lds_bytes(c, block);
  switch (c.n_shells + 3) {
    case 4: return svc_nch<4, MINW>(c, R, grid, block, lds, s, occ);
    case 5: return svc_nch<5, MINW>(c, R, grid, block, lds, s, occ);
    case 6: return svc_nch<6, MINW>(c, R, grid, block, lds, s, occ);
    case 7: return svc_nch<7, MINW>(c, R, grid, block, lds, s, occ);
    case 8: return svc_nch<8, MINW>(c, R, grid, block, lds, s, occ);
    case 9: return svc_nch<9, MINW>(c, R, grid, block, lds, s, occ);
    case 10: return svc_nch<10, MINW>(c, R, grid, block, lds, s, occ);
    case 11: return svc_nch<11, MINW>(c, R, grid, block, lds, s, occ);
    default: return hipErrorInvalidValue;
  }
}

bool valid_svc_minw(int w) { return w == 6 || w == 7 || w == 8; }

static hipError_t svc_any(int minw, const DevCfg& c, const RunArgs* R, int grid, int block, hipStream_t s, int* occ) {
  switch (minw) {
    case 6: return svc_dispatch<6>(c, R, grid, block, s, occ);
    case 7: return svc_dispatch<7>(c, R, grid, block, s, occ);
    case 8: return svc_dispatch<8>(c, R, grid, block, s, occ);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_transport_svc(const DevCfg& c, const RunArgs& R, int minw, int grid, int block, hipStream_t s) {
  if (c.mode != MCD_MODE_DS || block < 128 || block > 1024 || block % 64) return hipErrorInvalidValue;
  return svc_any(minw, c, &R, grid, block, s, nullptr);
}

int svc_blocks_per_cu(const DevCfg& c, int minw, int block) {
  int nb = 1;
  hipError_t e = svc_any(minw, c, nullptr, 0, block, 0, &nb);
  return e == hipSuccess && nb > 0 ? nb : 1;
}

int deferred_blocks_per_cu(const DevCfg& c, int phase, int block) {
  int nb = 1;
  hipError_t e = phase == 1 ? deferred_dispatch<1>(c, nullptr, 0, block, 0, &nb)
                            : deferred_dispatch<2>(c, nullptr, 0, block, 0, &nb);
  return e == hipSuccess && nb > 0 ? nb : 1;
}

}  // namespace mcd
