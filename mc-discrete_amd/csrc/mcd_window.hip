// mcd_window.hip — launches too small to fill the chip with one lane per
// electron (see mcd_window.h).
#include <hip/hip_runtime.h>

#include "mcd_device.h"
#include "mcd_internal.h"
#include "mcd_step.h"
#include "mcd_window.h"

namespace mcd {

template <class P, bool ROWS>
__global__ __launch_bounds__(256, ROWS ? 2 : P::kWaves) void k_window(DevCfg c, RunArgs R, int lg) {
  constexpr int M = win_turns<P, ROWS>();
  extern __shared__ float lds[];
  const DevTable* tabs = nullptr;
  if constexpr (P::kPickTable) {
    tabs = stage_single(c, lds);
  } else {
    DevTable* t = reinterpret_cast<DevTable*>(lds);
    if (threadIdx.x == 0) {
      t[0] = c.tm;
      t[1] = c.tg;
    }
    tabs = t;
  }
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  typename P::Staged* win =
      reinterpret_cast<typename P::Staged*>(reinterpret_cast<char*>(lds) + win_stage_offset<P>(c)) + win_stage(M) * wib;
  __syncthreads();
  uint32_t n_events = 0, n_fp64 = 0;
  // one group of lanes for each electron of the launch
  const uint64_t idx = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> lg;
  const int comp = (lane & 3) == 3 ? 0 : (lane & 3);
  window_loop<P, ROWS, M>(c, R, lds, tabs, win, lg, win_start<P>(c, R.first + idx, comp), idx < R.n, n_events, n_fp64);
  const uint64_t cnt[2] = {n_events, n_fp64};
  wave_add_counters(R.counters + MCD_CNT_EVENTS, cnt, 1, lane);
  wave_add_counters(R.counters + MCD_CNT_FP64_PICKS, cnt + 1, 1, lane);
}

// ---------------------------------------------------------------------------
// host-side launchers
constexpr int kWinBlock = 256;

template <class P, bool ROWS>
static size_t window_lds_bytes(const DevCfg& c) {
  return win_stage_offset<P>(c) + (kWinBlock / 64) * win_stage(win_turns<P, ROWS>()) * sizeof(typename P::Staged);
}

// log2 of the lanes per electron for a launch of n electrons, 0 where one lane
// per electron is the faster form.  Wider groups shorten a window's step until
// the wavefronts take turns on the SIMDs, so the widest group is taken whose
// lanes stay within a number of wavefronts per SIMD; quads go on to where one
// lane per electron catches up.  Times in us (MI355X, 256 CUs; 1: one lane):
//   DS FP32, 3.75 and 5 (Cu 20 keV 70 deg; 2000 electrons 313 at 64 lanes, 356
//     at 32; 4000: 448 at 64, 409 at 32; 10007: 655 at 32, 636 at 16, 741 at 8;
//     30000: 1201 at 16, 981 at 8, 1211 at 4; one lane per electron ends in quads
//     (kDrain): 65536: 1510 at 4, 2092 at 1, Au 30 keV 3783, 5686, Al 5 keV 521,
//     740; 80000: 2027, 2163, Au 4983, 5861, Al 718, 710; 98304: 2267, 2207, Au
//     5446, 5990, Si 10 keV 1452, 1278)
//   DS FP64, 1.5 and 4 (Cu; 4000: 1967 at 32, 1709 at 16; 8192: 2623 at 16,
//     2482 at 8; 16000: 3812 at 8, 4116 at 4; 65000: 9846 at 4, 10656 at 1;
//     131072: 16980 at 4, 16270 at 1)
//   continuous, 1 and 3 (Au 30 keV JL 70 deg; 2000: 424 at 32; 10007: 646 at 4;
//     32768: 833 at 4, 1380 at 1; 40000: 1093, 1340; 50021: 1320 to 1390, 1315;
//     60000: 1412, 1320), with the explicit law 1 and 1 (16384: 1176 at 4, 1642 at
//     1; 32768: 1747, 1600; 40000: 2347, 1600)
// Pick tables beyond 64 KB of LDS with the staged steps (512 nodes: 27 KB with
// 7 channels) take the other kernels, as does continuous mode in FP64.
int window_log2_lanes(const DevCfg& c, int precision, uint64_t n, int n_cu) {
  const bool ds = c.mode == MCD_MODE_DS, f64 = precision == MCD_PREC_FP64;
  if (ds && !f64 && window_lds_bytes<Fp32Ds<4>, false>(c) > 64 * 1024) return 0;
  if (!ds && f64) return 0;
  const double wide = ds ? (f64 ? 1.5 : 3.75) : 1.;
  const double quad = ds ? (f64 ? 4. : 5.) : (c.bethe == MCD_BETHE_EXPLICIT ? 1. : 3.);
  const double lanes = (double)n_cu * 4 * 64;  // one wavefront per SIMD
  for (int lg = 6; lg > 2; --lg)
    if ((double)n * (1 << lg) <= wide * lanes) return lg;
  return (double)n * 4 <= quad * lanes ? 2 : 0;
}

template <class P>
static hipError_t window(const DevCfg& c, const RunArgs& R, int lg, hipStream_t s) {
  const uint64_t per = kWinBlock >> lg;
  const uint64_t grid = (R.n + per - 1) / per;
  const void* k = R.rows ? reinterpret_cast<const void*>(&k_window<P, true>)
                         : reinterpret_cast<const void*>(&k_window<P, false>);
  void* args[] = {(void*)&c, (void*)&R, (void*)&lg};
  const size_t lds = R.rows ? window_lds_bytes<P, true>(c) : window_lds_bytes<P, false>(c);
  return hipLaunchKernel(k, dim3((unsigned)grid), dim3(kWinBlock), args, lds, s);
}

template <template <int> class P>
static hipError_t window_ds(const DevCfg& c, const RunArgs& R, int lg, hipStream_t s) {
  switch (c.n_shells + 3) {
    case 4: return window<P<4>>(c, R, lg, s);
    case 5: return window<P<5>>(c, R, lg, s);
    case 6: return window<P<6>>(c, R, lg, s);
    case 7: return window<P<7>>(c, R, lg, s);
    case 8: return window<P<8>>(c, R, lg, s);
    case 9: return window<P<9>>(c, R, lg, s);
    case 10: return window<P<10>>(c, R, lg, s);
    case 11: return window<P<11>>(c, R, lg, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_window(const DevCfg& c, const RunArgs& R, int precision, int lg, hipStream_t s) {
  if (lg < 2 || lg > 6) return hipErrorInvalidValue;
  if (c.mode == MCD_MODE_DS)
    return precision == MCD_PREC_FP64 ? window_ds<Fp64Ds>(c, R, lg, s) : window_ds<Fp32Ds>(c, R, lg, s);
  if (precision == MCD_PREC_FP64) return hipErrorInvalidValue;
  return c.bethe == MCD_BETHE_EXPLICIT ? window<Fp32Cont<true>>(c, R, lg, s) : window<Fp32Cont<false>>(c, R, lg, s);
}

}  // namespace mcd
