// mcd_tables.hip — device-side table construction.
//
// * k_build_cdf: the inverse-CDF energy-loss rows of probTable.computeBlock
//   (MC/tools/probTables.py:415-462).  One wavefront per energy row; FP64
//   trapezoids and cumulative sums (rounded to float32 once), or the float32
//   arithmetic of the reference.  The mask W[j+1] > (E - E_F)/2 is evaluated in
//   float32 exactly as the reference's float32 arrays do (:429-439).
// * k_pick_nodes / k_pick_cells / k_pick_check / k_pick_exact: the LDS pick table (sorted
//   cumulative channel probabilities and ln mfp on a ln E grid), the kinds of its
//   cells, and its interpolation-error check against the exact FP64 pick, which
//   sets the guard band.  What the host needs of them is a PickSummary.
#include <hip/hip_runtime.h>

#include "mcd_device.h"
#include "mcd_internal.h"

namespace mcd {

#pragma clang fp contract(off)
__device__ __forceinline__ double d_moller_dcs(double E, double W, double n) {  // extFunctions.py:159-184
  double eps = W / E;
  if (!(eps < 1.)) return 0.;
  return n * kPiEFour * (1. / (eps * eps) + (1. / ((1. - eps) * (1. - eps))) - (1. / (eps * (1. - eps)))) /
         (E * E * E);
}
__device__ __forceinline__ double d_gryz_dcs(double E, double W, double n, double Eb) {  // :189-219
  double eps = W / E, epsB = Eb / E;
  if (!(eps < 1. && epsB < 1.)) return 0.;
  return n * kPiEFour * eps * pow(1. + epsB, -1.5) * pow(1. - eps, epsB / (epsB + eps)) *
         ((1. - epsB) + 4. * epsB * log(2.7 + sqrt((1. - eps) / epsB)) / (3. * eps)) / (W * W * W);
}
#pragma clang fp contract(on)

__device__ __forceinline__ float f_moller_dcs(float E, float W, float kn) {
  float eps = W / E;
  float om = 1.f - eps;
  float v = kn * (1.f / (eps * eps) + (1.f / (om * om)) - (1.f / (eps * om))) / powf(E, 3.f);
  return eps < 1.f ? v : 0.f;
}
__device__ __forceinline__ float f_gryz_dcs(float E, float W, float kn, float Eb) {
  float eps = W / E, epsB = Eb / E;
  float v = kn * eps * powf(1.f + epsB, -1.5f) * powf(1.f - eps, epsB / (epsB + eps)) *
            ((1.f - epsB) + 4.f * epsB * logf(2.7f + sqrtf((1.f - eps) / epsB)) / (3.f * eps)) / powf(W, 3.f);
  return (eps < 1.f && epsB < 1.f) ? v : 0.f;
}

// Energy row i of a table's CDF (computeBlock, probTables.py:415-462), one
// wavefront to a row.  The lanes share the integrand's values and the
// trapezoids of a tile of loss bins; one lane adds them up in order, so the
// running sums are those of one bin after the other.  Rows wider than a tile
// take two passes, the first for the total alone.
// Bound by the FP64 integrand (Gryzinski: two pow, a log, a sqrt and seven
// divisions a value).  One thread to a row evaluated every value twice on 47
// wavefronts: 371 us for 3000 x 199 Gryzinski cells and 137 us for 2000 x 199
// Moller cells on MI355X, now 21 and 16 us.
constexpr int kCdfTile = 256, kCdfWaves = 4;

__device__ __forceinline__ double dcs(int kind, double E, double W, double n_el, double Eb) {
  return kind == MCD_TABLE_MOLLER ? d_moller_dcs(E, W, n_el) : d_gryz_dcs(E, W, n_el, Eb);
}
__device__ __forceinline__ float dcs(int kind, float E, float W, float kn, float Eb) {
  return kind == MCD_TABLE_MOLLER ? f_moller_dcs(E, W, kn) : f_gryz_dcs(E, W, kn, Eb);
}
template <class Real>
__device__ __forceinline__ float cdf_value(Real acc, Real tot) {
  return (float)(acc / tot);
}

// Real: FP64, or the float32 arithmetic of the reference.  k: n_el, times
// pi e^4 in float32.  part: kCdfTile + 1 values of LDS.
template <class Real>
__device__ __forceinline__ void cdf_row(float E32, const float* __restrict__ Ws, int nb, double Ef, int kind, Real k,
                                        Real Eb, float* __restrict__ row, Real* part) {
  const int lane = threadIdx.x & 63;
  const float wmax32 = (E32 - (float)Ef) * 0.5f;  // float32 mask, probTables.py:429-439
  // number of valid bins: W[j+1] <= wmax32 (Ws increasing)
  int nvalid = 0, end = nb;
  while (nvalid < end) {
    const int mid = (nvalid + end) >> 1;
    if (!(Ws[mid + 1] > wmax32)) nvalid = mid + 1; else end = mid;
  }
  const Real E = (Real)E32;
  Real tot = 0;
  for (int pass = nvalid > kCdfTile ? 0 : 1; pass < 2; ++pass) {
    Real acc = 0;
    for (int j0 = 0; j0 < nvalid; j0 += kCdfTile) {
      const int m = min(kCdfTile, nvalid - j0);
      for (int j = lane; j <= m; j += 64) part[j] = dcs(kind, E, (Real)Ws[j0 + j], k, Eb);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      Real f0[kCdfTile / 64], f1[kCdfTile / 64];
#pragma unroll
      for (int q = 0; q < kCdfTile / 64; ++q) {
        const int j = lane + 64 * q;
        f0[q] = j < m ? part[j] : 0;
        f1[q] = j < m ? part[j + 1] : 0;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < kCdfTile / 64; ++q) {
        const int j = lane + 64 * q;
        if (j < m) part[j] = ((Real)Ws[j0 + j + 1] - (Real)Ws[j0 + j]) * (f0[q] + f1[q]) / (Real)2;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane == 0) {
#pragma unroll 8
        for (int j = 0; j < m; ++j) {
          acc += part[j];
          part[j] = acc;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      acc = part[m - 1];
      if (pass == 1) {
        if (nvalid <= kCdfTile) tot = acc;
        for (int j = lane; j < m; j += 64) row[j0 + j] = cdf_value(part[j], tot);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (pass == 0) tot = acc;
  }
  for (int j = nvalid + lane; j < nb; j += 64) row[j] = kMasked;
}

__device__ __forceinline__ void cdf_row(const float* __restrict__ Es, const float* __restrict__ Ws, int i, int nW,
                                        double Ef, int kind, double n_el, double Eb, int precision,
                                        float* __restrict__ cdf) {
  __shared__ double part[kCdfWaves][kCdfTile + 1];
  double* p = part[threadIdx.x >> 6];
  const int nb = nW - 1;
  float* row = cdf + (size_t)i * nb;
  if (precision == MCD_PREC_FP64)
    cdf_row<double>(Es[i], Ws, nb, Ef, kind, n_el, Eb, row, p);
  else
    cdf_row<float>(Es[i], Ws, nb, Ef, kind, (float)(n_el * kPiEFour), (float)Eb, row, reinterpret_cast<float*>(p));
}

__global__ __launch_bounds__(64 * kCdfWaves) void k_build_cdf(const float* __restrict__ Es,
                                                              const float* __restrict__ Ws, int nE, int nW, double Ef,
                                                              int kind, double n_el, double Eb, int precision,
                                                              float* __restrict__ cdf) {
  const int i = (int)blockIdx.x * kCdfWaves + (int)(threadIdx.x >> 6);
  if (i >= nE) return;
  cdf_row(Es, Ws, i, nW, Ef, kind, n_el, Eb, precision, cdf);
}

// The job holding global row g of a batch: jobs cover consecutive row ranges
// [row0, row0 + nE) in order.
__device__ __forceinline__ int job_of_row(const CdfJob* __restrict__ jobs, int n_jobs, long long g) {
  int lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].row0 <= g) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The CDF rows of many tables in one launch, as in k_build_cdf.
__global__ __launch_bounds__(64 * kCdfWaves) void k_build_cdf_batched(const CdfJob* __restrict__ jobs, int n_jobs,
                                                                      long long total_rows, int precision) {
  const long long g = (long long)blockIdx.x * kCdfWaves + (threadIdx.x >> 6);
  if (g >= total_rows) return;
  const CdfJob& j = jobs[job_of_row(jobs, n_jobs, g)];
  cdf_row(j.Es, j.Ws, (int)(g - j.row0), j.nW, j.Ef, j.kind, j.n_el, j.Eb, precision, j.cdf);
}

hipError_t launch_build_cdf(const float* Es, const float* Ws, int nE, int nW, double Ef, int kind, double n_el,
                            double Eb, int precision, float* cdf, hipStream_t s) {
  hipLaunchKernelGGL(k_build_cdf, dim3((nE + kCdfWaves - 1) / kCdfWaves), dim3(64 * kCdfWaves), 0, s, Es, Ws, nE, nW,
                     Ef, kind, n_el, Eb, precision, cdf);
  return hipGetLastError();
}

// Likelihood-ratio scores of loss-table column picks for the derivative
// replay, from the discrete tables themselves (their float32 CDFs, masks
// included).  p_j is the mass of column j of a row (CDF difference; 0 where
// masked).
__device__ __forceinline__ double col_mass(const float* row, int j) {
  const float c = row[j];
  if (c == kMasked) return 0.;
  return (double)c - (j > 0 ? (double)row[j - 1] : 0.);
}

// Parameter score: (p_j(+) - p_j(-)) / (2 delta p_j) from the tables rebuilt
// at the parameter +- delta (the central difference of the column
// probabilities, masks included).
__global__ void k_ratio_score(const float* __restrict__ c0, const float* __restrict__ cp,
                              const float* __restrict__ cm, int nE, int nb, double inv_2delta,
                              float* __restrict__ out) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (size_t)nE * nb) return;
  const size_t i = k / nb;
  const int j = (int)(k - i * nb);
  const float* r0 = c0 + i * nb;
  const double p0 = col_mass(r0, j);
  out[k] = p0 > 0. ? (float)((col_mass(cp + i * nb, j) - col_mass(cm + i * nb, j)) * inv_2delta / p0) : 0.f;
}

// Energy score: rows are piecewise constant in energy (row i serves
// (Es[i-1], Es[i]]); the score of a pick from row i is the row-to-row change
// (p_j(i) - p_j(i-1)) / ((Es[i] - Es[i-1]) p_j(i)).
__global__ void k_row_score(const float* __restrict__ cdf, const float* __restrict__ Es, int nE, int nb,
                            float* __restrict__ out) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (size_t)nE * nb) return;
  const size_t i = k / nb;
  const int j = (int)(k - i * nb);
  const double p = col_mass(cdf + i * nb, j);
  if (i == 0 || !(p > 0.)) {
    out[k] = 0.f;
    return;
  }
  const double q = col_mass(cdf + (i - 1) * nb, j);
  out[k] = (float)((p - q) / (((double)Es[i] - (double)Es[i - 1]) * p));
}

hipError_t launch_ratio_score(const float* c0, const float* cp, const float* cm, int nE, int nW, double inv_2delta,
                              float* out, hipStream_t s) {
  const size_t n = (size_t)nE * (nW - 1);
  hipLaunchKernelGGL(k_ratio_score, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, c0, cp, cm, nE, nW - 1,
                     inv_2delta, out);
  return hipGetLastError();
}

hipError_t launch_row_score(const float* cdf, const float* Es, int nE, int nW, float* out, hipStream_t s) {
  const size_t n = (size_t)nE * (nW - 1);
  hipLaunchKernelGGL(k_row_score, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, cdf, Es, nE, nW - 1, out);
  return hipGetLastError();
}

// Row records (layout in mcd_device.h): bracket energies and the quantile
// guide q -> bisect_left(cdf_row, q / G) (masked entries hold kMasked, above
// every q / G).  One workgroup per row.
__device__ __forceinline__ void row_record(const float* __restrict__ cdf, const float* __restrict__ Es, int row,
                                           int nW, int narrow, uint8_t* __restrict__ rows) {
  const int nb = nW - 1;
  const float* r = cdf + (size_t)row * nb;
  uint8_t* rec = rows + (size_t)row * kRowBytes;
  if (threadIdx.x == 0) {
    float2 br;
    br.x = Es[row > 0 ? row - 1 : 0];
    br.y = Es[row];
    *reinterpret_cast<float2*>(rec) = br;
  }
  const int G = narrow ? kGuideNarrow : kGuideWide;
  const int used = kRowHeader + (narrow ? 1 : 2) * (G + 1);
  for (int b = used + threadIdx.x; b < kRowBytes; b += blockDim.x) rec[b] = 0;
  for (int q = threadIdx.x; q <= G; q += blockDim.x) {
    const float v = (float)q / (float)G;
    int lo = 0, hi = nb;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (r[mid] < v) lo = mid + 1; else hi = mid;
    }
    if (narrow) rec[kRowHeader + q] = (uint8_t)lo;
    else reinterpret_cast<uint16_t*>(rec + kRowHeader)[q] = (uint16_t)lo;
  }
}

__global__ void k_build_rows(const float* __restrict__ cdf, const float* __restrict__ Es, int nE, int nW, int narrow,
                             uint8_t* __restrict__ rows) {
  row_record(cdf, Es, blockIdx.x, nW, narrow, rows);
}

// Row records of many tables in one launch: one workgroup per energy row of
// any table.
__global__ void k_build_rows_batched(const CdfJob* __restrict__ jobs, int n_jobs) {
  const long long g = blockIdx.x;
  const CdfJob& j = jobs[job_of_row(jobs, n_jobs, g)];
  row_record(j.cdf, j.Es, (int)(g - j.row0), j.nW, j.nW - 1 <= 255, j.rows);
}

hipError_t launch_build_tables_batched(const CdfJob* jobs, int n_jobs, long long total_rows, int precision,
                                       hipStream_t s) {
  if (n_jobs < 1 || total_rows < 1 || total_rows > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_build_cdf_batched, dim3((unsigned)((total_rows + kCdfWaves - 1) / kCdfWaves)),
                     dim3(64 * kCdfWaves), 0, s, jobs, n_jobs, total_rows, precision);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_build_rows_batched, dim3((unsigned)total_rows), dim3(128), 0, s, jobs, n_jobs);
  return hipGetLastError();
}

hipError_t launch_build_rows(const float* cdf, const float* Es, int nE, int nW, uint8_t* rows, hipStream_t s) {
  const int narrow = nW - 1 <= 255;
  hipLaunchKernelGGL(k_build_rows, dim3(nE), dim3(128), 0, s, cdf, Es, nE, nW, narrow, rows);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// pick-table nodes: FP64 sorted cumulative probabilities, ln mfp, labels.
// The table's (zeroed) summary follows the last node.
__global__ void k_pick_nodes(DevCfg c, int n_nodes, double lnE0, double dln, float* nodes, int stride) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n_nodes) return;
  double lnE = k == n_nodes - 1 ? log(c.E0) : lnE0 + k * dln;
  double E = k == n_nodes - 1 ? c.E0 : (k == 0 ? c.Emin : exp(lnE));
  double sig[MCD_MAX_CHANNELS], probs[MCD_MAX_CHANNELS];
  int lab[MCD_MAX_CHANNELS], order[MCD_MAX_CHANNELS];
  const int n = d_sigma_set(E, c, sig, lab);
  double s = 0.;
  for (int i = 0; i < n; ++i) s += sig[i];
  d_sorted_probs(sig, n, order, probs);
  // Zero-probability channels are never picked, so their labels are free:
  // order them by rising threshold so that a channel switching on at its
  // threshold keeps its position and the cell needs no reordering.
  int nz = 0;
  while (nz < n && sig[order[nz]] > 0.) ++nz;
  double thr[MCD_MAX_CHANNELS];
  for (int i = 0; i < n; ++i) {
    const int l = lab[i];
    thr[i] = l == MCD_CH_MOLLER ? c.Wc : (l == MCD_CH_QUINN ? c.Epl : (l >= MCD_CH_GRYZ0 ? c.Eb[l - MCD_CH_GRYZ0] : 0.));
  }
  for (int i = nz + 1; i < n; ++i) {
    int v = order[i], j = i - 1;
    while (j >= nz && thr[order[j]] > thr[v]) { order[j + 1] = order[j]; --j; }
    order[j + 1] = v;
  }
  float* o = nodes + (size_t)k * stride;
  for (int i = 0; i < n - 1; ++i) o[i] = (float)probs[i];
  o[n - 1] = (float)log2(1. / (c.atnd * s) * 1e14 * M_LN2);  // log2(mfp ln 2)
  uint32_t lo = 0, hi = 0;
  for (int i = 0; i < n; ++i) {
    uint32_t l = (uint32_t)lab[order[i]];
    if (i < 8) lo |= l << (4 * i); else hi |= l << (4 * (i - 8));
  }
  o[n] = __uint_as_float(lo);
  o[n + 1] = __uint_as_float(hi | (kMetaNoSwap << 12));
  for (int i = n + 2; i < stride; ++i) o[i] = 0.f;
  if (k == 0) *reinterpret_cast<PickSummary*>(nodes + (size_t)n_nodes * stride) = PickSummary{0u, 0, 0};
}

// The kind of cell k (node k to k + 1): the same order of the channels at both
// ends, two neighbours swapped, or exact (any other reordering, a NaN node).
__global__ void k_pick_cells(int n_nodes, int n_ch, float* nodes, int stride) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k + 1 >= n_nodes) return;
  float* a = nodes + (size_t)k * stride;
  const float* b = a + stride;
  auto label = [n_ch](const float* node, int pos) {
    return (__float_as_uint(node[n_ch + (pos >> 3)]) >> (4 * (pos & 7))) & 15u;
  };
  int ndiff = 0, first = -1;
  for (int q = 0; q < n_ch; ++q)
    if (label(a, q) != label(b, q)) {
      if (first < 0) first = q;
      ++ndiff;
    }
  uint32_t swap = kMetaNoSwap;
  bool exact = false;
  if (ndiff == 2 && first + 1 < n_ch && label(a, first) == label(b, first + 1) && label(a, first + 1) == label(b, first))
    swap = (uint32_t)first;
  else if (ndiff != 0)
    exact = true;
  for (int q = 0; q < stride; ++q)
    if (!(a[q] == a[q])) exact = true;
  const uint32_t hi = (__float_as_uint(a[n_ch + 1]) & 0xFFFu) | (swap << 12) | (exact ? kMetaExact : 0u);
  a[n_ch + 1] = __uint_as_float(hi);
  PickSummary* sum = reinterpret_cast<PickSummary*>(nodes + (size_t)n_nodes * stride);
  if (swap != kMetaNoSwap) atomicAdd(&sum->n_swap, 1);
}

hipError_t launch_pick_nodes(const DevCfg& c, int n_nodes, double lnE0, double dln, float* nodes, int stride,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_pick_nodes, dim3((n_nodes + 63) / 64), dim3(64), 0, s, c, n_nodes, lnE0, dln, nodes, stride);
  hipLaunchKernelGGL(k_pick_cells, dim3((n_nodes + 63) / 64), dim3(64), 0, s, n_nodes, c.n_shells + 3, nodes, stride);
  return hipGetLastError();
}

// Check points t = (m + 0.5)/16 inside every cell: compare the FP32
// interpolation (the transport's own f_pick_eval) with the exact FP64 order and
// cumulative probabilities.  err = max boundary error, err_ab = error of pA - pB
// in swap cells; bad = order mismatch not explained by the swap.
template <int NCH>
__device__ __forceinline__ void pick_point(const DevCfg& c, int k, int m, float& err, float& err_ab, bool& bad) {
  const int ncell = c.pick.n_nodes - 1;
  const double lnE0 = log(c.Emin);
  const double lnE = lnE0 + ((double)k + ((double)m + 0.5) / (double)kPickChecks) * (log(c.E0) - lnE0) / (double)ncell;
  const double E = exp(lnE);
  PickEval<NCH> o;
  f_pick_eval<NCH>(c.pick.nodes, c.pick, (float)E, o);
  err = 0.f;
  err_ab = 0.f;
  bad = false;
  if (o.exact) return;
  double sig[MCD_MAX_CHANNELS], probs[MCD_MAX_CHANNELS];
  int lab[MCD_MAX_CHANNELS], order[MCD_MAX_CHANNELS];
  const int n = d_sigma_set(E, c, sig, lab);
  d_sorted_probs(sig, n, order, probs);
  // last position with non-zero probability
  int last = 0;
  for (int q = 0; q < n; ++q)
    if (sig[order[q]] > 0.) last = q;
  float eb = 0.f;
  int mism = 0;
  for (int q = 0; q <= last; ++q) {
    if (perm_label(o.perm_lo, o.perm_hi, q) != lab[order[q]]) mism = 1;
  }
  for (int q = 0; q < NCH - 1; ++q) eb = fmaxf(eb, fabsf((float)((double)o.B[q] - probs[q])));
  if (o.swap != (int)kMetaNoSwap) {
    const int j = o.swap;
    // true probabilities of the node-k position-j (A) and j+1 (B) channels
    uint32_t la = (uint32_t)perm_label(__float_as_uint(c.pick.nodes[(size_t)k * c.pick.stride + NCH]),
                                       __float_as_uint(c.pick.nodes[(size_t)k * c.pick.stride + NCH + 1]) & 0xFFFu, j);
    uint32_t lb = (uint32_t)perm_label(__float_as_uint(c.pick.nodes[(size_t)k * c.pick.stride + NCH]),
                                       __float_as_uint(c.pick.nodes[(size_t)k * c.pick.stride + NCH + 1]) & 0xFFFu,
                                       j + 1);
    double s = 0., sa = 0., sb = 0.;
    for (int q = 0; q < n; ++q) {
      s += sig[q];
      if ((uint32_t)lab[q] == la) sa = sig[q];
      if ((uint32_t)lab[q] == lb) sb = sig[q];
    }
    const double dtrue = (sa - sb) / s;
    err_ab = fabsf((float)((double)(o.pA - o.pB) - dtrue));
    if (mism) {
      // allowed only when the two orders differ by the swap itself (then the
      // guard must catch it: the boundary error at j is not meaningful)
      int other = 0;
      for (int q = 0; q <= last; ++q)
        if (q != j && q != j + 1 && perm_label(o.perm_lo, o.perm_hi, q) != lab[order[q]]) other = 1;
      mism = other;
      float eb2 = 0.f;
      for (int q = 0; q < NCH - 1; ++q)
        if (q != j) eb2 = fmaxf(eb2, fabsf((float)((double)o.B[q] - probs[q])));
      eb = eb2;
    }
  }
  err = eb;
  bad = mism != 0;
}

// The cells' verdicts, behind the summary.
__device__ __forceinline__ uint8_t* pick_verdicts(float* nodes, int n_nodes, int stride) {
  return reinterpret_cast<uint8_t*>(nodes + (size_t)n_nodes * stride) + sizeof(PickSummary);
}

// 16 lanes to a cell.  A cell with a bad point, or an error that is NaN or above
// 1e-4 (badly resolved), becomes exact; the largest error of the others is the
// table's.  In cells a few ulp of ln E wide a point can fall into a neighbour
// (8192 nodes from 1000 to 1100 eV: 1 % of them), so the cells stay as they are
// until every point is checked (k_pick_exact).
template <int NCH>
__global__ __launch_bounds__(64) void k_pick_check(DevCfg c, float* nodes) {
  static_assert(kPickChecks == 16, "16 lanes share a cell");
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = i / kPickChecks, m = i % kPickChecks;
  if (k >= c.pick.n_nodes - 1) return;
  float err, err_ab;
  bool bad;
  pick_point<NCH>(c, k, m, err, err_ab, bad);
  bad = bad || !(err == err) || !(err_ab == err_ab);
  float ek = fmaxf(0.f, fmaxf(err, err_ab));
#pragma unroll
  for (int off = 1; off < kPickChecks; off <<= 1) ek = fmaxf(ek, __shfl_xor(ek, off));
  const uint64_t any_bad = (__ballot(bad) >> ((threadIdx.x & 63) & ~(kPickChecks - 1))) & 0xFFFFull;
  if (m) return;
  PickSummary* sum = reinterpret_cast<PickSummary*>(nodes + (size_t)c.pick.n_nodes * c.pick.stride);
  const uint32_t hi = __float_as_uint(nodes[(size_t)k * c.pick.stride + NCH + 1]);
  const bool exact = (hi & kMetaExact) || any_bad || (double)ek > 1e-4;
  pick_verdicts(nodes, c.pick.n_nodes, c.pick.stride)[k] = exact;
  if (exact) atomicAdd(&sum->n_exact, 1);
  else atomicMax(&sum->max_err, __float_as_uint(ek));
}

__global__ void k_pick_exact(int n_nodes, int n_ch, float* nodes, int stride) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k + 1 >= n_nodes || !pick_verdicts(nodes, n_nodes, stride)[k]) return;
  float* meta = nodes + (size_t)k * stride + n_ch + 1;
  *meta = __uint_as_float(__float_as_uint(*meta) | kMetaExact);
}

hipError_t launch_pick_check(const DevCfg& c, float* nodes, hipStream_t s) {
  const dim3 g(((c.pick.n_nodes - 1) * kPickChecks + 63) / 64), b(64);
  switch (c.n_shells + 3) {
    case 4: hipLaunchKernelGGL(k_pick_check<4>, g, b, 0, s, c, nodes); break;
    case 5: hipLaunchKernelGGL(k_pick_check<5>, g, b, 0, s, c, nodes); break;
    case 6: hipLaunchKernelGGL(k_pick_check<6>, g, b, 0, s, c, nodes); break;
    case 7: hipLaunchKernelGGL(k_pick_check<7>, g, b, 0, s, c, nodes); break;
    case 8: hipLaunchKernelGGL(k_pick_check<8>, g, b, 0, s, c, nodes); break;
    case 9: hipLaunchKernelGGL(k_pick_check<9>, g, b, 0, s, c, nodes); break;
    case 10: hipLaunchKernelGGL(k_pick_check<10>, g, b, 0, s, c, nodes); break;
    case 11: hipLaunchKernelGGL(k_pick_check<11>, g, b, 0, s, c, nodes); break;
    default: return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(k_pick_exact, dim3((c.pick.n_nodes + 63) / 64), dim3(64), 0, s, c.pick.n_nodes, c.n_shells + 3,
                     nodes, c.pick.stride);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
__global__ void k_fill_u64(unsigned long long* p, unsigned long long v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

hipError_t launch_fill_u64(unsigned long long* p, unsigned long long v, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_u64, dim3((n + 63) / 64), dim3(64), 0, s, p, v, n);
  return hipGetLastError();
}

// masked sentinel -> 0 (the reference's stored layout), or 0 -> sentinel
__global__ void k_unmask(const float* __restrict__ src, float* __restrict__ dst, size_t n, int to_reference) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float v = src[i];
  if (to_reference) dst[i] = v == kMasked ? 0.f : v;
  else dst[i] = v == 0.f ? kMasked : v;
}

hipError_t launch_unmask(const float* src, float* dst, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_unmask, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, dst, n, 1);
  return hipGetLastError();
}

hipError_t launch_mask(const float* src, float* dst, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_unmask, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, dst, n, 0);
  return hipGetLastError();
}

}  // namespace mcd
