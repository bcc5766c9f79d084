// abc_select.hip -- model probabilities with bootstrap bounds per gene, the
// step after acceptance (scripts/model_probs.jl:1-63, constant_model_probs.jl,
// non_constant_model_probs.jl: get_model_probs and its per-gene branches).
//
// With l_m accepted particles in model group m and S = sum l: no group
// accepted gives zeros, one group gives 1 for it, and otherwise prob = l / S
// and n_boot resamples of the S labels with replacement.  model_prob_kernel
// spreads a gene's resamples over workgroups (rpb each) and stores every
// resample's share of each group; model_prob_bounds_kernel sorts them and
// takes Julia's type-7 quantiles at 1 - alpha and alpha.
// Draw i of resample b of gene g uses Philox4x32-10 with key (seed_lo,
// seed_hi ^ 0x5851F42D) and counter (i / 2, b, g, 0), words (0,1) or (2,3) as
// a 64-bit u, and takes label floor(u * S / 2^64) (the reference samples from
// Julia's unseeded global RNG, so only the law can match).  Counts are
// integers and every floating-point step is fixed, so the result equals the
// CPU replay bit for bit whatever the launch shape.
#include "abc_device.h"
#include "abc_kernels.h"

using namespace abcd;

namespace {

ABC_DEV double jl_quantile_sorted(const double* v, int n, double p) {
  if (n == 1) return v[0];
  const double m = 1.0 - p;
  const double aleph = (double)n * p + m;
  int j = (int)aleph;
  if (j < 1) j = 1;
  if (j > n - 1) j = n - 1;
  double g = aleph - (double)j;
  if (g < 0.0) g = 0.0;
  if (g > 1.0) g = 1.0;
  const double a = v[j - 1], b = v[j];
  return a + g * (b - a);
}

}  // namespace

// Workgroup (x, y): gene g0 + x, resamples y * rpb .. y * rpb + rpb - 1, one
// wave per resample (four or two on the labels of one or two resamples); each
// resample's share of every group goes to shares[(x M + m) n_boot + b].  A gene
// with at most one accepting group is written here by y = 0.
// Bound by VALU issue: a label is half a Philox block and one 64-bit comparison
// per group boundary, 41 instructions per two labels of two groups.  A label idx = floor(u S / 2^64) reaches the
// cumulative count A (idx >= A) exactly when u >= ceil(A 2^64 / S), so the
// boundaries are scaled once per workgroup and the index, a 64 x 32
// multiply-high per label, is never formed; the comparisons are counted by
// scalar popcounts of their lane masks, the M - 1 counts in scalar registers.  2,000 genes,
// 2 groups, 29,500 resampled labels a gene on average, 100 resamples: the call 8.8 ->
// 3.7 ms, of the 3.1 that the instructions take at one a cycle and lane.
template <int M>
__global__ __launch_bounds__(ABC_SEL_WG) void model_prob_kernel(
    int64_t G, int64_t g0, const int64_t* __restrict__ counts, uint32_t k0, uint32_t k1,
    int n_boot, int rpb, double* __restrict__ shares, double* __restrict__ prob,
    double* __restrict__ lb, double* __restrict__ ub) {
  const int64_t gl = blockIdx.x, g = g0 + gl;
  const int tid = threadIdx.x;
  int64_t S = 0;
  int nz = 0, which = -1;
  // over[k] = ceil(A_k 2^64 / S) - 1 with A_k = l_0 + ... + l_k: a draw u
  // reaches A_k when u > over[k] (never when A_k = S; always when A_k = 0)
  uint64_t over[M];
  bool all[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int64_t l = counts[g + G * m];
    S += l;
    over[m] = (uint64_t)S;
    if (l > 0) {
      nz++;
      which = m;
    }
  }
  if (nz <= 1) {  // uniform over the workgroup
    if (blockIdx.y == 0 && tid < M) {
      const double v = tid == which ? 1.0 : 0.0;
      prob[g + G * tid] = v;
      lb[g + G * tid] = v;
      ub[g + G * tid] = v;
    }
    return;
  }
  const uint32_t S32 = (uint32_t)S;  // S < 2^32 (the caller checks it)
#pragma unroll
  for (int k = 0; k < M - 1; ++k) {
    const uint64_t A = over[k];
    all[k] = A == 0;
    if (A == (uint64_t)S) {
      over[k] = ~0ull;
    } else {
      const uint64_t n1 = A << 32, q1 = n1 / S32, n2 = (n1 - q1 * S32) << 32, q0 = n2 / S32;
      over[k] = ((q1 << 32) | q0) - (n2 - q0 * S32 == 0 ? 1ull : 0ull);
    }
  }
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b_lo = (int)blockIdx.y * rpb;
  const int b_hi = b_lo + rpb < n_boot ? b_lo + rpb : n_boot;
  const uint32_t full = S32 >> 1;  // whole blocks of two draws
  // waves per resample: more than one only where there are fewer resamples than waves
  const int share = b_hi - b_lo > 2 ? 1 : (b_hi - b_lo == 2 ? 2 : 4);
  const int piece = wave & (share - 1);
  __shared__ uint32_t s_r[ABC_SEL_WG / 64][M];
  for (int b = b_lo + wave / share; b < b_hi; b += ABC_SEL_WG / 64 / share) {
    uint32_t r[M];  // draws that reach A_k, uniform over the wave
#pragma unroll
    for (int k = 0; k < M; ++k) r[k] = 0u;
    auto count = [&](uint32_t q, bool in) {
      const u4 w = philox(q, (uint32_t)b, (uint32_t)g, 0u, k0, k1);
      const uint64_t ua = (uint64_t)w.y << 32 | w.x, ub_ = (uint64_t)w.w << 32 | w.z;
#pragma unroll
      for (int k = 0; k < M - 1; ++k)
        r[k] += (uint32_t)__popcll(__ballot(in && ua > over[k])) +
                (uint32_t)__popcll(__ballot(in && ub_ > over[k]));
    };
    // q0 is uniform: the counts stay in scalar registers
    auto draws = [&](uint32_t q0, uint32_t step) {
      for (; q0 + 64u <= full; q0 += step) count(q0 + (uint32_t)lane, true);
      if (q0 < full) count(q0 + (uint32_t)lane, q0 + (uint32_t)lane < full);
    };
    if (share == 1) draws(0u, 64u);  // a loop of its own: with a variable step, 2 % more
    else draws(64u * (uint32_t)piece, 64u * (uint32_t)share);
    if (piece == 0 && (S32 & 1u)) {  // the last draw of an odd number
      const u4 w = philox(full, (uint32_t)b, (uint32_t)g, 0u, k0, k1);
      const uint64_t ua = (uint64_t)w.y << 32 | w.x;
#pragma unroll
      for (int k = 0; k < M - 1; ++k) r[k] += ua > over[k] ? 1u : 0u;
    }
    if (share > 1) {  // the whole workgroup: every wave is at its only piece
      if (lane == 0)
#pragma unroll
        for (int k = 0; k < M; ++k) s_r[wave][k] = r[k];
      __syncthreads();
      if (piece == 0)
        for (int w = 1; w < share; ++w)
#pragma unroll
          for (int k = 0; k < M; ++k) r[k] += s_r[wave + w][k];
    }
    if (piece == 0 && lane == 0) {
      uint32_t reach = S32;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const uint32_t next = m < M - 1 ? (all[m] ? S32 : r[m]) : 0u;
        shares[(gl * M + m) * n_boot + b] = (double)(reach - next) / (double)S;
        reach = next;
      }
    }
  }
}

template __global__ void model_prob_kernel<1>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<2>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<3>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<4>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<5>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<6>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<7>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);
template __global__ void model_prob_kernel<8>(int64_t, int64_t, const int64_t*, uint32_t, uint32_t,
                                              int, int, double*, double*, double*, double*);

// One workgroup per gene g0 + x with two or more accepting groups: each
// group's n_boot shares in ascending order (value i goes to place #{j: x_j <
// x_i} + #{j < i: x_j == x_i}; shares are finite and non-negative, so this is
// the order of any sort), then prob and Julia's type-7 quantiles at 1 - alpha
// and alpha.
__global__ __launch_bounds__(ABC_SEL_WG) void model_prob_bounds_kernel(
    int64_t G, int64_t g0, int M, const int64_t* __restrict__ counts, int n_boot, double alpha,
    const double* __restrict__ shares, double* __restrict__ prob, double* __restrict__ lb,
    double* __restrict__ ub) {
  __shared__ double x[ABC_SEL_MAX_GROUPS * ABC_SEL_MAX_BOOT];
  __shared__ double srt[ABC_SEL_MAX_GROUPS * ABC_SEL_MAX_BOOT];
  const int64_t gl = blockIdx.x, g = g0 + gl;
  const int tid = threadIdx.x;
  int64_t S = 0;
  int nz = 0;
  for (int m = 0; m < M; ++m) {
    const int64_t v = counts[g + G * m];
    S += v;
    nz += v > 0 ? 1 : 0;
  }
  if (nz <= 1) return;  // written by model_prob_kernel
  const double* sh = shares + gl * M * (int64_t)n_boot;
  for (int i = tid; i < M * n_boot; i += ABC_SEL_WG) x[i] = sh[i];
  __syncthreads();
  for (int i = tid; i < M * n_boot; i += ABC_SEL_WG) {
    const int m = i / n_boot, k = i - m * n_boot;
    const double* col = x + m * n_boot;
    const double v = col[k];
    int rank = 0;
    for (int j = 0; j < n_boot; ++j) rank += (col[j] < v || (col[j] == v && j < k)) ? 1 : 0;
    srt[m * n_boot + rank] = v;
  }
  __syncthreads();
  if (tid < M) {
    const double* col = srt + tid * n_boot;
    prob[g + G * tid] = (double)counts[g + G * tid] / (double)S;
    lb[g + G * tid] = jl_quantile_sorted(col, n_boot, 1.0 - alpha);
    ub[g + G * tid] = jl_quantile_sorted(col, n_boot, alpha);
  }
}
