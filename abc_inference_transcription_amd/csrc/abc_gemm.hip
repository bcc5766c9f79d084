// abc_gemm.hip -- particle x gene error screening on MFMA (split-BF16) with
// exact FP64 rescoring, the acceptance path of scripts/compute_errors.jl:30-70
// and scripts/accepted_particles.jl:12-32.
//
// err(i,g) = sum_k W_gk (d_gk - s_ik)^2 = c_g + sum_k s_ik (-2 W_gk d_gk) + sum_k s_ik^2 W_gk
// with W_gk = 1 / (K (se^2 + 0.01 d^2 + eps)) and c_g = sum_k W_gk d_gk^2.
// The two sums are one GEMM of A = [S | S^2] (n x 2K) with B = [-2WD ; W]
// (2K x G).  Every operand x is split x = hi + lo (two bf16) and the product
// uses hi*hi + hi*lo + lo*hi with FP32 accumulation on the matrix cores.
//
// Error bound (per element): |a*b - (ah*bh + ah*bl + al*bh)| <= 3.02*2^-16 |a||b|
// and FP32 accumulation of 3*Kp products adds <= 3*Kp*2^-24 sum|terms|; with
// Kp <= 128 both stay below DELTA = 2^-12 of sum_k |a_k||b_k|.  By
// Cauchy-Schwarz over W >= 0:  sum_k |a_k||b_k| <= 2 sqrt(y c) + y, where
// y = sum_k W s^2 is the second accumulator.  A pair is a candidate whenever
// its lower bound can reach the gene's threshold; candidates are rescored in
// FP64 in the reference order, so the accepted sets equal the FP64 ones.
#include <hip/hip_runtime.h>

#include "abc_kernels.h"

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SCREEN_DELTA 2.44140625e-4  // 2^-12
#define SCREEN_LIMIT 1e15           // operands beyond this go straight to FP64

__device__ __forceinline__ void split_bf16(double x, bf16* hi, bf16* lo) {
  const bf16 h = (bf16)(float)x;
  const double r = x - (double)(float)h;
  *hi = h;
  *lo = (bf16)(float)r;
}

// Both prep kernels: a workgroup makes the operand rows of 16 genes or
// particles, thread (p, q) the statistics k = q, q + 16, ... of row p.  The
// statistics of 16 neighbours are 128 consecutive bytes, the 16 finished rows
// one contiguous block of MFMA operands (32 statistics of all 16 rows, then the
// next 32, each as its 64 lanes' 16 bytes): they are staged in LDS (an odd
// number of words per row against bank conflicts) and written out word by word.
// Bound by memory; a
// thread per row, as before, wrote two bytes every row length: 4,096 particles
// x 90 statistics 87 -> 6 us, 2,000 genes x 90 110 -> 10 us.
#define PREP_ROWS 16
#define PREP_MAXK 128
typedef unsigned short u16;

__device__ __forceinline__ void stage_split(u16* hi, u16* lo, double x) {
  bf16 h, l;
  split_bf16(x, &h, &l);
  *hi = __builtin_bit_cast(u16, h);
  *lo = __builtin_bit_cast(u16, l);
}

// rows of W words (staged with a stride of W + 1) to the operands' block: lane l
// of operand t holds k = 32 t + (l / 16) 8 .. + 7 of row l % 16, four words
__device__ __forceinline__ void store_rows(const u16* st, int W, uint32_t* __restrict__ out) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(st);
  for (int q = threadIdx.x; q < PREP_ROWS * W; q += 256) {
    const int l = (q >> 2) & 63;
    out[q] = w[(l & 15) * (W + 1) + (q >> 8) * 16 + (l >> 4) * 4 + (q & 3)];
  }
}

// B's operands (of Bt[g][k], 2*Kp per gene), c_g, the operands of the FP64
// rescoring, and flags for genes whose weights leave the screened range (1) or
// whose operands leave div_by's (2).  Rows of genes G .. Gpad - 1 are zero.
__global__ __launch_bounds__(256) void gene_prep_kernel(const double* __restrict__ data,
                                                        const double* __restrict__ se, int64_t G,
                                                        int K, int Kp, int64_t Gpad,
                                                        bf16* __restrict__ Bh,
                                                        bf16* __restrict__ Bl,
                                                        double* __restrict__ cg,
                                                        uint8_t* __restrict__ gflag,
                                                        float* __restrict__ Wf,
                                                        ErrGene* __restrict__ genes) {
  __shared__ u16 sh[PREP_ROWS * (2 * PREP_MAXK + 2)], sl[PREP_ROWS * (2 * PREP_MAXK + 2)];
  __shared__ double s_c[PREP_MAXK][PREP_ROWS];
  __shared__ unsigned s_flag[PREP_ROWS];
  const int p = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int64_t g0 = (int64_t)blockIdx.x * PREP_ROWS, g = g0 + p;
  if (threadIdx.x < PREP_ROWS) s_flag[threadIdx.x] = 0u;
  __syncthreads();
  unsigned flag = 0u;
  u16* rh = sh + p * (2 * Kp + 2);
  u16* rl = sl + p * (2 * Kp + 2);
  for (int k = q; k < Kp; k += 16) {
    double b1 = 0.0, b2 = 0.0;
    if (g < G && k < K) {
      const double d = data[g + G * k];
      const double den = err_den(d, se[g + G * k]);
      const double W = 1.0 / ((double)K * den);
      const double WD = W * d;
      s_c[k][p] = WD * d;
      const Divisor v = divisor_of(den);
      genes[g * K + k] = ErrGene{d, v.y, v.zh, v.zl};
      if (!gene_range(d, den)) flag |= 2u;
      if (!(fabs(W) <= SCREEN_LIMIT) || !(fabs(WD) <= SCREEN_LIMIT)) flag |= 1u;
      Wf[g + G * k] = (float)W;
      b1 = -2.0 * WD;
      b2 = W;
    }
    stage_split(rh + k, rl + k, b1);
    stage_split(rh + Kp + k, rl + Kp + k, b2);
  }
  if (flag) atomicOr(&s_flag[p], flag);
  __syncthreads();
  store_rows(sh, Kp, reinterpret_cast<uint32_t*>(Bh + g0 * 2 * Kp));
  store_rows(sl, Kp, reinterpret_cast<uint32_t*>(Bl + g0 * 2 * Kp));
  if (q == 0 && g < G) {
    double c = 0.0;  // in the order of k
    for (int k = 0; k < K; ++k) c += s_c[k][p];
    cg[g] = c;
    gflag[g] = (uint8_t)(s_flag[p] | (!(c <= SCREEN_LIMIT) ? 1u : 0u));
  }
}

// A's operands, rows [s | s^2] split into bf16 hi/lo, and flags as gene_prep_kernel's.  Row
// i of the n rows is stats[i + ld * k] (a block of rows of a larger batch);
// rows n .. npad - 1 are zero, and so is a row from its first statistic beyond
// the screened range on.
__global__ __launch_bounds__(256) void particle_prep_kernel(const double* __restrict__ stats,
                                                            int64_t n, int64_t ld, int K, int Kp,
                                                            int64_t npad,
                                                            bf16* __restrict__ Ah,
                                                            bf16* __restrict__ Al,
                                                            uint8_t* __restrict__ pflag) {
  __shared__ u16 sh[PREP_ROWS * (2 * PREP_MAXK + 2)], sl[PREP_ROWS * (2 * PREP_MAXK + 2)];
  __shared__ int s_first[PREP_ROWS];     // first statistic beyond the screened range
  __shared__ unsigned s_odd[PREP_ROWS];
  const int p = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int64_t i0 = (int64_t)blockIdx.x * PREP_ROWS, i = i0 + p;
  if (threadIdx.x < PREP_ROWS) {
    s_first[threadIdx.x] = PREP_MAXK;
    s_odd[threadIdx.x] = 0u;
  }
  __syncthreads();
  double v[PREP_MAXK / 16];
#pragma unroll
  for (int c = 0; c < PREP_MAXK / 16; ++c) {
    const int k = q + 16 * c;
    v[c] = i < n && k < K ? stats[i + ld * k] : 0.0;
    if (!(fabs(v[c]) <= SCREEN_LIMIT)) atomicMin(&s_first[p], k);
    if (!err_range(v[c])) s_odd[p] = 1u;
  }
  __syncthreads();
  const int first = s_first[p];
  u16* rh = sh + p * (2 * Kp + 2);
  u16* rl = sl + p * (2 * Kp + 2);
#pragma unroll
  for (int c = 0; c < PREP_MAXK / 16; ++c) {
    const int k = q + 16 * c;
    if (k >= Kp) continue;
    const double s = k < first ? v[c] : 0.0;
    stage_split(rh + k, rl + k, s);
    stage_split(rh + Kp + k, rl + Kp + k, s * s);
  }
  __syncthreads();
  store_rows(sh, Kp, reinterpret_cast<uint32_t*>(Ah + i0 * 2 * Kp));
  store_rows(sl, Kp, reinterpret_cast<uint32_t*>(Al + i0 * 2 * Kp));
  if (q == 0 && i < n) pflag[i] = (uint8_t)((first < PREP_MAXK ? 1u : 0u) | (s_odd[p] ? 2u : 0u));
}

// 256 threads = 4 waves; the workgroup covers 64 particles x 64 genes, each
// wave a 32 x 32 block as 2 x 2 MFMA 16x16x32 tiles.  Lane layout of
// v_mfma_f32_16x16x32_bf16: A lane l holds row l%16, k = (l/16)*8 .. +7;
// B lane l holds column l%16, the same k; D lane l holds column l%16,
// rows (l/16)*4 .. +3.  The operands lie in that order, 1 KB per
// load: 20,480 particles x 3,419 genes of 53 statistics 338 us row by row (16
// pieces of 64 bytes a load), 223 so.
__global__ __launch_bounds__(256) void gemm_screen_kernel(
    const bf16* __restrict__ Ah, const bf16* __restrict__ Al, int64_t n, int Kp,
    const bf16* __restrict__ Bh, const bf16* __restrict__ Bl, int64_t G,
    const double* __restrict__ cg, const uint8_t* __restrict__ gflag,
    const uint8_t* __restrict__ pflag, const double* __restrict__ thr, double margin_rel,
    double clamp, Candidate* __restrict__ out, unsigned long long* __restrict__ count,
    unsigned long long cap, float* __restrict__ approx_out, float* __restrict__ bound_out,
    PoolEntry* __restrict__ pool, int64_t capg, uint32_t* __restrict__ pool_n) {
  __shared__ unsigned s_tot[4];
  __shared__ unsigned long long s_base;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t i0 = (int64_t)blockIdx.x * 64 + (wave >> 1) * 32;
  const int64_t g0 = (int64_t)blockIdx.y * 64 + (wave & 1) * 32;
  const int nt = Kp / 16;  // operands per 16 rows: 2 Kp / 32
  f32x4 accC[2][2], accS[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      accC[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      accS[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  const int nchunk = Kp / 32;
  // cross half (k < Kp) into accC, square half (k >= Kp) into accS
  auto chunk = [&](f32x4 (&acc)[2][2], int t) {
    bf16x8 ah[2], al[2], bh[2], bl[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t o = ((i0 / 16 + rb) * nt + t) * 512 + lane * 8;
      ah[rb] = *reinterpret_cast<const bf16x8*>(Ah + o);
      al[rb] = *reinterpret_cast<const bf16x8*>(Al + o);
    }
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int64_t o = ((g0 / 16 + cb) * nt + t) * 512 + lane * 8;
      bh[cb] = *reinterpret_cast<const bf16x8*>(Bh + o);
      bl[cb] = *reinterpret_cast<const bf16x8*>(Bl + o);
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[rb], bh[cb], acc[rb][cb], 0, 0, 0);
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[rb], bl[cb], acc[rb][cb], 0, 0, 0);
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[rb], bh[cb], acc[rb][cb], 0, 0, 0);
      }
  };
  for (int ch = 0; ch < nchunk; ++ch) chunk(accC, ch);
  for (int ch = 0; ch < nchunk; ++ch) chunk(accS, nchunk + ch);
  // epilogue: bounds, thresholds, candidate emission.  A pair is a candidate
  // unless its lower bound provably exceeds the gene's threshold; a
  // non-finite approximation or bound (FP32 overflow) makes it one.
  unsigned cm[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int64_t g = g0 + cb * 16 + (lane & 15);
    const bool gok = g < G;
    const double c = gok ? cg[g] : 0.0;
    const double t = gok ? thr[g] : 0.0;
    const bool gbad = gok && (gflag[g] & 1) != 0;
    unsigned cmask = 0;  // bit rb * 4 + q: row i0 + rb * 16 + (lane >> 4) * 4 + q
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t i = i0 + rb * 16 + (lane >> 4) * 4 + q;
        if (!gok || i >= n) continue;
        const double cross = (double)accC[rb][cb][q];
        const double sq = (double)accS[rb][cb][q];
        const double approx = (c + cross) + sq;
        const double y = fmax(sq, 0.0) * (1.0 + 2.0 * SCREEN_DELTA) + 1e-30;
        const double bound = SCREEN_DELTA * (2.0 * sqrt(y * fmax(c, 0.0)) + y) +
                             1e-12 * fabs(approx) + 1e-30;
        if (approx_out) {
          approx_out[i + n * g] = (float)approx;
          bound_out[i + n * g] = (float)bound;
        }
        double lo = approx - bound;
        if (t < 1e300) lo -= margin_rel * fabs(t);
        if (lo > clamp) lo = clamp;
        const bool must = (pflag[i] & 1) != 0 || gbad;
        if (must || !(lo > t)) cmask |= 1u << (rb * 4 + q);
      }
    cm[cb] = cmask;
    if (pool) {
      // lanes l, l + 16, l + 32, l + 48 hold the same gene: one atomic per
      // gene and wave reserves their pool slots
      const int col = lane & 15, rgrp = lane >> 4;
      const unsigned cnt = (unsigned)__popc(cmask);
      const unsigned c0 = __shfl(cnt, col), c1 = __shfl(cnt, col + 16),
                     c2 = __shfl(cnt, col + 32), c3 = __shfl(cnt, col + 48);
      const unsigned tot = c0 + c1 + c2 + c3;
      const unsigned pre = (rgrp > 0 ? c0 : 0u) + (rgrp > 1 ? c1 : 0u) + (rgrp > 2 ? c2 : 0u);
      unsigned base = 0;
      if (rgrp == 0 && tot > 0) base = atomicAdd(pool_n + g, tot);
      base = __shfl(base, col);
      int64_t slot = (int64_t)base + pre;
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        if (!(cmask & (1u << bit))) continue;
        const int64_t i = i0 + (bit >> 2) * 16 + (lane >> 4) * 4 + (bit & 3);
        if (slot < capg) pool[g * capg + slot] = PoolEntry{0.0, i};
        slot++;
      }
    }
  }
  if (!pool && out) {
    // one atomic per workgroup reserves the list slots of its candidates (one
    // per candidate bit had set the kernel's time: 20,480 particles x 3,419
    // genes 1,409 -> 329 us)
    const unsigned mine = (unsigned)(__popc(cm[0]) + __popc(cm[1]));
    unsigned inc = mine;
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned y = __shfl_up(inc, o);
      if (lane >= o) inc += y;
    }
    if (lane == 63) s_tot[wave] = inc;
    __syncthreads();
    const unsigned w0 = s_tot[0], w1 = s_tot[1], w2 = s_tot[2], w3 = s_tot[3];
    if (threadIdx.x == 0 && w0 + w1 + w2 + w3 > 0)
      s_base = atomicAdd(count, (unsigned long long)(w0 + w1 + w2 + w3));
    __syncthreads();
    unsigned long long slot = s_base + (wave > 0 ? w0 : 0u) + (wave > 1 ? w1 : 0u) +
                              (wave > 2 ? w2 : 0u) + (inc - mine);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int64_t g = g0 + cb * 16 + (lane & 15);
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        if (!(cm[cb] & (1u << bit))) continue;
        const int64_t i = i0 + (bit >> 2) * 16 + (lane >> 4) * 4 + (bit & 3);
        if (slot < cap) out[slot] = Candidate{0.0, i, (int32_t)g, 0};
        slot++;
      }
    }
  }
}

// FP64 rescoring of the batch's *count candidates, those of [q0, q1), in the
// reference operation order (compute_errors.jl:30-64); those with err <=
// eps_acc join the session's accepted pairs acc[0 .. *n_acc), counted per gene.
// With more candidates than cap the batch is screened again, so nothing is
// accepted; pairs past room are counted and not stored.  Candidate.particle
// holds the batch-local row on entry, the global particle index (pidx[row], or
// first_index + row) in acc.
__global__ __launch_bounds__(256) void rescore_kernel(const double* __restrict__ stats, int64_t n,
                                                      const double* __restrict__ data,
                                                      const double* __restrict__ se, int64_t G,
                                                      ErrSpec E,
                                                      const Candidate* __restrict__ cand,
                                                      const unsigned long long* __restrict__ count,
                                                      unsigned long long cap, int64_t q0, int64_t q1,
                                                      double eps_acc, int64_t first_index,
                                                      const int64_t* __restrict__ pidx,
                                                      Candidate* __restrict__ acc,
                                                      unsigned long long room,
                                                      unsigned long long* __restrict__ n_acc,
                                                      uint32_t* __restrict__ gene_n) {
  const unsigned long long q = q0 + (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned long long m = *count;
  if (m > cap || q >= m || q >= (unsigned long long)q1) return;
  Candidate c = cand[q];
  const int64_t i = c.particle, g = c.gene;
  const double s2 = 0.1 * 0.1;
  double err = 0.0;
  int k = 0;
  for (int pp = 0; pp < E.n_parts; ++pp) {
    double e = 0.0;
    const int end = k + E.parts[pp];
    for (; k < end; ++k) {
      const double d = data[g + G * k];
      const double sg = se[g + G * k];
      const double s = stats[i + n * k];
      const double eps = (sg + d != 0.0) ? 0.0 : 0.0001;
      const double diff = d - s;
      e += (diff * diff) / ((sg * sg + s2 * (d * d)) + eps);
    }
    err += e / (double)E.K;
  }
  if (err > E.clamp) err = E.clamp;
  if (err <= eps_acc) {  // never for NaN
    c.err = err;
    c.particle = pidx ? pidx[i] : first_index + i;
    const unsigned long long at = atomicAdd(n_acc, 1ull);
    if (at < room) acc[at] = c;
    atomicAdd(gene_n + g, 1u);
  }
}
