// abc_kernels.hip -- gfx950 kernels of the ABC simulation hot path.
//
//   prior_kernel ...... fix_params (scripts/abc_simulation.jl:3-11) and the
//                       config priors; one thread per particle
//   rates_kernel ...... log10 parameters -> per-particle rates, thinning
//                       bounds, periodic gene law, burn-in length, cost key
//                       (scripts/model.jl:1-43)
//   bucket_*, cell_* .. heaviest-first queue orders: particles for the burn-in,
//                       cells for the window
//   burn_kernel ....... burn-in of every cell (gene path + Poisson means of the
//                       unlabelled molecules) up to its labelling window; the
//                       stochastic counterpart of scripts/model.jl:114-142
//   ssa_kernel ........ persistent Gillespie simulation of the labelling
//                       window, one (cell, sub-lane) item per lane, lanes refill
//                       from a global item queue the moment their item ends
//                       (lane-level work stealing); replaces the moment ODE
//                       solves of scripts/model.jl:146-206
//   stats_kernel ...... per-particle statistics from observed cell counts with
//                       exact integer accumulation in LDS
//                       (scripts/abc_simulation.jl:23-46 semantics on cells,
//                       estimators of scripts/data_summary_statistics.jl)
//   err_fp64_kernel ... reference-order FP64 error matrix
//                       (scripts/compute_errors.jl:30-70)
#include "abc_kernels.h"

using namespace abcd;

// ------------------------------------------------------------------ layout
struct Layout {
  int n_kon, n_al, n_ga, o_kon, o_koff, o_al, o_ga, o_lam, o_spl, n_par;
};

__host__ __device__ inline Layout layout_of(int model, int nb) {
  Layout L;
  L.n_kon = model == 3 ? nb : 1;
  L.n_al = model == 4 ? nb : 1;
  L.n_ga = model == 5 ? nb : 1;
  L.o_kon = 0;
  L.o_koff = L.n_kon;
  L.o_al = L.o_koff + 1;
  L.o_ga = L.o_al + L.n_al;
  L.o_lam = L.o_ga + L.n_ga;
  L.o_spl = L.o_lam + 1;
  L.n_par = L.o_spl + 1;
  return L;
}

int abc_layout_n_params(int model, int nb) { return layout_of(model, nb).n_par; }

// ------------------------------------------------------------------- prior
struct PriorStream {
  uint32_t k0, k1, tag, pid;  // tag: 0xFF000000 | model, disjoint from every cell word
  int q;
  u4 w;
  ABC_DEV double next() {
    const int call = q >> 1, half = q & 1;
    if (half == 0) w = philox((uint32_t)call, 0u, tag, pid, k0, k1);
    q++;
    return half == 0 ? u01_53(w.x, w.y) : u01_53(w.z, w.w);
  }
  ABC_DEV double unif(double lo, double hi) {
    const double u = next();
    return lo + (hi - lo) * u;
  }
};

#define FC_LO (-0.698970004336018804786)
#define FC_HI (0.698970004336018804786)

__global__ __launch_bounds__(256) void prior_kernel(const DesignDev* __restrict__ D, int model,
                                                    uint32_t k0, uint32_t k1, uint32_t first,
                                                    int64_t n, double* __restrict__ theta) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int nb = D->nb;
  const Layout L = layout_of(model, nb);
  PriorStream s{k0, k1, 0xFF000000u | (uint32_t)model, first + (uint32_t)i, 0, u4{0, 0, 0, 0}};
  double* th = theta + i;  // column c at th[n * c]
  if (D->prior_mode == 0) {
    for (int c = 0; c < L.n_kon; ++c) th[n * (L.o_kon + c)] = s.unif(-3.0, 3.0);
    th[n * L.o_koff] = s.unif(-3.0, 3.0);
    for (int c = 0; c < L.n_al; ++c) th[n * (L.o_al + c)] = s.unif(-3.0, 3.0);
    for (int c = 0; c < L.n_ga; ++c) th[n * (L.o_ga + c)] = s.unif(-3.0, 2.0);
    th[n * L.o_lam] = s.unif(-0.7, 0.0);
    th[n * L.o_spl] = D->splice_log10;
  } else {
    const double kb = s.unif(-2.0, 2.0);
    if (L.n_kon > 1) {
      for (int c = 0; c < nb; ++c) th[n * (L.o_kon + c)] = kb + s.unif(FC_LO, FC_HI);
    } else {
      th[n * L.o_kon] = kb;
    }
    const double koff = s.unif(-3.0, 3.0);
    th[n * L.o_koff] = koff;
    const double bb = s.unif(-1.0, 3.0);
    if (L.n_al > 1) {
      for (int c = 0; c < nb; ++c) th[n * (L.o_al + c)] = (bb + s.unif(FC_LO, FC_HI)) + koff;
    } else {
      th[n * L.o_al] = bb + koff;
    }
    const double gb = s.unif(-2.0, 1.0);
    if (L.n_ga > 1) {
      for (int c = 0; c < nb; ++c) th[n * (L.o_ga + c)] = gb + s.unif(FC_LO, FC_HI);
    } else {
      th[n * L.o_ga] = gb;
    }
    th[n * L.o_lam] = s.unif(-0.7, 0.0);
    th[n * L.o_spl] = s.unif(-1.0, 2.0);
  }
}

// ------------------------------------------------------------------- rates
__global__ __launch_bounds__(256) void rates_kernel(const DesignDev* __restrict__ D, int model,
                                                    int64_t n, const double* __restrict__ theta,
                                                    PRates* __restrict__ R,
                                                    float* __restrict__ cost) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int nb = D->nb;
  const Layout L = layout_of(model, nb);
  const double T = D->T;
  const double h = T / (double)nb;
  PRates r;
  r.scaling = model != 2;
  r.step = model == 2 ? nb : 1;
  for (int j = 0; j < nb; ++j) {
    r.kon[j] = ex10(theta[i + n * (L.o_kon + (L.n_kon > 1 ? j : 0))]);
    r.koff[j] = ex10(theta[i + n * L.o_koff]);
    const double al = ex10(theta[i + n * (L.o_al + (L.n_al > 1 ? j : 0))]);
    r.amax[j] = r.scaling ? (al * (double)(nb + j + 1)) / (double)nb : al;
    r.gam[j] = ex10(theta[i + n * (L.o_ga + (L.n_ga > 1 ? j : 0))]);
  }
  r.bs = ex10(theta[i + n * L.o_spl]);
  for (int j = 0; j < nb; ++j) {
    r.ikon[j] = 1.0 / r.kon[j];
    r.ikoff[j] = 1.0 / r.koff[j];
    r.iku[j] = 1.0 / (r.gam[j] + r.bs);
    r.ikt[j] = 1.0 / r.gam[j];
  }
  const double lam = ex10(theta[i + n * L.o_lam]);
  r.thr_lam = (uint64_t)(lam * 4294967296.0);
  double pi;
  if (L.n_kon > 1) {
    double p = 0.0, E = 1.0;
    for (int j = 0; j < nb; ++j) {
      const double rr = r.kon[j] + r.koff[j];
      const double pj = r.kon[j] / rr;
      const double e = ex(-(rr * h));
      p = pj + (p - pj) * e;
      E = E * e;
    }
    pi = p / (1.0 - E);
  } else {
    pi = r.kon[0] / (r.kon[0] + r.koff[0]);
  }
  if (pi > 1.0) pi = 1.0;
  if (pi < 0.0) pi = 0.0;
  r.thr_pi = (uint64_t)(pi * 4294967296.0);
  double gsum = r.gam[0];
  for (int j = 1; j < nb; ++j) gsum = gsum + r.gam[j];
  const double s = 0.5 * ex(-(gsum * h));
  double S = 1.0;
  for (int q = 0; q < D->bmin; ++q) S = S * s;
  int B = D->bmin;
  while (S > D->burn_eps && B < D->bmax) { S = S * s; B++; }
  r.B = B;
  r.gene_varies = L.n_kon > 1;
  // Mean birth rate with the gene's activity (before capture): the per-cell
  // split below uses it with the operations of the CPU replay, since it
  // selects random streams.  The typical sub-lanes M of an average cell
  // (longest window, mean capture) only orders the burn-in's queue.
  double births = 0.0;
  for (int j = 0; j < nb; ++j) births = births + r.amax[j] * (r.kon[j] / (r.kon[j] + r.koff[j]));
  r.brate = births / (double)nb;
  int M = 1;
  if (D->split_target > 0.0) {
    const double est = ((r.brate * D->split_scale) * D->wmax) * 3.0;
    while (M < D->split_max && est > D->split_target * (double)M) M *= 2;
  }
  // Expected Philox draws per work item (a scheduling key only, never a
  // result): gene switches over the whole path + molecule events (births
  // times 1 + splicing + loss, a 1/M share) over about half the longest window.
  double sw = 0.0, obs = 0.0, loss = 0.0;
  for (int j = 0; j < nb; ++j) {
    const double pon = r.kon[j] / (r.kon[j] + r.koff[j]);
    sw += 2.0 * r.kon[j] * (1.0 - pon);
    const double b = r.amax[j] * pon * D->capture_mean;
    obs += b;
    loss += b * (r.bs / (r.bs + r.gam[j]) + 1.0);
  }
  r.swrate = (float)(sw / (double)nb);
  r.gmean = (float)(gsum / (double)nb);
  R[i] = r;
  cost[i] = (float)((sw / (double)nb) * T * ((double)B + 0.5) +
                    ((obs + loss) / ((double)nb * (double)M)) * (0.5 * D->wmax) + 4.0);
}

// -------------------------------------------------------------- queue order
// Particles enter the work queue heaviest first (longest-processing-time
// order) through a bucket sort of the expected cost on its float exponent and
// top two mantissa bits (quarter-octave buckets).  Order inside a bucket is
// whatever the atomics give: every random stream is keyed by particle, cell
// and sub-lane, never by queue position, so the order changes the schedule
// and nothing else.  These are plain kernels (no library sort, no memset
// node), so a simulate call can be captured in a HIP graph.
__device__ __forceinline__ int cost_bucket(float c) {
  const int k = (int)((__float_as_uint(c) >> 21) & 0x3FFu) - 127 * 4;  // 4*exponent + 2 bits
  return k < 0 ? 0 : (k > ABC_NBUCKET - 1 ? ABC_NBUCKET - 1 : k);
}

__global__ __launch_bounds__(256) void bucket_hist_kernel(const float* __restrict__ cost, int64_t n,
                                                          unsigned* __restrict__ hist) {
  __shared__ unsigned h[ABC_NBUCKET];
  for (int b = threadIdx.x; b < ABC_NBUCKET; b += blockDim.x) h[b] = 0u;
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&h[cost_bucket(cost[i])], 1u);
  __syncthreads();
  for (int b = threadIdx.x; b < ABC_NBUCKET; b += blockDim.x)
    if (h[b]) atomicAdd(&hist[b], h[b]);
}

// cursor[b] = number of particles in heavier buckets (launch: 1 x ABC_NBUCKET)
__global__ __launch_bounds__(ABC_NBUCKET) void bucket_scan_kernel(const unsigned* __restrict__ hist,
                                                                  unsigned* __restrict__ cursor) {
  __shared__ unsigned s[ABC_NBUCKET];
  const int t = threadIdx.x;
  const unsigned x = hist[ABC_NBUCKET - 1 - t];  // heaviest bucket first
  s[t] = x;
  __syncthreads();
  for (int d = 1; d < ABC_NBUCKET; d <<= 1) {
    const unsigned v = t >= d ? s[t - d] : 0u;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  cursor[ABC_NBUCKET - 1 - t] = s[t] - x;
}

__global__ __launch_bounds__(256) void bucket_scatter_kernel(const float* __restrict__ cost,
                                                             int64_t n, unsigned* __restrict__ cursor,
                                                             int32_t* __restrict__ order) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned pos = atomicAdd(&cursor[cost_bucket(cost[i])], 1u);
  order[pos] = (int32_t)i;
}

// Identity of the particles of one model in a multi-model batch: global
// particle index src[i] (first + i without src) and the model's tag
// (model << 24) for the cell word of its counters.
__global__ __launch_bounds__(256) void fill_ids_kernel(int64_t n, int64_t first,
                                                       const int64_t* __restrict__ src,
                                                       uint32_t mtag, int64_t* __restrict__ pidx,
                                                       uint32_t* __restrict__ mtags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    pidx[i] = src ? src[i] : first + i;
    mtags[i] = mtag;
  }
}

__global__ __launch_bounds__(256) void copy_u64_kernel(const unsigned long long* __restrict__ src,
                                                       unsigned long long* __restrict__ dst,
                                                       int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// ---------------------------------------------------------- cell queue order
// ssa_kernel takes the cells of all particles heaviest item first, through a
// counting sort on the key burn_kernel leaves per cell: bucket = 16 * (cost
// class of one of the cell's items, a quarter octave) + log2 of its sub-lanes
// M.  All cells of a bucket have the same M, so a queue position is found from
// the bucket tables alone: cell cbase + (q - ioff) / M, sub-lane (q - ioff) % M.
// What sets a launch's end is its last long item: a particle's items differ by
// their conditions' windows (0.5 to 28 h, a factor of 50 in events), which an
// order of whole particles left mixed.  ssa_kernel, five configured models:
// 353 ms in particle order with two items a claim, 335 ms in this order, 296 ms
// with claims by weight as well (5 x 1,024 particles); 1,068 -> 991 ms at
// 5 x 4,096; 56 -> 40 ms at 5 x 64, where the longest item sets the time.
// Ranks run from the heaviest bucket (rank 0 = bucket ABC_CELL_BUCKETS - 1).
__global__ __launch_bounds__(256) void cell_hist_kernel(const uint32_t* __restrict__ key,
                                                        int64_t cells,
                                                        unsigned* __restrict__ hist) {
  __shared__ unsigned h[ABC_CELL_BUCKETS];
  for (int b = threadIdx.x; b < ABC_CELL_BUCKETS; b += blockDim.x) h[b] = 0u;
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < cells;
       i += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&h[key[i] & (ABC_CELL_BUCKETS - 1)], 1u);
  __syncthreads();
  for (int b = threadIdx.x; b < ABC_CELL_BUCKETS; b += blockDim.x)
    if (h[b]) atomicAdd(&hist[b], h[b]);
}

// Bucket tables by rank (launch: 1 x ABC_CELL_BUCKETS): first cell and first
// item of the rank (T.ioff[ABC_CELL_BUCKETS]: all items), scatter cursors.
__global__ __launch_bounds__(ABC_CELL_BUCKETS) void cell_scan_kernel(
    const unsigned* __restrict__ hist, CellTables* __restrict__ T) {
  __shared__ unsigned sc[ABC_CELL_BUCKETS];
  __shared__ unsigned long long si[ABC_CELL_BUCKETS];
  const int t = threadIdx.x, id = ABC_CELL_BUCKETS - 1 - t;
  const unsigned x = hist[id];
  const unsigned long long it = (unsigned long long)x << (id & 15);
  sc[t] = x;
  si[t] = it;
  __syncthreads();
  for (int d = 1; d < ABC_CELL_BUCKETS; d <<= 1) {
    const unsigned a = t >= d ? sc[t - d] : 0u;
    const unsigned long long b = t >= d ? si[t - d] : 0ull;
    __syncthreads();
    sc[t] += a;
    si[t] += b;
    __syncthreads();
  }
  T->cbase[t] = sc[t] - x;
  T->cursor[t] = sc[t] - x;
  T->ioff[t] = si[t] - it;
  if (t == ABC_CELL_BUCKETS - 1) T->ioff[ABC_CELL_BUCKETS] = si[t];
  __shared__ double sd[ABC_CELL_BUCKETS];
  sd[t] = (double)it * ex(0x1.62e42fee00000p-1 * (2.0 + 0.25 * (id >> 4)));  // 4 draws in class 0
  for (int d = ABC_CELL_BUCKETS / 2; d > 0; d >>= 1) {
    __syncthreads();
    if (t < d) sd[t] += sd[t + d];
  }
  if (t == 0) T->draws = sd[0];
}

// Each workgroup places a tile of cells: ranks within the tile from LDS
// counters, one global atomic per bucket and tile, so the cells of a tile
// (mostly one or two particles) stay together inside a bucket.
__global__ __launch_bounds__(256) void cell_scatter_kernel(const uint32_t* __restrict__ key,
                                                           int64_t cells,
                                                           CellTables* __restrict__ T,
                                                           uint32_t* __restrict__ cellord) {
  constexpr int PER = ABC_CELL_TILE / 256;
  __shared__ unsigned h[ABC_CELL_BUCKETS];
  for (int b = threadIdx.x; b < ABC_CELL_BUCKETS; b += blockDim.x) h[b] = 0u;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * ABC_CELL_TILE;
  unsigned k[PER], at[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int64_t i = base + q * 256 + threadIdx.x;
    k[q] = i < cells ? key[i] & (ABC_CELL_BUCKETS - 1) : 0u;
    at[q] = i < cells ? atomicAdd(&h[k[q]], 1u) : 0u;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < ABC_CELL_BUCKETS; b += blockDim.x)
    if (h[b]) h[b] = atomicAdd(&T->cursor[ABC_CELL_BUCKETS - 1 - b], h[b]);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int64_t i = base + q * 256 + threadIdx.x;
    if (i < cells) cellord[h[k[q]] + at[q]] = (uint32_t)i;
  }
}

// ------------------------------------------------------- shared helpers
// Random streams of a cell: counter (draw_lo, draw_hi[15:0] | stream << 16,
// cell | model << 24, particle), key (seed_lo, seed_hi); stream 0 holds the
// set-up draws and the gene clock, stream 1 + sub the molecule events and
// division coins of sub-lane sub.
// time of grid edge k (edges every h = T / nb hours; edge nbB is t = 0)
__device__ __forceinline__ double grid_time(int64_t k, int64_t nbB, double h) {
  return (double)(k - nbB) * h;
}

__device__ __forceinline__ u4 draw(uint64_t ctr, uint32_t stream, uint32_t cell, uint32_t pid,
                                   uint32_t k0, uint32_t k1) {
  return philox((uint32_t)ctr, ((uint32_t)(ctr >> 32) & 0xFFFFu) | (stream << 16), cell, pid, k0, k1);
}

// ----- burn-in: before the labelling window molecules are never labelled and
// never act on the gene or on each other, so given the gene path the observed
// unspliced and spliced molecules alive at the window start are independent
// Poisson counts (births a Poisson process of rate alpha(t) beta / M while the
// gene is on; decay, splicing and halving at division thin every molecule
// independently; Jahnke & Huisinga, J. Math. Biol. 54, 2007).  The burn-in
// simulates the gene path only and carries the two Poisson means lu
// (unspliced: leave at gamma + splice) and lt (all: leave at gamma).

// E1 = int_0^D e^{-k(D-s)} ds, E2 = int_0^D s e^{-k(D-s)} ds, e = e^{-kD}, ik = 1/k
__device__ __forceinline__ void seg_int(double k, double ik, double D, double e, double& E1,
                                        double& E2) {
  const double x = k * D;
  if (x < 1e-3) {
    E1 = D * (1.0 - x * (0.5 - x * (1.0 / 6.0 - x * (1.0 / 24.0))));
    E2 = (D * D) * (0.5 - x * (1.0 / 6.0 - x * (1.0 / 24.0 - x * (1.0 / 120.0))));
  } else {
    E1 = (1.0 - e) * ik;
    E2 = (D - E1) * ik;
  }
}

// advance the Poisson means over [t, t + D]: birth rate c0 + c1 s while on;
// ku, kt are the exit rates (with reciprocals iku, ikt)
__device__ __forceinline__ void burn_accum(double& lu, double& lt, bool g, double c0, double c1,
                                           double ku, double iku, double kt, double ikt, double D) {
  if (!(D > 0.0)) return;
  // arguments <= 0 (D > 0, rates > 0): no NaN or overflow test
  double eu, et;
  ex_core2(-(ku * D), -(kt * D), eu, et);
  lu = lu * eu;
  lt = lt * et;
  if (g) {
    double E1u, E2u, E1t, E2t;
    seg_int(ku, iku, D, eu, E1u, E2u);
    seg_int(kt, ikt, D, et, E1t, E2t);
    lu = lu + (c0 * E1u + c1 * E2u);
    lt = lt + (c0 * E1t + c1 * E2t);
  }
}

// consecutive words of a sub-lane's molecule stream
struct WordSrc {
  u4 w;
  int i;  // next word; 4 = empty
  uint64_t& ctr;  // Philox blocks drawn so far on this stream
  uint32_t stream, cell, pid, k0, k1;
  __device__ uint32_t next() {
    if (i == 4) {
      w = draw(ctr++, stream, cell, pid, k0, k1);
      i = 0;
    }
    const uint32_t v = i == 0 ? w.x : (i == 1 ? w.y : (i == 2 ? w.z : w.w));
    i++;
    return v;
  }
};

// ln(k!) for integer-valued k >= 0: table below 10, Stirling series above
__device__ __forceinline__ double logfact(double kd, const LogEntry* lt) {
  if (kd < 10.0) return abc_logfact[(int)kd];
  const double x = kd + 1.0, ix = 1.0 / x, ix2 = ix * ix;
  return ((x - 0.5) * ln(x, lt) - x) +
         (0x1.d67f1c864beb5p-1 +
          ix * (1.0 / 12.0 - ix2 * (1.0 / 360.0 - ix2 * (1.0 / 1260.0 - ix2 * (1.0 / 1680.0)))));
}

// Poisson(mu): inversion below 10, else the transformed rejection method with
// squeeze (Hormann, Insurance: Math. Econ. 12, 1993), at most 1000 tries.
__device__ uint32_t poisson(WordSrc& src, double mu, const LogEntry* lt, const double* rk) {
  if (!(mu > 0.0)) return 0u;
  if (mu < 10.0) {
    // inversion: p_k = p_{k-1} * mu * RN(1/k) (rk: the table in LDS)
    const uint32_t w0 = src.next(), w1 = src.next();
    const double u = u01_53(w0, w1);
    double p = ex(-mu), F = p;
    uint32_t k = 0;
    while (u > F && k < 200u) {
      k++;
      p = (p * mu) * rk[k];
      F = F + p;
    }
    return k;
  }
  const double smu = ex(0.5 * ln(mu, lt));
  const double bb = 0.931 + 2.53 * smu, aa = -0.059 + 0.02483 * bb;
  const double vr = 0.9277 - 3.6224 / (bb - 2.0);
  for (int tries = 0; tries < 1000; ++tries) {
    const double U = u01_32(src.next()) - 0.5;
    const double V = u01_32(src.next());
    const double us = 0.5 - fabs(U);
    const double kd = floor(((2.0 * aa) / us + bb) * U + mu + 0.43);
    if (kd < 0.0) continue;
    if (us >= 0.07 && V <= vr) return (uint32_t)kd;
    if (us < 0.013 && V > us) continue;
    // rare: the envelope constant and ln(mu) are recomputed here (same bits)
    const double inva = 1.1239 + 1.1328 / (bb - 3.4);
    if ((ln(V, lt) + ln(inva, lt)) - ln(aa / (us * us) + bb, lt) <=
        (kd * ln(mu, lt) - mu) - logfact(kd, lt))
      return (uint32_t)kd;
  }
  return (uint32_t)floor(mu + 0.5);
}

// Set-up of cell c of particle p on its stream 0 (counter 0 ...): age and bin,
// the gene's state from its periodic stationary law, the capture efficiency.
struct CellSetup {
  double age, bc;
  int bin;
  bool g;
};

__device__ __forceinline__ CellSetup cell_setup(const DesignDev* __restrict__ D, const PRates* rp,
                                                int c, uint32_t cw, uint32_t pid, uint32_t k0,
                                                uint32_t k1,
                                                const double* __restrict__ betas,
                                                const int64_t* __restrict__ goff, uint64_t& gctr) {
  const double T = D->T;
  const int nb = D->nb, J = D->J;
  CellSetup o;
  const u4 w = draw(gctr++, 0u, cw, pid, k0, k1);
  if (D->age_mode == 1) {
    const double th = u01_53(w.x, w.y);
    o.age = th * T;
    o.bin = (int)(th * (double)nb);
    if (o.bin >= nb) o.bin = nb - 1;
  } else {
    o.bin = (c / J) % nb;
    o.age = ((double)(2 * o.bin + 1) / (double)(2 * nb)) * T;
  }
  o.g = (uint64_t)w.z < rp->thr_pi;
  const int cond = c % J;
  if (D->cap_mode == 2) {
    const int grp = o.bin * 2 + D->is_chase[cond];
    const int64_t off0 = goff[grp];
    const uint32_t cnt = (uint32_t)(goff[grp + 1] - off0);
    o.bc = betas[off0 + (int64_t)lemire(w.w, cnt)];
  } else if (D->cap_mode == 1) {
    // Beta(a, b) = a-th smallest of a+b-1 uniforms
    const int a = D->beta_a, nu = D->beta_a + D->beta_b - 1;
    uint32_t s0 = 0xFFFFFFFFu, s1 = 0xFFFFFFFFu, s2 = 0xFFFFFFFFu, s3 = 0xFFFFFFFFu;
    u4 v{0, 0, 0, 0};
    for (int qq = 0; qq < nu; ++qq) {
      if ((qq & 3) == 0) v = draw(gctr++, 0u, cw, pid, k0, k1);
      const int sel = qq & 3;
      const uint32_t x = sel == 0 ? v.x : (sel == 1 ? v.y : (sel == 2 ? v.z : v.w));
      if (x < s3) {
        s3 = x;
        if (s3 < s2) { const uint32_t tt = s2; s2 = s3; s3 = tt; }
        if (s2 < s1) { const uint32_t tt = s1; s1 = s2; s2 = tt; }
        if (s1 < s0) { const uint32_t tt = s0; s0 = s1; s1 = tt; }
      }
    }
    o.bc = u01_32(a == 1 ? s0 : (a == 2 ? s1 : (a == 3 ? s2 : s3)));
  } else {
    o.bc = 1.0;
  }
  return o;
}

// Burn-in, one lane per cell (persistent, cells of the heaviest particles
// first): the gene path from the start of the burn-in to the labelling window
// start ws, carrying the Poisson means of the cell's observed unspliced (lu)
// and all (lt) molecules; the cell's state at ws goes to rec[p * C + c].
// A small launch ends with its longest cell's chain of steps, so the step's two
// exponentials run side by side: 16 particles of 550 cells 7.9 -> 7.1 ms (the
// next waiting time drawn one step ahead as well: 6.8, but 42 ms for 38 in a
// launch of 5 x 1,024 particles of 2,500 cells, which VALU issue bounds; fewer
// lanes per wave: 8 to 15 ms).  Five waves per SIMD: 37.9 ms there, four 38.9.
__global__ __launch_bounds__(SSA_WG) __attribute__((amdgpu_waves_per_eu(5))) void burn_kernel(const DesignDev* __restrict__ D,
                                                      const PRates* __restrict__ R,
                                                      const int32_t* __restrict__ order, int64_t n,
                                                      uint32_t first, uint32_t k0, uint32_t k1,
                                                      uint32_t mtag_all,
                                                      const uint32_t* __restrict__ mtags,
                                                      const double* __restrict__ betas,
                                                      const int64_t* __restrict__ goff,
                                                      unsigned long long* __restrict__ queue,
                                                      CellStart* __restrict__ rec,
                                                      uint32_t* __restrict__ cellkey,
                                                      unsigned long long* __restrict__ steps_out,
                                                      const int64_t* __restrict__ pidx,
                                                      unsigned long long* __restrict__ burn_tally) {
  const double T = D->T;
  const int nb = D->nb, J = D->J, C = D->C;
  const double h = T / (double)nb;  // hours between rate-bin edges
  const unsigned long long total = (unsigned long long)n * (unsigned long long)C;
  unsigned long long lane_steps = 0;  // this lane's burn-in draws, added to *burn_tally at exit
  __shared__ LogEntry32 ltab32[ABC_LOG_N];
  load_log32_table(ltab32);
  __syncthreads();
  for (;;) {
    const unsigned long long q = atomicAdd(queue, 1ull);
    if (q >= total) break;
    const int p = order[q / (unsigned long long)C];
    const int c = (int)(q % (unsigned long long)C);
    const PRates* rp = R + p;
    const uint32_t pid = pidx ? (uint32_t)pidx[p] : first + (uint32_t)p;
    // counter word: the cell and the particle's model (the key is the seed alone)
    const uint32_t cw = (uint32_t)c | (mtags ? mtags[p] : mtag_all);
    uint64_t gctr = 0;
    const CellSetup cs0 = cell_setup(D, rp, c, cw, pid, k0, k1, betas, goff, gctr);
    const int cond = c % J;
    const double age = cs0.age, bc = cs0.bc;
    const double ws = age - D->pulse[cond] - D->chase[cond];
    const int step = rp->step;
    const bool scaling = rp->scaling, gvar = rp->gene_varies;
    const double bs = rp->bs;
    const int64_t nbB = (int64_t)rp->B * nb;
    int64_t k = 0, knext = step;
    int j = 0;
    double t = grid_time(0, nbB, h), cs = t, gk = grid_time(knext, nbB, h), tg = 0.0;
    double lu = 0.0, lt = 0.0;
    bool g = cs0.g, gneed = true;
    double ikon = rp->ikon[0], ikoff = rp->ikoff[0];
    double atx = rp->amax[0] * bc, gam = rp->gam[0], bound = D->bound[0];
    double iku = rp->iku[0], ikt = rp->ikt[0], abnd = atx / bound;
    unsigned long long st = 0;
    for (;;) {
      double tb = age;
      if (gk < tb) tb = gk;
      if (ws < tb) tb = ws;
      if (gneed) {
        const u4 v = draw(gctr++, 0u, cw, pid, k0, k1);
        st++;
        tg = t + (double)exp1_32(v.x, ltab32) * (g ? ikoff : ikon);
        gneed = false;
      }
      // births at rate atx (T + a) / bound_j (size scaling) or atx, a = t - cycle start
      {
        const double t1 = tg < tb ? tg : tb;
        double c0 = atx, c1 = 0.0;
        if (scaling) {
          c1 = abnd;
          c0 = c1 * (T + (t - cs));
        }
        burn_accum(lu, lt, g, c0, c1, gam + bs, iku, gam, ikt, t1 - t);
      }
      if (tg < tb) {
        t = tg;
        g = !g;
        gneed = true;
        continue;
      }
      t = tb;
      if (tb == gk) {
        k = knext;
        knext += step;
        j += step;  // k mod nb (step is 1 or nb)
        if (j >= nb) j -= nb;
        if (j == 0) {
          cs = tb;
          lu = lu * 0.5;  // division halves the Poisson means
          lt = lt * 0.5;
        }
        if (step == 1) {
          ikon = rp->ikon[j];
          ikoff = rp->ikoff[j];
          atx = rp->amax[j] * bc;
          gam = rp->gam[j];
          bound = D->bound[j];
          iku = rp->iku[j];
          ikt = rp->ikt[j];
          abnd = atx / bound;
        }
        if (gvar) gneed = true;  // the gene's rate changed: restart its clock
        gk = grid_time(knext, nbB, h);
      }
      if (tb == ws) break;
    }
    CellStart r;
    r.age = age;
    r.bc = bc;
    r.tg = tg;
    r.lu = lu;
    r.lt = lt;
    r.k = k;
    r.gctr = gctr;
    r.bin = (uint8_t)cs0.bin;
    r.g = (uint8_t)g;
    r.gneed = (uint8_t)gneed;
    // sub-lanes of this cell: smallest power of two M with the cell's expected
    // molecule events in its window <= split_target * M (M selects random
    // streams: the CPU replay uses the same operations).  Events: the
    // unlabelled molecules at the window start (at most 2 each) and births
    // at the cell's own capture over its own window (3 events each).
    {
      int M = 1, msh = 0;
      if (D->split_target > 0.0) {
        const double w = D->pulse[cond] + D->chase[cond];
        const double est = (lu + lt) + ((rp->brate * bc) * w) * 3.0;
        while (M < D->split_max && est > D->split_target * (double)M) {
          M *= 2;
          msh++;
        }
      }
      r.msh = (uint8_t)msh;
      // key of the cell's place in the window queue (a schedule only): expected
      // draws of one of its items, quarter-octave classes from 4 draws up.
      // Gene switches of the window; a 1/M share of the births and of the
      // splicing and loss of those molecules and of the ones at the start
      const float w = (float)(D->pulse[cond] + D->chase[cond]);
      const float ps = fminf(1.0f, (float)bs * w), pd = fminf(1.0f, rp->gmean * w);
      const float mol = (float)lu * ps + (float)lt * pd +
                        (float)(rp->brate * bc) * w * (1.0f + 0.5f * ps + 0.5f * pd);
      const float cost = rp->swrate * w + ldexpf(mol, -msh) + 4.0f;
      int cls = (int)((__float_as_uint(cost) >> 21) & 0x3FFu) - 127 * 4 - 8;
      cls = cls < 0 ? 0 : (cls > ABC_CELL_BUCKETS / 16 - 1 ? ABC_CELL_BUCKETS / 16 - 1 : cls);
      cellkey[(size_t)p * (size_t)C + (size_t)c] = (uint32_t)(cls * 16 + msh);
    }
    rec[(size_t)p * (size_t)C + (size_t)c] = r;
    atomicAdd(steps_out + p, st);
    lane_steps += st;
  }
  atomicAdd(burn_tally, lane_steps);
}

// ---------------------------------------------------------------- the SSA
// Labelling window of a work item = (particle, cell, sub-lane).  Sub-lane sub
// draws its unlabelled molecules at the window start, Poisson(lu / M)
// unspliced and Poisson((lt - lu) / M) spliced, from its own stream 1 + sub,
// then simulates the four species to the sampling age: it replays the cell's
// gene path from the shared stream 0 (continued from the burn-in) and carries
// its own 1/M share of the births and those molecules' fates (direct method).
// Molecules never act on the gene, so the sum over sub-lanes has the law of
// the whole cell.  Lanes refill from a global item queue the moment their item
// ends, so heavy and light particles share the machine without idle lanes.
// Held to 128 VGPRs, four waves per SIMD: the compiler's own allocation (140
// VGPRs, three waves) leaves more of the FP64 and Philox latency exposed.
// The four-wave build measured 7 % less SSA time per step; with the Philox
// key the same in every lane it fits 128 VGPRs without spilling.
__global__ __launch_bounds__(SSA_WG) __attribute__((amdgpu_waves_per_eu(4))) void ssa_kernel(const DesignDev* __restrict__ D,
                                                     const PRates* __restrict__ R,
                                                     const CellTables* __restrict__ tabs,
                                                     const uint32_t* __restrict__ cellord,
                                                     uint32_t first, uint32_t k0, uint32_t k1,
                                                     uint32_t mtag_all,
                                                     const uint32_t* __restrict__ mtags,
                                                     const CellStart* __restrict__ rec,
                                                     unsigned long long* __restrict__ queue,
                                                     uint32_t* __restrict__ out_u,
                                                     uint32_t* __restrict__ out_l,
                                                     uint8_t* __restrict__ out_bin,
                                                     unsigned long long* __restrict__ steps_out,
                                                     const int64_t* __restrict__ pidx,
                                                     uint32_t claim) {
  const double T = D->T;
  const int nb = D->nb, J = D->J, C = D->C;
  const double h = T / (double)nb;  // hours between rate-bin edges
  __shared__ LogEntry ltab[ABC_LOG_N];
  __shared__ LogEntry32 ltab32[ABC_LOG_N];
  __shared__ double rk[ABC_RECIP_N];
  __shared__ unsigned long long ioff[ABC_CELL_BUCKETS + 1];
  load_log_table(ltab);
  load_log32_table(ltab32);
  for (int q = threadIdx.x; q < ABC_RECIP_N; q += blockDim.x) rk[q] = abc_recip_k[q];
  for (int q = threadIdx.x; q <= ABC_CELL_BUCKETS; q += blockDim.x) ioff[q] = tabs->ioff[q];
  __syncthreads();
  const unsigned long long total = ioff[ABC_CELL_BUCKETS];
  // expected draws of two lanes' shares of the call, which no claim exceeds
  const float share = 2.0f * (float)tabs->draws / (float)(gridDim.x * SSA_WG);

  uint32_t cw = 0;  // counter word of the current item: cell | model << 24
  // per-lane item state
  bool have = false;
  int p = 0, c = 0, j = 0, step = 1, scaling = 0, gvar = 0;
  uint32_t pid = 0, sstream = 1, n0 = 0, n1 = 0, n2 = 0, n3 = 0;
  // Philox blocks drawn on the gene stream (continued from the burn-in, which
  // had drawn gctr0) and on the item's molecule stream: every step draws one
  // block on exactly one of them, so the item's steps are mctr + gctr - gctr0
  uint64_t gctr = 0, gctr0 = 0, mctr = 0;
  // labelled when pw <= thr_m1 = floor(lambda 2^32) - 1 (lab_on: lambda > 0)
  uint32_t thr_m1 = 0, shi = 0;  // shi: the molecule stream's counter word, stream << 16
  bool lab_on = false;
  int64_t k = 0, knext = 0, nbB = 0;
  // tcs = T - (start of the current cycle): the size-scaling test compares
  // with t + tcs = T + (time since the cycle start)
  double t = 0.0, tb = 0.0, gk = 0.0, tg = 0.0, age = 0.0, we = 0.0, tcs = 0.0;
  double ikon = 0.0, ikoff = 0.0, atx = 0.0, gam = 0.0, bs = 0.0, bc = 1.0, bound = 0.0;
  double ishare = 1.0;  // 1 / (the cell's sub-lanes), a power of two
  bool g = false, in_win = false, div = false;
  int div_s = 0;
  uint32_t div_rem = 0, div_keep = 0;
  // gene clock to (re)draw; pending molecule candidate (its residual Exp(1)
  // hazard and unused words)
  bool gneed = false, pend = false;
  double erem = 0.0;
  uint32_t py = 0, pz = 0, pw = 0;
  // The lane's claim: qleft more items from queue position qnext on.  A refill
  // holds up the whole wave for the queue's atomic, so light items are claimed
  // several at a time, the more the lighter (twice as many per two octaves of
  // cost, from claim * 2 just below class ABC_LIGHT_CLASS, 2,048 draws); heavy
  // ones singly, since a second one waiting behind the first would end late.
  // 5 x 1,024 particles: 329 ms with one item a claim throughout, 312 ms with
  // claims of `claim` items below class 36, 296 ms so; the line at class 32 or
  // 40 measured 297 and 299 ms.  Nor more than twice a lane's share of the call's
  // draws, or a call of light items alone ends with the lanes that claimed many:
  // 20,000 particles of 55 cells with 43 / 128 draws a cell 6.2 / 9.4 ms without
  // that, 4.7 / 7.1 with it (with `claim` 8 12 / 19 and 4.7 / 7.3).  Half a share,
  // one, two, no limit: 3,000 particles of 2,000 cells 12.7, 11.0, 9.9, 10.5 ms,
  // 20,000 of 55 cells with 969 draws 15.0, 14.3, 16.8, 16.5.
  unsigned long long qnext = 0;
  uint32_t qleft = 0;
  // the bucket that the lane's last item lies in: its rank, first item, the
  // item after its last and its first cell.  The lane's queue positions only
  // grow, so the bucket is searched again only once they pass its end.
  unsigned long long qbase = 0, qend = 0;
  uint32_t qcell = 0;
  int qrank = 0;

  for (;;) {
    if (!have) {
      if (qleft == 0u) {
        const int cls = (ABC_CELL_BUCKETS - 1 - qrank) >> 4;
        qleft = 1u;
        if (cls < ABC_LIGHT_CLASS) {
          const uint32_t want = claim << ((ABC_LIGHT_CLASS + 8 - cls) >> 3);
          const float cap = share * __builtin_amdgcn_exp2f(-2.0f - 0.25f * (float)cls);
          qleft = cap < (float)want ? (cap > 1.0f ? (uint32_t)cap : 1u) : want;
        }
        qnext = atomicAdd(queue, (unsigned long long)qleft);
      }
      const unsigned long long q = qnext++;
      qleft--;
      if (q >= total) break;
      if (q >= qend) {
        int lo = qrank, hi = ABC_CELL_BUCKETS;  // largest rank with ioff[rank] <= q
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (ioff[mid] <= q) lo = mid; else hi = mid;
        }
        qrank = lo;
        qbase = ioff[lo];
        qend = ioff[lo + 1];
        qcell = tabs->cbase[lo];
      }
      const int qsh = (ABC_CELL_BUCKETS - 1 - qrank) & 15;
      const uint32_t cell = cellord[qcell + (uint32_t)((q - qbase) >> qsh)];
      const int sub = (int)((uint32_t)(q - qbase) & ((1u << qsh) - 1u));
      p = (int)(cell / (uint32_t)C);
      c = (int)(cell - (uint32_t)p * (uint32_t)C);
      const PRates* rp = R + p;
      pid = pidx ? (uint32_t)pidx[p] : first + (uint32_t)p;
      cw = (uint32_t)c | (mtags ? mtags[p] : mtag_all);
      sstream = 1u + (uint32_t)sub;
      shi = sstream << 16;
      const CellStart* rc = rec + ((size_t)p * (size_t)C + (size_t)c);
      ishare = ldexp(1.0, -qsh);  // x / M == x * ishare exactly
      mctr = 0;
      // every loop-carried value is reset here, so none stays live across the
      // sampler below
      div_s = 0;
      div_rem = 0;
      div_keep = 0;
      erem = 0.0;
      py = pz = pw = 0;
      {
        // the sub-lane's unlabelled molecules at the window start
        WordSrc src{u4{0, 0, 0, 0}, 4, mctr, sstream, cw, pid, k0, k1};
        const double lu0 = rc->lu, ls = rc->lt - lu0;
        n0 = poisson(src, lu0 * ishare, ltab, rk);
        n1 = poisson(src, ls > 0.0 ? ls * ishare : 0.0, ltab, rk);
      }
      const CellStart r0 = *rc;
      n2 = n3 = 0;
      const int cond = c % J;
      age = r0.age;
      bc = r0.bc;
      we = age - D->chase[cond];
      if (sub == 0) out_bin[(size_t)p * (size_t)C + (size_t)c] = r0.bin;
      step = rp->step;
      scaling = rp->scaling;
      gvar = rp->gene_varies;
      lab_on = rp->thr_lam != 0ull;
      thr_m1 = (uint32_t)(rp->thr_lam - 1ull);
      bs = rp->bs;
      nbB = (int64_t)rp->B * nb;
      k = r0.k;
      knext = k + step;
      j = (int)((uint64_t)k % (uint64_t)nb);
      tcs = T - grid_time(k - j, nbB, h);
      gk = grid_time(knext, nbB, h);
      t = age - D->pulse[cond] - D->chase[cond];
      gctr = r0.gctr;
      gctr0 = gctr;
      g = r0.g != 0;
      tg = r0.tg;
      gneed = r0.gneed != 0;
      ikon = rp->ikon[j];  // gene clock: waiting time = E * (1 / rate)
      ikoff = rp->ikoff[j];
      atx = (rp->amax[j] * bc) * ishare;
      gam = rp->gam[j];
      bound = D->bound[j];
      in_win = true;
      div = false;
      pend = false;
      tb = age;
      if (gk < tb) tb = gk;
      if (we < tb) tb = we;
      have = true;
    }

    // propensities of this sub-lane's molecule channels (direct method)
    const double a_tx = g ? atx : 0.0;
    const uint32_t nun = n0 + n2, ntot = n0 + n1 + n2 + n3;
    const double a_spl = bs * (double)nun;
    const double a_dec = gam * (double)ntot;
    const double c1 = a_tx, c2 = c1 + a_spl;
    const double a0 = c2 + a_dec;

    // One Philox block per lane and iteration, in uniform control flow:
    // division coins, the gene clock (shared stream 0) or a new molecule
    // candidate (stream 1 + sub).  A candidate pre-empted by the gene clock or
    // a boundary stays pending: its words are unused and its Exp(1) hazard,
    // less what the interval used up, is again Exp(1) (memoryless).
    // (division coins, else the gene clock, else a new candidate, else no draw)
    const bool kgen = !div && gneed;
    const bool kmol = !div && !gneed && !pend && a0 > 0.0;
    const bool mol = div || kmol;
    const uint64_t ctr = mol ? mctr : gctr;
    const u4 w = philox((uint32_t)ctr, ((uint32_t)(ctr >> 32) & 0xFFFFu) | (mol ? shi : 0u), cw,
                        pid, k0, k1);
    mctr += mol ? 1ull : 0ull;
    gctr += kgen ? 1ull : 0ull;
    if (div) {
      // binomial(count, 1/2) partition of species div_s, 128 coin flips per block
      const uint32_t m = div_rem < 128u ? div_rem : 128u;
      uint32_t cnt = __popc(m >= 32u ? w.x : (w.x & ((1u << m) - 1u)));
      if (m > 32u) cnt += __popc(m >= 64u ? w.y : (w.y & ((1u << (m - 32u)) - 1u)));
      if (m > 64u) cnt += __popc(m >= 96u ? w.z : (w.z & ((1u << (m - 64u)) - 1u)));
      if (m > 96u) cnt += __popc(m >= 128u ? w.w : (w.w & ((1u << (m - 96u)) - 1u)));
      div_keep += cnt;
      div_rem -= m;
      if (div_rem == 0u) {
        if (div_s == 0) n0 = div_keep;
        else if (div_s == 1) n1 = div_keep;
        else if (div_s == 2) n2 = div_keep;
        else n3 = div_keep;
        div_s++;
        while (div_s < 4 && (div_s == 1 ? n1 : (div_s == 2 ? n2 : n3)) == 0u) div_s++;
        if (div_s < 4) {
          div_rem = div_s == 1 ? n1 : (div_s == 2 ? n2 : n3);
          div_keep = 0;
        } else {
          div = false;
        }
      }
      continue;
    }
    const double E = (double)exp1_32(w.x, ltab32);
    if (kgen) {
      tg = t + E * (g ? ikoff : ikon);
      gneed = false;
      if (!pend && a0 > 0.0) continue;  // a molecule candidate comes first
    } else if (kmol) {
      erem = E;
      py = w.y;
      pz = w.z;
      pw = w.w;
      pend = true;
    }

    // next event: the molecule candidate, the gene switch or a boundary
    const double tm = (pend && a0 > 0.0) ? t + erem / a0 : __longlong_as_double(0x7ff0000000000000ll);
    if (tm < tg && tm < tb) {
      t = tm;
      pend = false;
      // The channel, then its molecule, as predicated arithmetic: lanes of a
      // wave that fire different channels run one instruction stream.
      //   transcription (rr < c1): kept by the size-scaling thinning test on
      //     pz, labelled when pw < thr_lam inside the window;
      //   splicing (c1 <= rr < c2): molecule lemire(pz, n0 + n2) of the
      //     unspliced, unlabelled first;
      //   decay (rr >= c2): molecule lemire(pz, ntot) in species order.
      // u01_32(py) * a0 with the power-of-two scale on a0: the same single
      // rounding of the same exact product, one instruction less
      const double rr = ((double)py + 0.5) * (a0 * 0x1p-32);
      const bool tx = rr < c1;
      const bool spl = !tx && rr < c2;
      const bool dec = !tx && !spl;
      const bool acc = tx && (!scaling || u01_32(pz) * bound < t + tcs);
      const bool lab = in_win && lab_on && pw <= thr_m1;
      const uint32_t x = lemire(pz, spl ? nun : ntot);
      const bool ge0 = x >= n0, ge1 = x >= n0 + n1, ge2 = x >= n0 + n1 + n2;
      // each species gains one, loses one or stays (the conditions exclude
      // each other): one select chain and one add per species
      n0 += (acc && !lab) ? 1u : ((!tx && !ge0) ? 0xFFFFFFFFu : 0u);
      n1 += (spl && !ge0) ? 1u : ((dec && ge0 && !ge1) ? 0xFFFFFFFFu : 0u);
      n2 += (acc && lab) ? 1u : (((spl && ge0) || (dec && ge1 && !ge2)) ? 0xFFFFFFFFu : 0u);
      n3 += (spl && ge0) ? 1u : ((dec && ge2) ? 0xFFFFFFFFu : 0u);
      continue;
    }
    if (pend) {
      // no molecule event before min(tg, tb): a0 times that interval is used up
      const double t1 = tg < tb ? tg : tb;
      erem = erem - a0 * (t1 - t);
      if (erem < 0.0) erem = 0.0;
    }
    if (tg < tb) {
      t = tg;
      g = !g;
      gneed = true;
      continue;
    }
    // boundary: sampling age, rate-bin / cycle edge, or the window end
    t = tb;
    if (tb == age) {
      const size_t o = (size_t)p * (size_t)C + (size_t)c;
      atomicAdd(out_u + o, n0 + n1);
      atomicAdd(out_l + o, n2 + n3);
      atomicAdd(steps_out + p, (unsigned long long)(mctr + (gctr - gctr0)));
      have = false;
      continue;
    }
    if (tb == gk) {
      k = knext;
      knext += step;
      j += step;  // k mod nb (step is 1 or nb)
      if (j >= nb) j -= nb;
      if (j == 0) {
        tcs = T - tb;
        div_s = 0;
        while (div_s < 4 && (div_s == 0 ? n0 : (div_s == 1 ? n1 : (div_s == 2 ? n2 : n3))) == 0u) div_s++;
        if (div_s < 4) {
          div = true;
          div_rem = div_s == 0 ? n0 : (div_s == 1 ? n1 : (div_s == 2 ? n2 : n3));
          div_keep = 0;
        }
      }
      if (step == 1) {
        const PRates* rp = R + p;
        ikon = rp->ikon[j];
        ikoff = rp->ikoff[j];
        atx = (rp->amax[j] * bc) * ishare;
        gam = rp->gam[j];
        bound = D->bound[j];
      }
      if (gvar) gneed = true;  // the gene's rate changed: restart its clock (memoryless)
      gk = grid_time(knext, nbB, h);
    }
    if (in_win && tb == we) in_win = false;
    tb = age;
    if (gk < tb) tb = gk;
    if (in_win && we < tb) tb = we;
  }
}

// -------------------------------------------------------------- statistics
__device__ __forceinline__ void add128(unsigned long long* lo, unsigned long long* hi,
                                       unsigned long long x) {
  const unsigned long long old = atomicAdd(lo, x);
  if (old + x < old) atomicAdd(hi, 1ull);
}

struct U128 { uint64_t hi, lo; };

__device__ __forceinline__ U128 mul64(uint64_t a, uint64_t b) {
  return U128{__umul64hi(a, b), a * b};
}
__device__ __forceinline__ U128 add(U128 a, U128 b) {
  U128 r{a.hi + b.hi, a.lo + b.lo};
  if (r.lo < a.lo) r.hi++;
  return r;
}
__device__ __forceinline__ U128 sub(U128 a, U128 b) {  // requires a >= b
  U128 r{a.hi - b.hi, a.lo - b.lo};
  if (a.lo < b.lo) r.hi--;
  return r;
}
__device__ __forceinline__ bool ge(U128 a, U128 b) {
  return a.hi > b.hi || (a.hi == b.hi && a.lo >= b.lo);
}
// n * (hi:lo) with n < 2^32 and the product < 2^128
__device__ __forceinline__ U128 mul_small(uint64_t n, U128 v) {
  U128 lo = mul64(n, v.lo);
  lo.hi += n * v.hi;
  return lo;
}

__device__ __forceinline__ double var_of(uint64_t n, uint64_t S, U128 SS) {
  const U128 num = sub(mul_small(n, SS), mul64(S, S));
  return u128_to_f64(num.hi, num.lo) / ((double)n * (double)(n - 1));
}
__device__ __forceinline__ double cov_of(uint64_t n, uint64_t Sa, uint64_t Sb, U128 Sab) {
  const U128 a = mul_small(n, Sab), b = mul64(Sa, Sb);
  const double den = (double)n * (double)(n - 1);
  if (ge(a, b)) { const U128 d = sub(a, b); return u128_to_f64(d.hi, d.lo) / den; }
  const U128 d = sub(b, a);
  return -(u128_to_f64(d.hi, d.lo) / den);
}

__device__ __forceinline__ double wcov(const double* x, const double* y, const double* w, int nb) {
  double mx = w[0] * x[0], my = w[0] * y[0];
  for (int b = 1; b < nb; ++b) mx = mx + w[b] * x[b];
  for (int b = 1; b < nb; ++b) my = my + w[b] * y[b];
  double acc = w[0] * ((x[0] - mx) * (y[0] - my));
  for (int b = 1; b < nb; ++b) acc = acc + w[b] * ((x[b] - mx) * (y[b] - my));
  return acc;
}

__global__ __launch_bounds__(256) void stats_kernel(const DesignDev* __restrict__ D,
                                                    const uint32_t* __restrict__ cu,
                                                    const uint32_t* __restrict__ cl,
                                                    const uint8_t* __restrict__ cb, int64_t n,
                                                    double* __restrict__ stats_ref,
                                                    double* __restrict__ moments,
                                                    double* __restrict__ superset) {
  const int nb = D->nb, J = D->J, C = D->C, NBJ = nb * J;
  __shared__ unsigned int s_n[ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ unsigned long long s_su[ABC_MAX_BINS * ABC_MAX_CONDS], s_sl[ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ unsigned long long s_uu[2][ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ unsigned long long s_ll[2][ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ unsigned long long s_ul[2][ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ double s_m1[ABC_MAX_BINS * ABC_MAX_CONDS], s_m2[ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ double s_v1[ABC_MAX_BINS * ABC_MAX_CONDS], s_v2[ABC_MAX_BINS * ABC_MAX_CONDS];
  __shared__ double s_c12[ABC_MAX_BINS * ABC_MAX_CONDS];
  // one particle per workgroup at a time (grid-stride over particles)
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    for (int q = threadIdx.x; q < NBJ; q += blockDim.x) {
      s_n[q] = 0; s_su[q] = 0; s_sl[q] = 0;
      s_uu[0][q] = s_uu[1][q] = 0; s_ll[0][q] = s_ll[1][q] = 0; s_ul[0][q] = s_ul[1][q] = 0;
    }
    __syncthreads();
    const uint32_t* u = cu + (size_t)i * C;
    const uint32_t* l = cl + (size_t)i * C;
    const uint8_t* bn = cb + (size_t)i * C;
    for (int c = threadIdx.x; c < C; c += blockDim.x) {
      if (bn[c] >= nb) continue;  // never produced by the SSA; keeps LDS indexing in range
      const int idx = bn[c] + nb * (c % J);
      const unsigned long long a = u[c], b = l[c];
      atomicAdd(&s_n[idx], 1u);
      atomicAdd(&s_su[idx], a);
      atomicAdd(&s_sl[idx], b);
      add128(&s_uu[0][idx], &s_uu[1][idx], a * a);
      add128(&s_ll[0][idx], &s_ll[1][idx], b * b);
      add128(&s_ul[0][idx], &s_ul[1][idx], a * b);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < NBJ; idx += blockDim.x) {
      const uint64_t nn = s_n[idx];
      const U128 uu{s_uu[1][idx], s_uu[0][idx]}, ll{s_ll[1][idx], s_ll[0][idx]},
          ul{s_ul[1][idx], s_ul[0][idx]};
      double mt = 0.0, fft = 0.0, m1 = 0.0, m2 = 0.0, v1 = 0.0, v2 = 0.0, c12 = 0.0;
      if (nn > 0) {
        const double q = (double)nn;
        m1 = (double)s_su[idx] / q;
        m2 = (double)s_sl[idx] / q;
        v1 = var_of(nn, s_su[idx], uu);
        v2 = var_of(nn, s_sl[idx], ll);
        c12 = cov_of(nn, s_su[idx], s_sl[idx], ul);
        const uint64_t St = s_su[idx] + s_sl[idx];
        const U128 Stt = add(add(uu, add(ul, ul)), ll);
        mt = (double)St / q;
        const double vt = var_of(nn, St, Stt);
        fft = vt / (mt + (mt == 0.0 ? 0.0001 : 0.0));
      }
      s_m1[idx] = m1; s_m2[idx] = m2; s_v1[idx] = v1; s_v2[idx] = v2; s_c12[idx] = c12;
      if (moments) {
        double* mo = moments + i;
        const int64_t base = 6 * (int64_t)idx;
        mo[n * (base + 0)] = (double)nn;
        mo[n * (base + 1)] = m1;
        mo[n * (base + 2)] = m2;
        mo[n * (base + 3)] = v1;
        mo[n * (base + 4)] = c12;
        mo[n * (base + 5)] = v2;
        if (nn == 0) {
          for (int qq = 0; qq < 6; ++qq) mo[n * (base + qq)] = 0.0;
        }
      }
      if (superset) {
        superset[i + n * idx] = mt;
        superset[i + n * (NBJ + idx)] = fft;
      }
    }
    __syncthreads();
    const int tid = threadIdx.x;
    if (stats_ref && tid < 2 * nb) {
      const int grp = tid / nb, b = tid % nb;
      uint64_t nn = 0, St = 0;
      U128 Stt{0, 0};
      for (int jj = 0; jj < J; ++jj) {
        if (D->is_chase[jj] != grp) continue;
        const int idx = b + nb * jj;
        nn += s_n[idx];
        St += s_su[idx] + s_sl[idx];
        const U128 uu{s_uu[1][idx], s_uu[0][idx]}, ll{s_ll[1][idx], s_ll[0][idx]},
            ul{s_ul[1][idx], s_ul[0][idx]};
        Stt = add(Stt, add(add(uu, add(ul, ul)), ll));
      }
      double mean = 0.0, ff = 0.0;
      if (nn > 0) {
        mean = (double)St / (double)nn;
        const double v = var_of(nn, St, Stt);
        ff = v / (mean + (mean == 0.0 ? 0.0001 : 0.0));
      }
      stats_ref[i + n * ((2 * grp) * nb + b)] = mean;
      stats_ref[i + n * ((2 * grp + 1) * nb + b)] = ff;
    } else if (stats_ref && tid >= 64 && tid < 64 + J) {
      const int jj = tid - 64;
      uint64_t nn = 0, su = 0, sl = 0;
      bool anynz = false;
      for (int b = 0; b < nb; ++b) {
        const int idx = b + nb * jj;
        nn += s_n[idx]; su += s_su[idx]; sl += s_sl[idx];
        if (s_c12[idx] != 0.0) anynz = true;
      }
      double ratio = 0.0;
      if (nn > 0) {
        const double a1 = (double)su / (double)nn, a2 = (double)sl / (double)nn;
        if (a1 + a2 > 0.0) ratio = a2 / (a1 + a2);
      }
      const double* w = D->weights + nb * jj;
      const double* m1 = s_m1 + nb * jj;
      const double* m2 = s_m2 + nb * jj;
      const double* v1 = s_v1 + nb * jj;
      const double* v2 = s_v2 + nb * jj;
      const double* c12 = s_c12 + nb * jj;
      double s1 = w[0] * v1[0], s2 = w[0] * v2[0], s12 = w[0] * c12[0];
      for (int b = 1; b < nb; ++b) s1 = s1 + w[b] * v1[b];
      for (int b = 1; b < nb; ++b) s2 = s2 + w[b] * v2[b];
      for (int b = 1; b < nb; ++b) s12 = s12 + w[b] * c12[b];
      const double tv1 = s1 + wcov(m1, m1, w, nb);
      const double tv2 = s2 + wcov(m2, m2, w, nb);
      double mc = 0.0, cm = 0.0;
      if (anynz && tv1 != 0.0 && tv2 != 0.0) mc = s12 / sqrt(fabs(tv1 * tv2));
      if (tv1 != 0.0 && tv2 != 0.0) cm = wcov(m1, m2, w, nb) / sqrt(fabs(tv1 * tv2));
      stats_ref[i + n * (4 * nb + jj)] = ratio;
      stats_ref[i + n * (4 * nb + J + jj)] = mc;
      stats_ref[i + n * (4 * nb + 2 * J + jj)] = cm;
    }
    __syncthreads();  // the LDS sums are cleared for the next particle
  }
}

// ------------------------------------------------------------------ errors
// FP64 errors of gene g and N particles in the order of compute_errors.jl:30-64.
template <int N>
__device__ __forceinline__ void err_pairs(const double* __restrict__ data,
                                          const double* __restrict__ se, int64_t G, int64_t g,
                                          const double* __restrict__ stats, int64_t n,
                                          const int64_t (&i)[N], const ErrSpec& E,
                                          double (&err)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) err[j] = 0.0;
  int k = 0;
  for (int pp = 0; pp < E.n_parts; ++pp) {
    double e[N] = {};
    const int end = k + E.parts[pp];
    for (; k < end; ++k) {
      const double d = data[g + G * k];
      const double den = err_den(d, se[g + G * k]);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const double diff = d - stats[i[j] + n * k];
        e[j] += (diff * diff) / den;
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) err[j] += e[j] / (double)E.K;
  }
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (err[j] > E.clamp) err[j] = E.clamp;
}

__device__ __forceinline__ double err_pair(const double* __restrict__ data,
                                           const double* __restrict__ se, int64_t G, int64_t g,
                                           const double* __restrict__ stats, int64_t n,
                                           int64_t i, const ErrSpec& E) {
  const int64_t at[1] = {i};
  double err[1];
  err_pairs<1>(data, se, G, g, stats, n, at, E, err);
  return err[0];
}

// err holds the columns of genes g0 .. g0 + gridDim.y - 1; one lane per pair,
// for calls too small for err_tile_kernel
__global__ __launch_bounds__(256) void err_fp64_kernel(const double* __restrict__ stats,
                                                       int64_t n, const double* __restrict__ data,
                                                       const double* __restrict__ se, int64_t G,
                                                       int64_t g0, ErrSpec E,
                                                       double* __restrict__ err) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t g = g0 + blockIdx.y;
  if (i >= n) return;
  err[i + n * (int64_t)blockIdx.y] = err_pair(data, se, G, g, stats, n, i, E);
}

// The same errors, 64 genes x PT particles per wave, four waves (4 PT
// particles) to a workgroup: a lane holds one gene, and the particles'
// statistics are uniform over the wave (scalar loads, one term ahead).  The
// genes' denominators and their reciprocals are formed once per workgroup, a
// quarter by each wave, ERR_KC terms at a time through LDS.  Bound by FP64
// issue: 7 operations a term (difference, square, four for the division by the
// known denominator, sum) against 22 with a division sequence and the
// denominator formed per pair.  The operations and their order are err_pair's
// and the quotients correctly rounded, so the bits are the same.  Pairs whose
// operands leave err_range / gene_range (infinite statistics among them) are
// formed by err_pairs: a tile's few such genes one pair a lane, such particles
// four at a time (9,973 x 3,419 pairs, one such value in every particle or in 5 %
// of the genes: 1.3 and 0.7 ms; one particle at a time for every lane that had
// one of either, 3.1 and 2.7).  Waves at the end of the particles
// overlap the ones before (the same values are written twice).  POOL: errors
// and global particle indices behind the pool_n[g] entries of the genes'
// acceptance pools instead, for a batch that meets no threshold yet.
// 9,973 particles x 3,419 genes: 1,524 -> 558 us with 53 statistics, 3,093 ->
// 840 us with 90 (0.65 of the FP64 issue peak by the 7 operations).
#define ERR_KC 16
template <int PT, bool POOL>
__global__ __launch_bounds__(256) void err_tile_kernel(const double* __restrict__ stats, int64_t n,
                                                       int64_t ld, const double* __restrict__ data,
                                                       const double* __restrict__ se, int64_t G,
                                                       ErrSpec E, double* __restrict__ err_out,
                                                       PoolEntry* __restrict__ pool, int64_t capg,
                                                       int64_t first_index,
                                                       const int64_t* __restrict__ pidx,
                                                       const uint32_t* __restrict__ pool_n) {
  __shared__ double s_d[ERR_KC][64], s_y[ERR_KC][64], s_zh[ERR_KC][64], s_zl[ERR_KC][64];
  __shared__ unsigned long long s_gbad;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t g = (int64_t)blockIdx.y * 64 + lane;
  int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * PT;
  if (i0 + PT > n) i0 = n - PT;  // n >= PT (the caller checks it)
  const int K = E.K;
  if (threadIdx.x == 0) s_gbad = 0ull;
  // particles of the wave with a statistic outside err_range
  uint32_t bad = 0u;
  for (int q = lane; q < PT * K; q += 64) {
    const int k = q / PT, p = q - k * PT;
    if (!err_range(stats[i0 + p + ld * k])) bad |= 1u << p;
  }
  for (int o = 32; o > 0; o >>= 1) bad |= (uint32_t)__shfl_xor((int)bad, o);
  const int64_t gc = g < G ? g : G - 1;  // lanes past the last gene repeat it and store nothing
  const Divisor dk = divisor_of((double)K);
  double err[PT], e[PT], s[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    err[p] = e[p] = 0.0;
    s[p] = stats[i0 + p];
  }
  int part = 0, end = E.parts[0];
  for (int k0 = 0; k0 < K; k0 += ERR_KC) {
    __syncthreads();
    bool gbad = false;
#pragma unroll
    for (int q = 0; q < ERR_KC / 4; ++q) {
      const int kk = q * 4 + wave;
      const int k = k0 + kk < K ? k0 + kk : K - 1;
      const double d = data[gc + G * k];
      const Divisor w = divisor_of(err_den(d, se[gc + G * k]));
      gbad |= !gene_range(d, w.y);
      s_d[kk][lane] = d;
      s_y[kk][lane] = w.y;
      s_zh[kk][lane] = w.zh;
      s_zl[kk][lane] = w.zl;
    }
    const unsigned long long gb = __ballot(gbad);
    if (lane == 0 && gb) atomicOr(&s_gbad, gb);
    __syncthreads();
    // no particle in range: only the genes are looked at.  bad stays in a vector
    // register, since the loop's statistics fill the scalar ones
    asm volatile("" : "+v"(bad));
    const bool none = __builtin_amdgcn_readfirstlane(bad) == (1u << PT) - 1u;
    const int kc = none ? 0 : (K - k0 < ERR_KC ? K - k0 : ERR_KC);
    double d = s_d[0][lane], y = s_y[0][lane], zh = s_zh[0][lane], zl = s_zl[0][lane];
    // waited for here, so that the wait at the top of the loop is not for them
    asm volatile("" : "+v"(d), "+v"(y), "+v"(zh), "+v"(zl));
    for (int kk = 0; kk < kc; ++kk) {
      while (k0 + kk == end) {  // the part is complete (an empty part adds its zero)
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          err[p] += div_by(e[p], dk.y, dk.zh, dk.zl);
          e[p] = 0.0;
        }
        end += E.parts[++part];
      }
      const int kn = k0 + kk + 1 < K ? k0 + kk + 1 : K - 1;
      double sn[PT];
#pragma unroll
      for (int p = 0; p < PT; ++p) sn[p] = stats[i0 + p + ld * kn];
      // LDS and scalar loads share a counter, so the genes' operands are read
      // one term ahead as well
      const int kl = kk + 1 < kc ? kk + 1 : kk;
      const double dn = s_d[kl][lane], yn = s_y[kl][lane], zhn = s_zh[kl][lane],
                   zln = s_zl[kl][lane];
      __builtin_amdgcn_sched_barrier(0);  // issue the loads before the term's arithmetic
      // div_by of four particles side by side: a wave's own chains overlap
#pragma unroll
      for (int p0 = 0; p0 < PT; p0 += 4) {
        double x[4], q[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = d - s[p0 + j];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = x[j] * x[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = x[j] * zl;
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = fma(x[j], zh, q[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = fma(-q[j], y, x[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = fma(x[j], zh, q[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) e[p0 + j] += q[j];
        __builtin_amdgcn_sched_barrier(0);
      }
      d = dn;
      y = yn;
      zh = zhn;
      zl = zln;
#pragma unroll
      for (int p = 0; p < PT; ++p) s[p] = sn[p];
    }
  }
#pragma unroll
  for (int p = 0; p < PT; ++p) err[p] += div_by(e[p], dk.y, dk.zh, dk.zl);
  bad = __builtin_amdgcn_readfirstlane(bad);
  const int64_t left = G - (int64_t)blockIdx.y * 64;  // genes of this tile
  const unsigned long long gbad = s_gbad & (left < 64 ? (1ull << left) - 1ull : ~0ull);
  const bool mine = g < G && !((gbad >> lane) & 1ull);
  auto put = [&](PoolEntry* pg, double* eg, int p, double v) {
    if (POOL)
      pg[i0 + p] = PoolEntry{v, pidx ? pidx[i0 + p] : first_index + i0 + p};
    else
      eg[i0 + p] = v;
  };
  auto store = [&](int64_t gene, int p, double v) {
    put(POOL ? pool + gene * capg + pool_n[gene] : nullptr, POOL ? nullptr : err_out + n * gene, p, v);
  };
  if (mine) {
    PoolEntry* pg = POOL ? pool + g * capg + pool_n[g] : nullptr;
    double* eg = POOL ? nullptr : err_out + n * g;
    if (bad == 0u) {
#pragma unroll
      for (int p = 0; p < PT; ++p) put(pg, eg, p, err[p] > E.clamp ? E.clamp : err[p]);
    } else {
#pragma unroll
      for (int p = 0; p < PT; ++p)
        if (!((bad >> p) & 1u)) put(pg, eg, p, err[p] > E.clamp ? E.clamp : err[p]);
    }
  }
  if (gbad) {
    // lane r: the tile's r-th gene outside the range
    const int nb = __popcll(gbad);
    const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(gbad >> 32),
                                                __builtin_amdgcn_mbcnt_lo((unsigned)gbad, 0u));
    const int at = (gbad >> lane) & 1ull ? below : nb + lane - below;
    const int ordered = __builtin_amdgcn_ds_permute(4 * at, lane);
    for (int q0 = 0; q0 < nb * PT; q0 += 64) {
      const int q = q0 + lane, p = q % PT;
      const int64_t gene = (int64_t)blockIdx.y * 64 + __shfl(ordered, (q / PT) & 63);
      if (q < nb * PT) store(gene, p, err_pair(data, se, G, gene, stats, ld, i0 + p, E));
    }
  }
  while (mine && bad) {
    int64_t at[4];
    double v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // the last one again where fewer are left
      at[j] = i0 + __ffs(bad) - 1;
      if (bad & (bad - 1u) || j == 3) bad &= bad - 1u;
    }
    err_pairs<4>(data, se, G, g, stats, ld, at, E, v);
#pragma unroll
    for (int j = 0; j < 4; ++j) store(g, (int)(at[j] - i0), v[j]);
  }
}

template __global__ void err_tile_kernel<16, false>(const double*, int64_t, int64_t, const double*,
                                                    const double*, int64_t, ErrSpec, double*,
                                                    PoolEntry*, int64_t, int64_t, const int64_t*,
                                                    const uint32_t*);
template __global__ void err_tile_kernel<16, true>(const double*, int64_t, int64_t, const double*,
                                                   const double*, int64_t, ErrSpec, double*,
                                                   PoolEntry*, int64_t, int64_t, const int64_t*,
                                                   const uint32_t*);
template __global__ void err_tile_kernel<4, false>(const double*, int64_t, int64_t, const double*,
                                                   const double*, int64_t, ErrSpec, double*,
                                                   PoolEntry*, int64_t, int64_t, const int64_t*,
                                                    const uint32_t*);

// The device's elementary functions on n inputs, for validation: kind 0 =
// ex (every kernel except the loops below), 1 = ex_core (the burn-in and the
// moment model's loops; arguments <= 709.78), 2 = ln (LDS table)
__global__ __launch_bounds__(256) void math_probe_kernel(int kind, int64_t n,
                                                         const double* __restrict__ x,
                                                         double* __restrict__ y) {
  __shared__ LogEntry ltab[ABC_LOG_N];
  load_log_table(ltab);
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double v = x[i];
    y[i] = kind == 0 ? ex(v) : (kind == 1 ? ex_core(v) : ln(v, ltab));
  }
}

__global__ void zero_u64_kernel(unsigned long long* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}
