// abc_accept.hip -- per-gene top-k acceptance kept in device memory: the
// selection of scripts/accepted_particles.jl:12-32 (per gene, particles
// ordered by error with ties by index, a stable sortperm) over errors of
// scripts/compute_errors.jl:30-70, for the top-k rule with k accepted
// particles per gene.
//
// Every gene owns a pool of capg = k + n_sub entries (error, particle index)
// in HBM.  Between batches a pool holds at most k entries: the gene's best k
// so far, and its threshold thr[g] is the k-th error.  One batch of at most
// n_sub particles then proceeds without a host round trip:
//   gemm_screen_kernel (abc_gemm.hip) appends each (particle, gene) pair whose
//     proven lower bound can reach thr[g] to the gene's pool (at most n_sub
//     new entries per gene, so a pool never overflows);
//   pool_rescore_kernel replaces each new entry by its FP64 error in the
//     reference operation order and its global particle index;
//   pool_select_kernel keeps each gene's k smallest (error, index) keys
//     (selected in LDS, or in place by a radix select over the 128-bit key) and
//     lowers thr[g] to the k-th error.
// list_sort_kernel orders each gene's final entries by (error, index) and packs
// them into the lists the host receives; the fixed-epsilon rule's accepted pairs
// reach it through list_scatter_kernel.
#include <hip/hip_runtime.h>

#include "abc_kernels.h"

namespace {

constexpr int kWG = 256;

// Order-preserving map of an FP64 value onto uint64 (x <= y iff key(x) <=
// key(y) for non-NaN values; errors are >= +0, but the map is total).
__device__ __forceinline__ uint64_t err_key(double e) {
  const uint64_t b = (uint64_t)__double_as_longlong(e);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double key_err(uint64_t k) {
  const uint64_t b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
  return __longlong_as_double((long long)b);
}

__device__ __forceinline__ bool key_le(uint64_t ah, uint64_t al, uint64_t bh, uint64_t bl) {
  return ah < bh || (ah == bh && al <= bl);
}

// Exclusive prefix of a per-thread flag over the 256 threads of the
// workgroup, in thread order; *total gets the sum.  Uses scratch[4].
__device__ __forceinline__ unsigned block_scan_flag(bool f, unsigned* scratch, unsigned* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long m = __ballot(f);
  const unsigned below = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
  if (lane == 0) scratch[wave] = (unsigned)__popcll(m);
  __syncthreads();
  unsigned pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kWG / 64; ++w) {
    const unsigned s = scratch[w];
    if (w < wave) pre += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return pre + below;
}

}  // namespace

// Workgroups (blockIdx.x over genes, grid-stride; blockIdx.y of gridDim.y
// over each gene's entries): the FP64 error of every entry appended since the
// last selection, in the order of compute_errors.jl:30-64 (no contraction),
// and its global particle index.  One lane per entry.  The batch's statistics
// are read in their column-major layout (row i, stat k at scol[i + ld k]):
// a gene's new entries come from the screen in nearly increasing row order,
// so the lanes' loads of one statistic are mostly contiguous.  An entry's
// index field holds its batch row on entry.
// The gene's data values, denominators and their reciprocals (genes[g K + k])
// are uniform over the workgroup: scalar loads, and quotients by the known
// denominators (div_by) unless the gene (gflag bit 1) or the particle (pflag
// bit 1) leaves the range for that.  2,000 genes x 4,096 rows x 90 statistics:
// 522 -> 363 us, bound by the L2 reads of the statistics (16 TB/s).
__global__ __launch_bounds__(256) void pool_rescore_kernel(
    const double* __restrict__ scol, int64_t ld, const ErrGene* __restrict__ genes,
    const uint8_t* __restrict__ gflag, const uint8_t* __restrict__ pflag, int64_t G, ErrSpec E,
    PoolEntry* __restrict__ pool, int64_t capg, const uint32_t* __restrict__ pool_n,
    const uint32_t* __restrict__ pool_base, int64_t first_index,
    const int64_t* __restrict__ pidx) {
  const int K = E.K;
  const Divisor dk = divisor_of((double)K);
  const int64_t stride = (int64_t)kWG * gridDim.y;
  for (int64_t g = blockIdx.x; g < G; g += gridDim.x) {
    const int64_t cnt = min((int64_t)pool_n[g], capg);
    const int64_t b = pool_base[g] + (int64_t)blockIdx.y * kWG;
    if (cnt <= b) continue;  // uniform over the workgroup
    const ErrGene* gg = genes + g * K;
    const bool gbad = (gflag[g] & 2) != 0;
    PoolEntry* pg = pool + g * capg;
    for (int64_t e = b + threadIdx.x; e < cnt; e += stride) {
      const int64_t i = pg[e].idx;
      const double* s = scol + i;
      double err = 0.0;
      int k = 0;
      if (!gbad && !(pflag[i] & 2)) {
        for (int pp = 0; pp < E.n_parts; ++pp) {
          double acc = 0.0;
          const int end = k + E.parts[pp];
#pragma unroll 5
          for (; k < end; ++k) {
            const ErrGene w = gg[k];
            const double diff = w.d - s[ld * k];
            acc += div_by(diff * diff, w.y, w.zh, w.zl);
          }
          err += div_by(acc, dk.y, dk.zh, dk.zl);
        }
      } else {
        for (int pp = 0; pp < E.n_parts; ++pp) {
          double acc = 0.0;
          const int end = k + E.parts[pp];
          for (; k < end; ++k) {
            const double diff = gg[k].d - s[ld * k];
            acc += (diff * diff) / gg[k].y;
          }
          err += acc / (double)K;
        }
      }
      if (err > E.clamp) err = E.clamp;
      pg[e] = PoolEntry{err, pidx ? pidx[i] : first_index + i};
    }
  }
}

// n rows were appended to every gene's pool
__global__ __launch_bounds__(256) void pool_grow_kernel(uint32_t* __restrict__ pool_n, int64_t G,
                                                        uint32_t n) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < G) pool_n[g] += n;
}

// The smallest and largest of a per-thread 64-bit key over the workgroup,
// through scratch (every thread gets them).
struct Extent {
  uint64_t lo, hi;
};
__device__ __forceinline__ Extent block_extent(uint64_t lo, uint64_t hi, uint64_t* scratch) {
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t a = (uint64_t)__shfl_xor((unsigned long long)lo, o);
    const uint64_t b = (uint64_t)__shfl_xor((unsigned long long)hi, o);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    scratch[2 * (threadIdx.x >> 6)] = lo;
    scratch[2 * (threadIdx.x >> 6) + 1] = hi;
  }
  __syncthreads();
  Extent r{scratch[0], scratch[1]};
#pragma unroll
  for (int w = 1; w < kWG / 64; ++w) {
    r.lo = scratch[2 * w] < r.lo ? scratch[2 * w] : r.lo;
    r.hi = scratch[2 * w + 1] > r.hi ? scratch[2 * w + 1] : r.hi;
  }
  return r;
}

// The key of rank r (0-based) among key(0 .. n - 1), counting only entries with
// use(e): 256 equal bins of the live range a turn, narrowed to the bin that
// holds the rank, until one value or one entry is left.  *rank: the rank among
// the entries equal to the result.
template <class Key, class Use>
__device__ __forceinline__ uint64_t block_select(int n, Key key, Use use, unsigned r,
                                                 unsigned* hist, uint64_t* scratch,
                                                 unsigned* s_pick, unsigned* rank) {
  const int tid = threadIdx.x;
  uint64_t lo = ~0ull, hi = 0ull;
  for (int e = tid; e < n; e += kWG)
    if (use(e)) {
      const uint64_t v = key(e);
      lo = v < lo ? v : lo;
      hi = v > hi ? v : hi;
    }
  Extent x = block_extent(lo, hi, scratch);
  while (x.lo < x.hi) {
    const uint64_t span = x.hi - x.lo;
    const int bits = 64 - __clzll((long long)span);
    const int sh = bits > 8 ? bits - 8 : 0;
    hist[tid] = 0u;
    __syncthreads();
    for (int e = tid; e < n; e += kWG)
      if (use(e)) {
        const uint64_t v = key(e);
        if (v >= x.lo && v <= x.hi) atomicAdd(&hist[(unsigned)((v - x.lo) >> sh)], 1u);
      }
    __syncthreads();
    if (tid < 64) {  // the bin of rank r: four bins a lane, a scan over the wave
      const unsigned h0 = hist[4 * tid], h1 = hist[4 * tid + 1], h2 = hist[4 * tid + 2],
                     h3 = hist[4 * tid + 3];
      const unsigned sum = h0 + h1 + h2 + h3;
      unsigned inc = sum;
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned y = __shfl_up(inc, o);
        if (tid >= o) inc += y;
      }
      const unsigned pre = inc - sum;
      if (r >= pre && r < inc) {
        unsigned at = pre, d = 0;
        if (r >= at + h0) { at += h0; d = 1;
          if (r >= at + h1) { at += h1; d = 2;
            if (r >= at + h2) { at += h2; d = 3; } } }
        s_pick[0] = 4 * tid + d;
        s_pick[1] = r - at;
        s_pick[2] = d == 0 ? h0 : (d == 1 ? h1 : (d == 2 ? h2 : h3));
      }
    }
    __syncthreads();
    const uint64_t blo = x.lo + ((uint64_t)s_pick[0] << sh);
    const uint64_t bhi = blo + ((1ull << sh) - 1ull);
    r = s_pick[1];
    x.lo = blo;
    x.hi = bhi < x.hi ? bhi : x.hi;
    if (s_pick[2] == 1u) {  // uniform: one entry left, r is 0
      for (int e = tid; e < n; e += kWG)
        if (use(e)) {
          const uint64_t v = key(e);
          if (v >= x.lo && v <= x.hi) scratch[0] = v;
        }
      __syncthreads();
      x.lo = x.hi = scratch[0];
    }
    __syncthreads();
  }
  *rank = r;
  return x.lo;
}

// One workgroup per gene (grid-stride): keep the k smallest (error, index)
// keys among the pool's entries with a non-NaN error (NaN errors are never
// accepted), compact them to the front of the pool, and lower thr[g] to the
// k-th error once the pool holds k entries.  Genes without new entries are
// skipped.  n_rescored accumulates the FP64 rescorings (entries appended since
// the last selection).
// kth[2 g], kth[2 g + 1] hold the complement of the k-th key (error, index) of
// the last selection (zeros: none yet): an entry beyond it cannot be among the
// k smallest, so it is dropped as the pool is read, once, into LDS, where the
// selection runs.  Pools with more than ABC_POOL_LDS live entries are selected
// in place, reading them from memory once per 8 bits of the key (the path every
// pool took before: 628 us for 2,000 pools of 5,096 entries, k = 1,000, against
// 161 us in LDS).
__global__ __launch_bounds__(256) void pool_select_kernel(
    PoolEntry* __restrict__ pool, int64_t capg, uint32_t* __restrict__ pool_n,
    uint32_t* __restrict__ pool_base, int64_t G, int64_t k, double* __restrict__ thr,
    unsigned long long* __restrict__ kth, unsigned long long* __restrict__ n_rescored) {
  __shared__ uint64_t lh[ABC_POOL_LDS], ll[ABC_POOL_LDS];
  __shared__ unsigned hist[256];
  __shared__ unsigned scratch[4], s_pick[3], s_live;
  __shared__ uint64_t s_ext[8];
  __shared__ uint64_t s_ph, s_pl, s_mh, s_ml;  // key prefix found so far and its mask
  __shared__ unsigned s_rank, s_bincnt, s_running;
  __shared__ uint64_t s_kh, s_kl;              // the k-th key
  const int tid = threadIdx.x, lane = tid & 63;
  for (int64_t g = blockIdx.x; g < G; g += gridDim.x) {
    const int64_t cnt = min((int64_t)pool_n[g], capg);
    const int64_t b = pool_base[g];
    if (cnt == b) continue;  // uniform
    PoolEntry* pg = pool + g * capg;
    const uint64_t LH = ~kth[2 * g], LL = ~kth[2 * g + 1];  // live: key <= (LH, LL)
    if (tid == 0) {
      atomicAdd(n_rescored, (unsigned long long)(cnt - b));
      s_running = 0;
      s_live = 0;
    }
    __syncthreads();
    // live entries into LDS (any order: the lists are sorted at the end), as
    // far as they fit, and their number
    for (int64_t base = 0; base < cnt; base += kWG) {
      const int64_t e = base + tid;
      uint64_t kh = 0, kl = 0;
      bool f = false;
      if (e < cnt) {
        const PoolEntry x = pg[e];
        kh = err_key(x.err);
        kl = (uint64_t)x.idx;
        f = (x.err == x.err) && key_le(kh, kl, LH, LL);
      }
      const unsigned long long m = __ballot(f);
      unsigned at = 0;
      if (lane == 0 && m) at = atomicAdd(&s_live, (unsigned)__popcll(m));
      at = __shfl(at, 0) + __builtin_amdgcn_mbcnt_hi(
                               (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      if (f && at < ABC_POOL_LDS) {
        lh[at] = kh;
        ll[at] = kl;
      }
    }
    __syncthreads();
    const unsigned tot = s_live;
    const bool keep_all = (int64_t)tot <= k;
    uint64_t KH = ~0ull, KL = ~0ull;  // the k-th key, once there are k
    if (tot <= ABC_POOL_LDS) {
      const int S = (int)tot;
      if (!keep_all && k > 0) {
        unsigned r;
        KH = block_select(
            S, [&](int e) { return lh[e]; }, [&](int) { return true; }, (unsigned)(k - 1), hist,
            s_ext, s_pick, &r);
        KL = block_select(
            S, [&](int e) { return ll[e]; }, [&](int e) { return lh[e] == KH; }, r, hist, s_ext,
            s_pick, &r);
      } else if ((int64_t)tot == k && k > 0) {  // the largest key
        uint64_t mh = 0, ml = 0;
        for (int e = tid; e < S; e += kWG) mh = lh[e] > mh ? lh[e] : mh;
        KH = block_extent(mh, mh, s_ext).hi;
        for (int e = tid; e < S; e += kWG)
          if (lh[e] == KH) ml = ll[e] > ml ? ll[e] : ml;
        KL = block_extent(ml, ml, s_ext).hi;
      }
      for (int base = 0; base < S && k > 0; base += kWG) {
        const int e = base + tid;
        const bool f = e < S && key_le(lh[e], ll[e], KH, KL);
        const unsigned long long m = __ballot(f);
        unsigned at = 0;
        if (lane == 0 && m) at = atomicAdd(&s_running, (unsigned)__popcll(m));
        at = __shfl(at, 0) + __builtin_amdgcn_mbcnt_hi(
                                 (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        if (f) pg[at] = PoolEntry{key_err(lh[e]), (int64_t)ll[e]};
      }
      __syncthreads();
    } else {
      if (!keep_all && k > 0) {
        // radix select of the key of rank k-1 among the live entries, 8 bits a
        // pass from the top of the 128-bit key (error bits, then index)
        if (tid == 0) { s_ph = s_pl = s_mh = s_ml = 0; s_rank = (unsigned)(k - 1); }
        for (int pass = 0; pass < 16; ++pass) {
          hist[tid] = 0;
          __syncthreads();
          const uint64_t ph = s_ph, pl = s_pl, mh = s_mh, ml = s_ml;
          const bool hi = pass < 8;
          const int sh = 56 - 8 * (pass & 7);
          for (int64_t e = tid; e < cnt; e += kWG) {
            const PoolEntry x = pg[e];
            if (!(x.err == x.err)) continue;
            const uint64_t kh = err_key(x.err), kl = (uint64_t)x.idx;
            if (!key_le(kh, kl, LH, LL)) continue;
            if ((kh & mh) != ph || (kl & ml) != pl) continue;
            atomicAdd(&hist[(unsigned)(((hi ? kh : kl) >> sh) & 0xFF)], 1u);
          }
          __syncthreads();
          if (tid == 0) {
            const unsigned r = s_rank;
            unsigned c = 0;
            int d = 0;
            for (; d < 255; ++d) {
              if (c + hist[d] > r) break;
              c += hist[d];
            }
            s_rank = r - c;
            s_bincnt = hist[d];
            if (hi) { s_ph |= (uint64_t)d << sh; s_mh |= 0xFFull << sh; }
            else { s_pl |= (uint64_t)d << sh; s_ml |= 0xFFull << sh; }
          }
          __syncthreads();
          if (s_bincnt == 1) break;  // uniform: the prefix now names one entry
        }
        // the full k-th key: the entry matching the prefix (after all 16 passes
        // every match carries the same key)
        const uint64_t ph = s_ph, pl = s_pl, mh = s_mh, ml = s_ml;
        for (int64_t e = tid; e < cnt; e += kWG) {
          const PoolEntry x = pg[e];
          if (!(x.err == x.err)) continue;
          const uint64_t kh = err_key(x.err), kl = (uint64_t)x.idx;
          if (!key_le(kh, kl, LH, LL)) continue;
          if ((kh & mh) == ph && (kl & ml) == pl) { s_kh = kh; s_kl = kl; }
        }
        __syncthreads();
        KH = s_kh;
        KL = s_kl;
      } else if ((int64_t)tot == k && k > 0) {  // the largest live key
        uint64_t mh = 0, ml = 0;
        for (int64_t e = tid; e < cnt; e += kWG) {
          const PoolEntry x = pg[e];
          const uint64_t kh = err_key(x.err);
          if (x.err == x.err && key_le(kh, (uint64_t)x.idx, LH, LL)) mh = kh > mh ? kh : mh;
        }
        KH = block_extent(mh, mh, s_ext).hi;
        for (int64_t e = tid; e < cnt; e += kWG) {
          const PoolEntry x = pg[e];
          const uint64_t kl = (uint64_t)x.idx;
          if (x.err == x.err && err_key(x.err) == KH && key_le(KH, kl, LH, LL))
            ml = kl > ml ? kl : ml;
        }
        KL = block_extent(ml, ml, s_ext).hi;
      }
      // in-place compaction of the kept entries: the positions a chunk writes
      // never exceed those it reads, and all its reads precede its writes
      const uint64_t BH = key_le(KH, KL, LH, LL) ? KH : LH, BL = key_le(KH, KL, LH, LL) ? KL : LL;
      for (int64_t base = 0; base < cnt && k > 0; base += kWG) {
        const int64_t e = base + tid;
        PoolEntry x{};
        bool f = false;
        if (e < cnt) {
          x = pg[e];
          f = (x.err == x.err) && key_le(err_key(x.err), (uint64_t)x.idx, BH, BL);
        }
        const unsigned run = s_running;
        unsigned total;
        const unsigned pos = block_scan_flag(f, scratch, &total);
        if (f) pg[run + pos] = x;
        if (tid == 0) s_running = run + total;
        __syncthreads();
      }
    }
    if (tid == 0) {
      const unsigned kept = s_running;
      pool_n[g] = kept;
      pool_base[g] = kept;
      if (k > 0 && (int64_t)kept >= k) {
        const double e = key_err(KH);
        if (e < thr[g]) thr[g] = e;
        kth[2 * g] = ~KH;
        kth[2 * g + 1] = ~KL;
      } else if (k <= 0) {
        thr[g] = -HUGE_VAL;
      }
    }
    __syncthreads();
  }
}

// Exclusive scan of the genes' entry counts (off[G] = all entries); clears the
// scatter cursors when there are any.  One workgroup, 1,024 genes a turn: the
// counts of a session are a few kilobytes.
__global__ __launch_bounds__(1024) void list_scan_kernel(const uint32_t* __restrict__ cnt,
                                                         int64_t G,
                                                         unsigned long long* __restrict__ off,
                                                         uint32_t* __restrict__ cursor) {
  __shared__ unsigned long long s[1024];
  const int t = threadIdx.x;
  unsigned long long carry = 0;
  for (int64_t g0 = 0; g0 < G; g0 += 1024) {
    const int64_t g = g0 + t;
    const unsigned long long x = g < G ? cnt[g] : 0ull;
    s[t] = x;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
      const unsigned long long y = t >= d ? s[t - d] : 0ull;
      __syncthreads();
      s[t] += y;
      __syncthreads();
    }
    if (g < G) {
      off[g] = carry + s[t] - x;
      if (cursor) cursor[g] = 0u;
    }
    carry += s[1023];
    __syncthreads();
  }
  if (t == 0) off[G] = carry;
}

// The fixed-epsilon rule's accepted pairs grouped by gene: entry q goes to
// ent[off[gene] + its place among the gene's entries so far].
__global__ __launch_bounds__(256) void list_scatter_kernel(const Candidate* __restrict__ acc,
                                                           int64_t n,
                                                           const unsigned long long* __restrict__ off,
                                                           uint32_t* __restrict__ cursor,
                                                           PoolEntry* __restrict__ ent) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const Candidate c = acc[q];
  ent[off[c.gene] + atomicAdd(cursor + c.gene, 1u)] = PoolEntry{c.err, c.particle};
}

// One workgroup per gene (grid-stride): the gene's cnt[g] entries, at ent + g *
// stride (ent + off[g] when stride is 0), sorted by (error, index), go to the
// flat lists the host receives: 1-based indices and errors from off[g] on.  Up
// to ABC_POOL_SORT_MAX entries are sorted here, a bitonic sort in LDS; a
// longer list is copied as it is and sorted by the host.  Sorting and packing
// on the device instead of on the host: abc_accept_end of 2,000 genes x 1,000
// entries 33 -> 3 ms, most of it the copy.
__global__ __launch_bounds__(256) void list_sort_kernel(const PoolEntry* __restrict__ ent,
                                                        int64_t stride,
                                                        const uint32_t* __restrict__ n_of,
                                                        const unsigned long long* __restrict__ off,
                                                        int64_t G, int64_t* __restrict__ idx_out,
                                                        double* __restrict__ err_out) {
  __shared__ uint64_t kh[ABC_POOL_SORT_MAX], kl[ABC_POOL_SORT_MAX];
  const int tid = threadIdx.x;
  for (int64_t g = blockIdx.x; g < G; g += gridDim.x) {
    const int64_t cnt = n_of[g];
    if (cnt == 0) continue;  // uniform
    const PoolEntry* pg = stride ? ent + g * stride : ent + off[g];
    const unsigned long long o = off[g];
    if (cnt > ABC_POOL_SORT_MAX) {
      for (int64_t e = tid; e < cnt; e += kWG) {
        idx_out[o + e] = pg[e].idx + 1;
        err_out[o + e] = pg[e].err;
      }
      continue;
    }
    int N = 1;
    while (N < cnt) N <<= 1;
    for (int e = tid; e < N; e += kWG) {
      if (e < cnt) {
        const PoolEntry x = pg[e];
        kh[e] = err_key(x.err);
        kl[e] = (uint64_t)x.idx;
      } else {
        kh[e] = ~0ull;
        kl[e] = ~0ull;
      }
    }
    __syncthreads();
    for (int size = 2; size <= N; size <<= 1) {
      for (int st = size >> 1; st > 0; st >>= 1) {
        for (int t = tid; t < N / 2; t += kWG) {
          const int i = 2 * t - (t & (st - 1));
          const int j = i + st;
          const bool up = (i & size) == 0;
          const bool gt = !key_le(kh[i], kl[i], kh[j], kl[j]);
          if (gt == up) {
            const uint64_t a = kh[i], c = kl[i];
            kh[i] = kh[j]; kl[i] = kl[j];
            kh[j] = a; kl[j] = c;
          }
        }
        __syncthreads();
      }
    }
    for (int e = tid; e < cnt; e += kWG) {
      idx_out[o + e] = (int64_t)kl[e] + 1;
      err_out[o + e] = key_err(kh[e]);
    }
    __syncthreads();
  }
}

// thr[g] = min(thr[g], lower[g]) for the G genes (known upper bounds of the
// k-th error supplied by the caller).
__global__ __launch_bounds__(256) void thr_min_kernel(double* __restrict__ thr,
                                                      const double* __restrict__ lower,
                                                      int64_t G) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < G && lower[g] < thr[g]) thr[g] = lower[g];
}
