// abc_kernels.h -- device data layouts and kernel declarations shared by the
// kernels and the C-ABI host layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "abc_device.h"

#define ABC_MAX_BINS 8
#define ABC_MAX_CONDS 16
#define ABC_MAX_STATS 256
#define ABC_MAX_PARTS 16
#define SSA_WG 256
#define ABC_NBUCKET 256      // cost buckets of the queue order
#define ABC_CELL_BUCKETS 1024  // 64 cost classes x 16 sub-lane counts of the cell order
#define ABC_LIGHT_CLASS 36     // cost classes below this are claimed several items at a time
#define ABC_CELL_TILE 4096     // cells one workgroup places in the cell order

// Experimental design in device memory (read through uniform scalar loads).
struct DesignDev {
  double T;                        // cycle length (h)
  int nb, J, C;                    // age bins, conditions, cells per particle
  int age_mode, cap_mode;          // 0 bin centres / 1 uniform; capture 0/1/2
  int beta_a, beta_b;              // integer Beta(a, b) for cap_mode 1
  int bmin, bmax;                  // burn-in cycle bounds
  int prior_mode, pad0;
  double burn_eps;                 // residual survival target of the burn-in
  double splice_log10;             // splicing rate for the reference prior
  double capture_mean;             // mean capture efficiency (cost estimate)
  double split_target;             // molecule events per sub-lane (0 = no split)
  double split_scale;              // capture scale used by the split rule
  double wmax;                     // longest labelling window (pulse + chase), h
  int split_max, pad1;
  double pulse[ABC_MAX_CONDS], chase[ABC_MAX_CONDS];
  int is_chase[ABC_MAX_CONDS];
  double bound[ABC_MAX_BINS];      // T * (nb + j + 1) / nb (thinning bound, h)
  double weights[ABC_MAX_BINS * ABC_MAX_CONDS];  // age weights, col-major nb x J
};

// Per-particle rates (1/h) for each age bin.
struct __align__(16) PRates {
  double kon[ABC_MAX_BINS], koff[ABC_MAX_BINS], amax[ABC_MAX_BINS], gam[ABC_MAX_BINS];
  // 1 / kon, 1 / koff, 1 / (gam + splicing), 1 / gam per bin (the same IEEE
  // quotients the event loops would form at every bin edge)
  double ikon[ABC_MAX_BINS], ikoff[ABC_MAX_BINS], iku[ABC_MAX_BINS], ikt[ABC_MAX_BINS];
  double bs;                       // splicing rate
  double brate;                    // mean over the bins of alpha_max * P(gene on)
  uint64_t thr_lam;                // floor(lambda * 2^32): labelling threshold
  uint64_t thr_pi;                 // floor(P(gene on at cycle start) * 2^32)
  int32_t B, step, scaling;        // burn-in cycles, grid stride, size scaling
  int32_t gene_varies;             // kon differs between bins (burst-frequency model)
  float swrate, gmean;             // gene switches and decays per hour, means over the bins
                                   // (queue-order keys only)
  int32_t pad[2];
};

// A cell at the start of its labelling window (burn_kernel -> ssa_kernel).
struct __align__(16) CellStart {
  double age, bc;   // sampling age (h), capture efficiency
  double tg;        // next gene switch (absolute time)
  double lu, lt;    // Poisson means of the unspliced / all unlabelled molecules
  int64_t k;        // last grid edge passed
  uint64_t gctr;    // gene-stream counter
  uint8_t bin, g, gneed;
  uint8_t msh;      // log2 of the cell's sub-lanes M
};

// Tables of the cell order (cell_scan_kernel), by rank from the heaviest
// bucket: first item (and all items at the end), first cell, scatter cursor;
// and the expected draws of all items, by their classes.
struct CellTables {
  unsigned long long ioff[ABC_CELL_BUCKETS + 1];
  double draws;
  unsigned cbase[ABC_CELL_BUCKETS], cursor[ABC_CELL_BUCKETS];
};

struct ErrSpec {
  int K, n_parts;
  int parts[ABC_MAX_PARTS];
  double clamp;
};

// denominator of a squared difference (compute_errors.jl:30-43)
ABC_DEV double err_den(double d, double sg) {
  const double s2 = 0.1 * 0.1;
  const double eps = (sg + d != 0.0) ? 0.0 : 0.0001;
  return (sg * sg + s2 * (d * d)) + eps;
}

// ---- x / y for a divisor known in advance, correctly rounded without the
// division sequence (about 16 issue slots): with zh = RN(1 / y) and zl = 1 / y -
// zh, q = RN(x zh + RN(x zl)) is within an ulp of x / y, so x - q y is exact in
// one fused multiply-add and RN(q + (x - q y) zh) is RN(x / y) (Markstein, IBM
// J. Res. Dev. 34, 1990).  x >= 0; neither x, y nor the quotient may come near
// the ends of the exponent range: err_range below bounds the operands.
struct Divisor {
  double y, zh, zl;
};
ABC_DEV Divisor divisor_of(double y) {
  const double zh = 1.0 / y;
  return Divisor{y, zh, fma(-zh, y, 1.0) * zh};
}
ABC_DEV double div_by(double x, double y, double zh, double zl) {
  const double q = fma(x, zh, x * zl);
  return fma(fma(-q, y, x), zh, q);
}
// v is zero or 2^-120 <= |v| < 2^200: differences of two such values are zero
// or at least 2^-172, their squares over a denominator in [2^-300, 2^300] and
// the remainders above stay normal numbers.  NaN is in range too: it makes the
// quotient, and so the error, NaN either way.
ABC_DEV bool err_range(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t e = (uint32_t)(b >> 52) & 0x7FFu;
  return (e - (1023u - 120u)) < 320u || (b << 1) - 1ull >= 0xFFE0000000000000ull;  // 0 or NaN
}
ABC_DEV bool den_range(double y) {
  const uint32_t e = (uint32_t)((uint64_t)__double_as_longlong(y) >> 52);  // y > 0: no sign bit
  return (e - (1023u - 300u)) < 600u || y != y;
}
// data value and denominator of a gene; an infinite value's denominator is
// infinite (or NaN) and every quotient NaN, by div_by as by a division
ABC_DEV bool gene_range(double d, double y) {
  return (err_range(d) && den_range(y)) || __builtin_isinf(d);
}

// One gene's data value and denominator for one statistic.
struct __align__(32) ErrGene {
  double d, y, zh, zl;
};

// One entry of a gene's acceptance pool (abc_accept.hip): the FP64 error
// and the global 0-based particle index (the batch row until rescored).
struct PoolEntry {
  double err;
  int64_t idx;
};
#define ABC_POOL_SORT_MAX 2048  // entries per gene sorted on the device
#define ABC_POOL_LDS 4096       // entries per gene selected in LDS

struct Candidate {
  double err;
  int64_t particle;  // global 0-based particle index
  int32_t gene;
  int32_t pad;
};

int abc_layout_n_params(int model, int nb);

__global__ void prior_kernel(const DesignDev* D, int model, uint32_t k0, uint32_t k1,
                             uint32_t first, int64_t n, double* theta);
__global__ void rates_kernel(const DesignDev* D, int model, int64_t n, const double* theta,
                             PRates* R, float* cost);
__global__ void bucket_hist_kernel(const float* cost, int64_t n, unsigned* hist);
__global__ void bucket_scan_kernel(const unsigned* hist, unsigned* cursor);
__global__ void bucket_scatter_kernel(const float* cost, int64_t n, unsigned* cursor,
                                      int32_t* order);
__global__ void cell_hist_kernel(const uint32_t* key, int64_t cells, unsigned* hist);
__global__ void cell_scan_kernel(const unsigned* hist, CellTables* T);
__global__ void cell_scatter_kernel(const uint32_t* key, int64_t cells, CellTables* T,
                                    uint32_t* cellord);
__global__ void fill_ids_kernel(int64_t n, int64_t first, const int64_t* src, uint32_t mtag,
                                int64_t* pidx, uint32_t* mtags);
__global__ void copy_u64_kernel(const unsigned long long* src, unsigned long long* dst,
                                int64_t n);
__global__ void burn_kernel(const DesignDev* D, const PRates* R, const int32_t* order, int64_t n,
                            uint32_t first, uint32_t k0, uint32_t k1, uint32_t mtag_all,
                            const uint32_t* mtags, const double* betas,
                            const int64_t* goff, unsigned long long* queue, CellStart* rec,
                            uint32_t* cellkey, unsigned long long* steps_out,
                            const int64_t* pidx, unsigned long long* burn_tally);
__global__ void ssa_kernel(const DesignDev* D, const PRates* R, const CellTables* tabs,
                           const uint32_t* cellord, uint32_t first, uint32_t k0,
                           uint32_t k1, uint32_t mtag_all, const uint32_t* mtags,
                           const CellStart* rec,
                           unsigned long long* queue,
                           uint32_t* out_u, uint32_t* out_l, uint8_t* out_bin,
                           unsigned long long* steps_out,
                           const int64_t* pidx, uint32_t claim);
// Moment model (the reference simulator, scripts/model.jl): one call's
// configuration, passed by value as a kernel argument (about 1.9 kB).
#define ABC_MOM_MAX_AGES ABC_MAX_BINS
#define ABC_MOM_MAX_CONDS ABC_MAX_CONDS
struct MomCfgDev {
  double cycle;          // cell-cycle length T
  int n_steps;           // rate bins per cycle
  int n_ages, n_conds;
  int transient_mode;    // 0 = 1 % rule (model.jl:114-142), 1 = exact periodic state
  double t0;             // trajectory start
  double iv[9];          // transient start state
  double rtol, atol;     // Dormand-Prince tolerances
  int method;            // 0 = Dormand-Prince on all nine moments, 1 = gene block exact
  double ages[ABC_MOM_MAX_AGES];
  double pulse[ABC_MOM_MAX_CONDS], chase[ABC_MOM_MAX_CONDS];
  int is_chase[ABC_MOM_MAX_CONDS];
  int downsample;        // apply the capture moments below
  int pulse_cond, chase_cond;  // conditions feeding the mean / Fano statistics (-1: none)
  double cap[ABC_MOM_MAX_AGES * 2 * 3];  // per (age, pulse/chase): E b, E b^2, Var b
  double weights[ABC_MOM_MAX_AGES * ABC_MOM_MAX_CONDS];  // age weights, n_ages x n_conds
};
template <int METHOD>
__global__ void moment_cyclemap_kernel(MomCfgDev cfg, int model, int64_t n,
                                       const double* theta, int64_t ld, const int32_t* order,
                                       int64_t heavy, double* maps, unsigned long long* cost,
                                       unsigned long long* steps);
__global__ void moment_key_kernel(MomCfgDev cfg, int model, int64_t n, const double* theta,
                                  int64_t ld, unsigned long long* cost);
// particle order for the cycle-map and trajectory kernels: descending cost
#define ABC_MOM_ORDER_WG 1024
#define ABC_MOM_COST_BUCKETS 1024
__global__ void moment_order_kernel(int64_t n, const unsigned long long* cost, int32_t* order);
__global__ void moment_transient_kernel(MomCfgDev cfg, int64_t n, const double* maps,
                                        double* ss);
template <int METHOD>
__global__ void moment_traj_kernel(MomCfgDev cfg, int model, int64_t n,
                                   const double* theta, int64_t ld, const double* ss,
                                   const double* maps, const int32_t* order, int64_t heavy,
                                   double* out,
                                   unsigned long long* steps);
__global__ void moment_stats_kernel(MomCfgDev cfg, int64_t n, double* mom,
                                    double* stats);
// Data-side summary statistics with bootstrap SEs (scripts/data_summary_statistics.jl)
#define ABC_DATA_WG 256
#define ABC_DATA_MAX_CLUSTERS 8
#define ABC_DATA_MAX_CONDS 16
__global__ void data_stats_kernel(int64_t G, int64_t g0, int64_t n, const uint32_t* u,
                                  const uint32_t* l,
                                  const int32_t* age, const int32_t* cond, int nc, int J,
                                  const int32_t* pulse, int64_t np, const int32_t* chase,
                                  int64_t nch, const double* w_point, int n_boot, uint32_t k0,
                                  uint32_t k1, double* boot, double* out, unsigned int* bad_out);
#define ABC_DATA_SORTED_MAX 16384  // cells per family for data_stats_sorted_kernel (32 KiB of draw counters)
#define ABC_DATA_SETS_PER_WG 8    // sets per workgroup of data_stats_sorted_kernel
__global__ void data_pack_kernel(int64_t n, const uint32_t* u, const uint32_t* l, int64_t g0,
                                 const int32_t* pulse, int64_t np, const int32_t* chase,
                                 int64_t nch, const int32_t* perm, const int32_t* grp,
                                 int64_t slots, int64_t genes, unsigned long long* xs,
                                 uint32_t* xmax, unsigned int* bad_out);
__global__ void data_check_kernel(int64_t n, const uint32_t* u, const uint32_t* l,
                                  unsigned int* bad_out);
size_t data_sorted_lds(int64_t mm);  // its LDS bytes, for families of up to mm cells
template <bool SMALL>
__global__ void data_stats_sorted_kernel(int64_t genes, int nsb, int64_t g0,
                                         const unsigned long long* xs, int64_t slots,
                                         const uint32_t* xmax, int64_t n,
                                         int64_t np, int64_t nch, int nc, int J,
                                         const double* w_point, int n_boot, int spb, uint32_t k0,
                                         uint32_t k1, double* pt, double* boot);
__global__ void data_se_kernel(int64_t G, int64_t g0, int64_t genes, int nc, int J, int n_boot,
                               const double* pt, const double* boot, double* out);
// Model probabilities with bootstrap bounds (scripts/model_probs.jl)
#define ABC_SEL_WG 256
#define ABC_SEL_MAX_GROUPS 8
#define ABC_SEL_MAX_BOOT 256
#define ABC_SEL_BOOT_PER_WG 8  // resamples per workgroup of model_prob_kernel
template <int M>
__global__ void model_prob_kernel(int64_t G, int64_t g0, const int64_t* counts,
                                  uint32_t k0, uint32_t k1, int n_boot, int rpb, double* shares,
                                  double* prob, double* lb, double* ub);
__global__ void model_prob_bounds_kernel(int64_t G, int64_t g0, int M, const int64_t* counts,
                                         int n_boot, double alpha, const double* shares,
                                         double* prob, double* lb, double* ub);
__global__ void stats_kernel(const DesignDev* D, const uint32_t* cu, const uint32_t* cl,
                             const uint8_t* cb, int64_t n, double* stats_ref, double* moments,
                             double* superset);
__global__ void err_fp64_kernel(const double* stats, int64_t n, const double* data,
                                const double* se, int64_t G, int64_t g0, ErrSpec E, double* err);
template <int PT, bool POOL>
__global__ void err_tile_kernel(const double* stats, int64_t n, int64_t ld, const double* data,
                                const double* se, int64_t G, ErrSpec E, double* err_out,
                                PoolEntry* pool, int64_t capg, int64_t first_index,
                                const int64_t* pidx, const uint32_t* pool_n);
__global__ void zero_u64_kernel(unsigned long long* p, int64_t n);
__global__ void math_probe_kernel(int kind, int64_t n, const double* x, double* y);

// screening (abc_gemm.hip)
__global__ void gene_prep_kernel(const double* data, const double* se, int64_t G, int K, int Kp,
                                 int64_t Gpad, __bf16* Bh, __bf16* Bl, double* cg, uint8_t* gflag,
                                 float* Wf, ErrGene* genes);
// surrogate screen (abc_mlp.hip)
#define ABC_SCREEN_PT 8  // particles per workgroup of screen_kernel
template <bool SCORE>
__global__ void screen_kernel(const float* y, int64_t n, int K, const float* mean, const float* sd,
                              float z, const float* Wf, const double* data, int64_t G,
                              const double* thr, float margin, double clamp, uint8_t* pass, float* score);
struct abc_mlp;
extern "C" int32_t abc_mlp_forward_dev(abc_mlp* p, int64_t n, const float* x_dev, float* y_dev);
extern "C" int32_t abc_mlp_synchronize(abc_mlp* p);
extern "C" int32_t abc_mlp_n_stats(const abc_mlp* p);
__global__ void particle_prep_kernel(const double* stats, int64_t n, int64_t ld, int K, int Kp,
                                     int64_t npad,
                                     __bf16* Ah, __bf16* Al, uint8_t* pflag);
__global__ void gemm_screen_kernel(const __bf16* Ah, const __bf16* Al, int64_t n, int Kp,
                                   const __bf16* Bh, const __bf16* Bl, int64_t G, const double* cg,
                                   const uint8_t* gflag, const uint8_t* pflag, const double* thr,
                                   double margin_rel, double clamp, Candidate* out,
                                   unsigned long long* count, unsigned long long cap,
                                   float* approx_out, float* bound_out, PoolEntry* pool,
                                   int64_t capg, uint32_t* pool_n);
// per-gene top-k pools (abc_accept.hip)
__global__ void pool_rescore_kernel(const double* scol, int64_t ld, const ErrGene* genes,
                                    const uint8_t* gflag, const uint8_t* pflag, int64_t G,
                                    ErrSpec E, PoolEntry* pool, int64_t capg,
                                    const uint32_t* pool_n, const uint32_t* pool_base,
                                    int64_t first_index, const int64_t* pidx);
__global__ void pool_grow_kernel(uint32_t* pool_n, int64_t G, uint32_t n);
__global__ void pool_select_kernel(PoolEntry* pool, int64_t capg, uint32_t* pool_n,
                                   uint32_t* pool_base, int64_t G, int64_t k, double* thr,
                                   unsigned long long* kth,
                                   unsigned long long* n_rescored);
__global__ void list_scan_kernel(const uint32_t* cnt, int64_t G, unsigned long long* off,
                                 uint32_t* cursor);
__global__ void list_scatter_kernel(const Candidate* acc, int64_t n,
                                    const unsigned long long* off, uint32_t* cursor,
                                    PoolEntry* ent);
__global__ void list_sort_kernel(const PoolEntry* ent, int64_t stride, const uint32_t* n_of,
                                 const unsigned long long* off, int64_t G, int64_t* idx_out,
                                 double* err_out);
__global__ void thr_min_kernel(double* thr, const double* lower, int64_t G);
__global__ void rescore_kernel(const double* stats, int64_t n, const double* data,
                               const double* se, int64_t G, ErrSpec E, const Candidate* cand,
                               const unsigned long long* count, unsigned long long cap,
                               int64_t q0, int64_t q1, double eps_acc, int64_t first_index,
                               const int64_t* pidx, Candidate* acc, unsigned long long room,
                               unsigned long long* n_acc, uint32_t* gene_n);
