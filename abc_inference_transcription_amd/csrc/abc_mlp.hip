// abc_mlp.hip -- the surrogate: an MLP from (model, log10 parameters) to the
// mean and log-variance of every summary statistic, trained on the simulator's
// own output, and the screen that lets the exact simulation run only on
// particles that can still be accepted.  No reference counterpart (the
// reference simulates every prior particle, scripts/abc_simulation.jl:88-97).
//
// Network: x (n_in, zero-padded to 64) -> [width, SiLU] x depth -> n_out
// (padded to a multiple of 64).  Every product is a bf16 "NT" GEMM
// C[m][n] = sum_k A[m][k] * B[n][k] on v_mfma_f32_16x16x32_bf16 with FP32
// accumulation: forward Z = H W^T, backward dH = dZ W (W kept transposed as a
// second bf16 copy), dW = dZ^T H (epilogues store the transposed activations
// these need).  Master weights, gradients and Adam moments are FP32.
#include <hip/hip_runtime.h>

#include <cmath>
#include <random>
#include <string>
#include <vector>

#include "../../include/abc.h"
#include "abc_kernels.h"

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

enum { EPI_F32 = 0, EPI_SILU = 1, EPI_DSILU = 2, EPI_DW = 3 };

// K per pipeline stage (32-deep MFMA steps): 64, and 128 for the weight gradients
// in 64 x 64 tiles, whose few workgroups per CU wait at every stage's barrier.
// Larger tiles are for products that fill the machine, where the LDS of a deeper
// stage leaves room for one workgroup per CU instead of two (a step of width
// 4,096 and 8,192 samples 1,700 us with 128, 1,600 with 64).
constexpr int stage_k(int epi, int bm, int bn) { return epi == EPI_DW && bm * bn == 64 * 64 ? 128 : 64; }
constexpr int kDwChunk = 128;  // a chunk of a split gradient is whole stages

// s = 1 / (1 + e^-z) of four values.  The reciprocals of x = 1 + e^-z >= 1 are
// correctly rounded without the division sequence: the hardware's reciprocal
// and one Newton step give the division's bits for every x in [1, 2^126)
// (compared for all of them on gfx950); beyond, where the reciprocal is
// subnormal or x infinite, all four divide.
__device__ __forceinline__ void sigm4(const float* z, float* s) {
  float x[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    x[q] = 1.0f + __expf(-z[q]);
    const float r = __builtin_amdgcn_rcpf(x[q]);
    s[q] = fmaf(fmaf(-x[q], r, 1.0f), r, r);
  }
  if (fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])) >= 0x1p126f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = 1.0f / x[q];
  }
}

struct GemmArgs {
  const bf16 *A, *B;
  int M, N, K, ld;
  const float* bias;
  float* Cf;
  bf16 *Cb, *CbT;
  const float* Zprev;
  float* Zout;
};

// 256 threads, workgroup tile BM x BN (128 or 64 each), wave tile BM/2 x BN/2 (2
// x 2 waves).  EPI_DW sums K chunk z, [z*K, (z+1)*K), of rows with leading
// dimension ld (all of K): it writes its partial tile to Cf + z*M*N, and the
// partial row sums of A, its product with a column of ones, to Zout + z*M: a
// weight gradient and its bias's in one launch.  K advances in stages of BK
// through two LDS buffers: while the MFMAs read one stage, the next is loaded
// from global memory into registers and stored to the other buffer, one barrier
// per stage.  8,192 x 512 x 512 with the SiLU epilogue: 13.6 us, 8 of them its
// 34 MB of stores (K = 64 takes as long), then 0.8 us per stage; two or four
// stages in flight, padded rows, or B from the L2 in fragment order measured
// within 0.3 us or slower.  Every output sums its K in order, 32 at a time,
// whatever the tile.
template <int BM, int BN, int EPI>
__global__ __launch_bounds__(256) void gemm_nt_kernel(const bf16* __restrict__ A,
                                                      const bf16* __restrict__ B, int M, int N,
                                                      int K, int ld, const float* __restrict__ bias,
                                                      float* __restrict__ Cf,
                                                      bf16* __restrict__ Cb,
                                                      bf16* __restrict__ CbT,
                                                      const float* __restrict__ Zprev,
                                                      float* __restrict__ Zout) {
  constexpr int WN = BN / 2, NCB = WN / 16;
  constexpr int WM = BM / 2, NRB = WM / 16;
  constexpr int BK = stage_k(EPI, BM, BN), LDSK = BK + 8;  // 8 of padding against bank conflicts
  constexpr int BQ = BK / 8;                       // 16-byte pieces of a row's stage
  constexpr int NAQ = BM * BQ / 256, NBQ = BN * BQ / 256;
  __shared__ bf16 As[2][BM][LDSK];
  __shared__ bf16 Bs[2][BN][LDSK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // EPI_DW: K chunks fastest, so that one XCD's workgroups (every eighth) share
  // their chunks of A and B; with the row tiles fastest each XCD read an eighth
  // of A and all of B (8,192 x 512 x 512: 14.4 us, 13.7 so)
  const int bx = EPI == EPI_DW ? blockIdx.y : blockIdx.x;
  const int by = EPI == EPI_DW ? blockIdx.z : blockIdx.y, bz = EPI == EPI_DW ? blockIdx.x : 0;
  const int m0 = bx * BM, n0 = by * BN;
  const int kbeg = bz * K, kend = min(kbeg + K, ld);  // empty: past the last chunk
  if (EPI == EPI_DW) {
    Cf += (size_t)bz * M * N;
    Zout += (size_t)bz * M;
  }
  const bool rows = EPI == EPI_DW && by == 0 && wn == 0;  // the wave sums A's rows
  const bf16 one = (bf16)1.0f;
  const bf16x8 ones = {one, one, one, one, one, one, one, one};
  f32x4 rs[NRB];
#pragma unroll
  for (int a = 0; a < NRB; ++a) rs[a] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc[NRB][NCB];
#pragma unroll
  for (int a = 0; a < NRB; ++a)
#pragma unroll
    for (int b = 0; b < NCB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this thread's slice of a stage: rows c / BQ, 8 columns at c % BQ * 8
  bf16x8 ra[NAQ], rb[NBQ];
  auto load = [&](int k0) {
#pragma unroll
    for (int q = 0; q < NAQ; ++q) {
      const int c = tid + q * 256;
      ra[q] = *reinterpret_cast<const bf16x8*>(A + (size_t)(m0 + c / BQ) * ld + k0 + c % BQ * 8);
    }
#pragma unroll
    for (int q = 0; q < NBQ; ++q) {
      const int c = tid + q * 256;
      rb[q] = *reinterpret_cast<const bf16x8*>(B + (size_t)(n0 + c / BQ) * ld + k0 + c % BQ * 8);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int q = 0; q < NAQ; ++q) {
      const int c = tid + q * 256;
      *reinterpret_cast<bf16x8*>(&As[buf][c / BQ][c % BQ * 8]) = ra[q];
    }
#pragma unroll
    for (int q = 0; q < NBQ; ++q) {
      const int c = tid + q * 256;
      *reinterpret_cast<bf16x8*>(&Bs[buf][c / BQ][c % BQ * 8]) = rb[q];
    }
  };
  if (kbeg < kend) {
    load(kbeg);
    stash(0);
  }
  __syncthreads();
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    const bool more = k0 + BK < kend;
    if (more) load(k0 + BK);  // in flight while the MFMAs below run
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      bf16x8 af[NRB], bfr[NCB];
#pragma unroll
      for (int r4 = 0; r4 < NRB; ++r4)
        af[r4] = *reinterpret_cast<const bf16x8*>(
            &As[buf][wm * WM + r4 * 16 + (lane & 15)][ks * 32 + (lane >> 4) * 8]);
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
        bfr[cb] = *reinterpret_cast<const bf16x8*>(
            &Bs[buf][wn * WN + cb * 16 + (lane & 15)][ks * 32 + (lane >> 4) * 8]);
#pragma unroll
      for (int r4 = 0; r4 < NRB; ++r4)
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
          acc[r4][cb] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[r4], bfr[cb], acc[r4][cb], 0, 0, 0);
      if (rows)
#pragma unroll
        for (int r4 = 0; r4 < NRB; ++r4)
          rs[r4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[r4], ones, rs[r4], 0, 0, 0);
    }
    if (more) stash(buf ^ 1);  // the other buffer: its last readers passed the barrier below
    __syncthreads();
    buf ^= 1;
  }
  if (rows && (lane & 15) == 0)
#pragma unroll
    for (int r4 = 0; r4 < NRB; ++r4)
      *reinterpret_cast<f32x4*>(Zout + m0 + wm * WM + r4 * 16 + (lane >> 4) * 4) = rs[r4];
#pragma unroll
  for (int r4 = 0; r4 < NRB; ++r4)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      // this lane's 4 outputs are rows m..m+3 of column n: one 8-byte store
      // of the transposed copy (rows consecutive in C^T)
      const int mb = m0 + wm * WM + r4 * 16 + (lane >> 4) * 4;
      const int n = n0 + wn * WN + cb * 16 + (lane & 15);
      bf16x4 tv;
      float z[4], s[4];
      if (EPI == EPI_SILU || EPI == EPI_DSILU) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          z[q] = EPI == EPI_SILU ? acc[r4][cb][q] + bias[n] : Zprev[(size_t)(mb + q) * N + n];
        sigm4(z, s);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = mb + q;
        float v = acc[r4][cb][q];
        const size_t o = (size_t)m * N + n;
        if (EPI == EPI_F32) {
          v += bias[n];
          Cf[o] = v;
        } else if (EPI == EPI_DW) {
          Cf[o] = v;
        } else if (EPI == EPI_SILU) {
          Zout[o] = z[q];
          const bf16 h = (bf16)(z[q] * s[q]);
          Cb[o] = h;
          tv[q] = h;
        } else {
          const bf16 d = (bf16)(v * (s[q] * (1.0f + z[q] * (1.0f - s[q]))));
          Cb[o] = d;
          tv[q] = d;
        }
      }
      if (EPI == EPI_SILU || EPI == EPI_DSILU)
        *reinterpret_cast<bf16x4*>(CbT + (size_t)n * M + mb) = tv;
    }
}

// x (B x n_in FP32, row-major) -> X (B x in_pad bf16) and X^T (in_pad x B), one
// workgroup per 64 x 64 tile, the transpose through LDS (element by element,
// its scattered 2-byte stores took 7.0 us for 8,192 x 64, 4.2 so).
__global__ __launch_bounds__(256) void cast_input_kernel(const float* __restrict__ x, int Bn,
                                                         int Bpad, int n_in, int in_pad,
                                                         bf16* __restrict__ X,
                                                         bf16* __restrict__ XT) {
  __shared__ bf16 tile[64][64 + 2];
  const int b0 = blockIdx.x * 64, k0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int k = k0 + tx;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int b = b0 + 4 * i + ty;
    v[i] = x[(size_t)(b < Bn ? b : 0) * n_in + (k < n_in ? k : 0)];
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int b = b0 + 4 * i + ty;
    const bf16 h = (bf16)(b < Bn && k < n_in ? v[i] : 0.0f);
    X[(size_t)b * in_pad + k] = h;
    tile[4 * i + ty][tx] = h;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i)
    XT[(size_t)(k0 + 4 * i + ty) * Bpad + b0 + tx] = tile[tx][4 * i + ty];
}

// the sum of 256 threads' values, in thread 0
__device__ __forceinline__ float block_sum(float x, float* red) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// The loss from nll_kernel's n tiles, by one workgroup: *loss, and *out if given.
__device__ __forceinline__ void loss_total(const float* __restrict__ parts, int n,
                                           float* __restrict__ loss, float* __restrict__ out) {
  __shared__ float red[4];
  float x = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) x += parts[i];
  x = block_sum(x, red);
  if (threadIdx.x != 0) return;
  *loss = x;
  if (out) *out = x;
}

// Gaussian negative log-likelihood per element, mean over B*ns.
// O row: [mu (ns) | logvar (ns) | pad]; dO and dO^T in bf16.  The first n_cnt
// statistics are counts: their mu slot is a log-rate o with the Poisson
// negative log-likelihood exp(o) - t o (log t! dropped) on [-30, 8], continued
// linearly outside (the gradient there is the bound's, exp(bound) - t, so an
// output that strays is pulled back and exp never overflows), and their
// logvar slot is unused.
// One workgroup per 64 x 64 tile of (sample b, output k): the gradient is
// written row-major to dO with k fastest, and through an LDS transpose to dO^T
// with b fastest, so both stores are coalesced.  The tile's share of the loss
// goes to loss[tile], summed by loss_total (with one float atomic per tile, 512 at
// one address, 8,192 samples of 180 outputs took 12.1 us, 7.0 so).
__global__ __launch_bounds__(256) void nll_kernel(const float* __restrict__ O,
                                                  const float* __restrict__ T, int Bn, int Bpad,
                                                  int ns, int n_cnt, int out_pad,
                                                  bf16* __restrict__ dO, bf16* __restrict__ dOT,
                                                  float* __restrict__ loss) {
  __shared__ bf16 tile[64][64 + 2];
  __shared__ float red[4];
  const int b0 = blockIdx.x * 64, k0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 columns x 4 rows per pass
  const float scale = 1.0f / ((float)Bn * (float)ns);
  float l = 0.0f;
  const int k = k0 + tx, s = k < ns ? k : k - ns;
  const bool out = k < 2 * ns;
  // eight rows' loads in flight at a time
#pragma unroll
  for (int h = 0; h < 16; h += 8) {
    float mu8[8], lv8[8], y8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int b = b0 + 4 * (h + i) + ty;
      const size_t bb = b < Bn ? b : 0, ss = out ? s : 0;
      mu8[i] = O[bb * out_pad + ss];
      lv8[i] = O[bb * out_pad + ns + ss];
      y8[i] = T[bb * ns + ss];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rr = 4 * (h + i) + ty, b = b0 + rr;
      float g = 0.0f;
      if (b < Bn && out) {
        const float mu = mu8[i], lv_raw = lv8[i], y = y8[i];
        const bool clipped = lv_raw < -12.0f || lv_raw > 12.0f;
        const float lv = fminf(fmaxf(lv_raw, -12.0f), 12.0f);
        const float r = y - mu;
        const float inv = __expf(-lv);
        if (s < n_cnt) {
          if (k < ns) {
            const float o = fminf(fmaxf(mu, -30.0f), 8.0f);
            const float lam = __expf(o);
            g = (lam - y) * scale;
            l += ((lam - y * o) + (lam - y) * (mu - o)) * scale;
          }
        } else if (k < ns) {
          g = -r * inv * scale;
          l += 0.5f * (lv + r * r * inv) * scale;
        } else {
          g = clipped ? 0.0f : 0.5f * (1.0f - r * r * inv) * scale;
        }
      }
      const bf16 gb = (bf16)g;
      dO[(size_t)b * out_pad + k] = gb;
      tile[rr][tx] = gb;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i)
    dOT[(size_t)(k0 + 4 * i + ty) * Bpad + b0 + tx] = tile[tx][4 * i + ty];
  l = block_sum(l, red);
  if (threadIdx.x == 0) loss[blockIdx.y * gridDim.x + blockIdx.x] = l;
}

struct LayerDesc {
  int in, out;      // padded dims
  int64_t w_off;    // offset of W (out x in) in the flat parameter array
  int64_t b_off;    // offset of b (out)
};

// place of weight (o, i) of an out x in layer in the fragment-ordered copy: the
// 16 x 32 MFMA operand tiles (o / 16, i / 32), each as its 64 lanes' 16 bytes
__device__ __forceinline__ int64_t frag_at(int o, int i, int in) {
  return ((int64_t)(o >> 4) * in + (i & ~31)) * 16 + ((o & 15) + ((i >> 3) & 3) * 16) * 8 + (i & 7);
}

// One workgroup per 64 x 64 tile of a layer's weights (dims.x of them in all, in
// layer order), then one per 256 biases: tile and layer of workgroup `blk`.
struct TilePos {
  int layer, o0, i0;  // layer < 0: biases, o0 the first of the 256 (over all layers)
};
__device__ __forceinline__ TilePos tile_pos(int blk, const LayerDesc* __restrict__ L, int nl) {
  for (int l = 0; l < nl; ++l) {
    const int ti = L[l].in / 64, t = L[l].out / 64 * ti;
    if (blk < t) return TilePos{l, blk / ti * 64, blk % ti * 64};
    blk -= t;
  }
  return TilePos{-1, blk * 256, 0};
}

// bias q (over all layers): its layer (-1: past the last) and its row
struct BiasPos {
  int layer, row;
};
__device__ __forceinline__ BiasPos bias_at(int q, const LayerDesc* __restrict__ L, int nl) {
  for (int l = 0; l < nl; ++l) {
    if (q < L[l].out) return BiasPos{l, q};
    q -= L[l].out;
  }
  return BiasPos{-1, 0};
}

// The gradient as the EPI_DW launches left it: layer l's S[l] partial sums of its
// weights (out x in each) from p[l] on, then those of its biases (out each).
// Every reader adds them in the order 0, 1, ...
constexpr int kMaxLayers = 17;
struct GradParts {
  const float* p[kMaxLayers];
  int S[kMaxLayers];
};
__device__ __forceinline__ f32x4 grad_w4(const GradParts& P, int l, const LayerDesc& L, int64_t at) {
  const float* q = P.p[l] + at;
  const int64_t MN = (int64_t)L.out * L.in;
  const int S = P.S[l];  // a power of two
  f32x4 v = *reinterpret_cast<const f32x4*>(q);
  if (S < 8) {
    for (int s = 1; s < S; ++s) v += *reinterpret_cast<const f32x4*>(q + s * MN);
    return v;
  }
  for (int s = 0; s < S; s += 8) {  // eight loads in flight
    f32x4 x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = *reinterpret_cast<const f32x4*>(q + (s + e) * MN);
#pragma unroll
    for (int e = 0; e < 8; ++e) v = s + e > 0 ? v + x[e] : x[e];
  }
  return v;
}
__device__ __forceinline__ float grad_b(const GradParts& P, int l, const LayerDesc& L, int row) {
  const float* q = P.p[l] + P.S[l] * (int64_t)L.out * L.in + row;
  float v = q[0];
  for (int s = 1; s < P.S[l]; ++s) v += q[(int64_t)s * L.out];
  return v;
}

// the bf16 copies of a tile: v holds this thread's weights, v[j][e] that of
// (o0 + j * 32 + tid / 8, i0 + (tid & 7) * 8 + e); W and its fragment order
// take 16 bytes per 8 of them, W^T goes through LDS
__device__ __forceinline__ void store_copies(const float (&v)[2][8], const TilePos& T,
                                             const LayerDesc& L, int64_t off,
                                             bf16* __restrict__ Wb, bf16* __restrict__ WbT,
                                             bf16* __restrict__ Wf) {
  __shared__ bf16 tile[64][64 + 8];  // [i][o]
  const int ro = threadIdx.x >> 3, ri = (threadIdx.x & 7) * 8;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int o = T.o0 + j * 32 + ro, i = T.i0 + ri;
    bf16x8 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = (bf16)v[j][e];
      tile[ri + e][j * 32 + ro] = h[e];
    }
    *reinterpret_cast<bf16x8*>(Wb + off + (int64_t)o * L.in + i) = h;
    *reinterpret_cast<bf16x8*>(Wf + off + frag_at(o, i, L.in)) = h;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = j * 32 + ro;
    *reinterpret_cast<bf16x8*>(WbT + off + (int64_t)(T.i0 + i) * L.out + T.o0 + ri) =
        *reinterpret_cast<const bf16x8*>(&tile[i][ri]);
  }
}

// Adam on the flat FP32 parameters; refreshes the bf16 copies W (out x in), W^T
// (in x out) and W in fragment order of every weight.  Bound by memory: 8
// weights a thread in 16- and 32-byte pieces (a weight a thread with scattered
// copies: 12.1 us for 0.9 million weights, 9.2 so).  It adds the gradient's
// partial sums as it reads them, eight loads in flight: 17.5 us for 0.9 million
// weights and 8,192 samples, where a launch per layer for the sums and one for
// the biases took 45 us before it.  The last workgroup sums the loss.
__global__ __launch_bounds__(256) void adam_kernel(
    float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
    GradParts P, float lr, float b1, float b2, float eps, float wd, float c1,
    float c2, const LayerDesc* __restrict__ L, int nl, const int64_t* __restrict__ bf_off,
    bf16* __restrict__ Wb, bf16* __restrict__ WbT, bf16* __restrict__ Wf,
    const float* __restrict__ loss_parts, int n_loss, float* __restrict__ loss,
    float* __restrict__ loss_out) {
  if (blockIdx.x == gridDim.x - 1) loss_total(loss_parts, n_loss, loss, loss_out);
  auto step = [&](float gg, float& mp, float& vp, float ww) {
    const float mm = b1 * mp + (1.0f - b1) * gg;
    const float vv = b2 * vp + (1.0f - b2) * gg * gg;
    mp = mm;
    vp = vv;
    return ww - lr * ((mm / c1) / (sqrtf(vv / c2) + eps) + wd * ww);
  };
  const TilePos T = tile_pos((int)blockIdx.x, L, nl);
  if (T.layer < 0) {
    const BiasPos b = bias_at(T.o0 + (int)threadIdx.x, L, nl);
    if (b.layer < 0) return;
    const int64_t p = L[b.layer].b_off + b.row;
    w[p] = step(grad_b(P, b.layer, L[b.layer], b.row), m[p], v[p], w[p]);
    return;
  }
  const LayerDesc D = L[T.layer];
  float x[2][8];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int o = T.o0 + j * 32 + (threadIdx.x >> 3), i = T.i0 + (threadIdx.x & 7) * 8;
    const int64_t at = (int64_t)o * D.in + i, p = D.w_off + at;
#pragma unroll
    for (int h = 0; h < 8; h += 4) {
      const f32x4 gm = grad_w4(P, T.layer, D, at + h);
      f32x4 mm = *reinterpret_cast<const f32x4*>(m + p + h);
      f32x4 vv = *reinterpret_cast<const f32x4*>(v + p + h);
      f32x4 ww = *reinterpret_cast<const f32x4*>(w + p + h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = mm[e], b = vv[e];
        ww[e] = x[j][h + e] = step(gm[e], a, b, ww[e]);
        mm[e] = a;
        vv[e] = b;
      }
      *reinterpret_cast<f32x4*>(m + p + h) = mm;
      *reinterpret_cast<f32x4*>(v + p + h) = vv;
      *reinterpret_cast<f32x4*>(w + p + h) = ww;
    }
  }
  store_copies(x, T, D, bf_off[T.layer], Wb, WbT, Wf);
}

// the gradient itself, for a caller that asks for it (launch as adam_kernel).  A
// layer with one sum has it in g already (P.p points there): each value is read
// by the thread that writes it
__global__ __launch_bounds__(256) void grad_sum_kernel(GradParts P,
                                                       const LayerDesc* __restrict__ L, int nl,
                                                       float* g,
                                                       const float* __restrict__ loss_parts,
                                                       int n_loss, float* __restrict__ loss) {
  if (blockIdx.x == gridDim.x - 1) loss_total(loss_parts, n_loss, loss, nullptr);
  const TilePos T = tile_pos((int)blockIdx.x, L, nl);
  if (T.layer < 0) {
    const BiasPos b = bias_at(T.o0 + (int)threadIdx.x, L, nl);
    if (b.layer >= 0) g[L[b.layer].b_off + b.row] = grad_b(P, b.layer, L[b.layer], b.row);
    return;
  }
  const LayerDesc D = L[T.layer];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = T.o0 + j * 16 + (threadIdx.x >> 4), i = T.i0 + (threadIdx.x & 15) * 4;
    const int64_t at = (int64_t)o * D.in + i;
    *reinterpret_cast<f32x4*>(g + D.w_off + at) = grad_w4(P, T.layer, D, at);
  }
}

// the bf16 copies of every weight (launch: the weight tiles)
__global__ __launch_bounds__(256) void refresh_bf16_kernel(
    const float* __restrict__ w, const LayerDesc* __restrict__ L, int nl,
    const int64_t* __restrict__ bf_off, bf16* __restrict__ Wb, bf16* __restrict__ WbT,
    bf16* __restrict__ Wf) {
  const TilePos T = tile_pos((int)blockIdx.x, L, nl);
  if (T.layer < 0) return;
  const LayerDesc D = L[T.layer];
  float x[2][8];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[j][e] = w[D.w_off + (int64_t)(T.o0 + j * 32 + (threadIdx.x >> 3)) * D.in + T.i0 +
                  (threadIdx.x & 7) * 8 + e];
  store_copies(x, T, D, bf_off[T.layer], Wb, WbT, Wf);
}

// copy the (mu, logvar) block of O (Bpad x out_pad) into y (B x 2 ns)
__global__ void gather_out_kernel(const float* __restrict__ O, int Bn, int ns, int out_pad,
                                  float* __restrict__ y) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (int64_t)Bn * 2 * ns) return;
  const int b = (int)(q / (2 * ns)), k = (int)(q % (2 * ns));
  y[q] = O[(size_t)b * out_pad + k];
}

// The whole network on 16 RT rows per workgroup of eight waves, for inference:
// the activations stay in LDS from the features to the outputs and the weights
// come from the L2 once per workgroup, so a call is one launch and writes
// nothing but its outputs (layer by layer it wrote, per row and unit, the
// training step's pre-activation and two copies of the activation).  Wave w
// makes features [w, w + 1) * width / 8 of a layer: W fragments are the MFMA's
// rows and activations its columns, so a lane ends up with four consecutive
// features of one row, one 8-byte LDS store.  A layer's outputs are all in
// registers before the first replaces an input.  Every output sums its K in the
// order of gemm_nt_kernel, 32 at a time: the same bits.
// Bound by the L2 reads of the weights (1.7 MB a workgroup at width 512) and
// the activations' exponentials and reciprocals.  40,000 rows, 23 -> 4 x 512 ->
// 180: 395 -> 128 us, 77 rows 57 -> 38 us.
constexpr int kInferPad = 8;  // bf16 of padding per LDS row
template <int RT, int FT>
__global__ __launch_bounds__(512) void infer_kernel(const float* __restrict__ x, int64_t n, int n_in,
                                                    const LayerDesc* __restrict__ layers, int depth,
                                                    const int64_t* __restrict__ bf_off,
                                                    const bf16* __restrict__ Wf,
                                                    const float* __restrict__ w, int n_out,
                                                    int vec4, float* __restrict__ y) {
  extern __shared__ bf16 act[];
  constexpr int W = 128 * FT, D = 2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * (16 * RT);
  const int in_pad = layers[0].in;
  const int S = (in_pad > W ? in_pad : W) + kInferPad;
  for (int q = threadIdx.x; q < 16 * RT * in_pad; q += 512) {
    const int r = q / in_pad, k = q - r * in_pad;
    act[r * S + k] = (bf16)(r0 + r < n && k < n_in ? x[(r0 + r) * n_in + k] : 0.0f);
  }
  __syncthreads();
  const int li = lane & 15, kq = (lane >> 4) * 8;
  // acc[t][r]: features f0 + 16 t .. of a layer with K inputs, rows 16 r ..
  auto product = [&](const bf16* Wl, int K, int f0, auto& acc) {
    constexpr int T = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[t][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16* wp = Wl + (size_t)(f0 / 16) * K * 16 + lane * 8;  // tile t, step k: + (t K + k) * 16
    // weights D steps of 32 ahead: an L2 read takes longer than a step's MFMAs
    bf16x8 a[D][T];
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int t = 0; t < T; ++t)
        if (32 * d < K)
          a[d][t] = *reinterpret_cast<const bf16x8*>(wp + (size_t)(t * K + 32 * d) * 16);
    for (int k0 = 0; k0 < K; k0 += 32 * D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int k = k0 + 32 * d;
        if (k >= K) break;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const bf16x8 b = *reinterpret_cast<const bf16x8*>(act + (16 * r + li) * S + k + kq);
#pragma unroll
          for (int t = 0; t < T; ++t)
            acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][t], b, acc[t][r], 0, 0, 0);
        }
        const int kn = k + 32 * D;
        if (kn < K)
#pragma unroll
          for (int t = 0; t < T; ++t)
            a[d][t] = *reinterpret_cast<const bf16x8*>(wp + (size_t)(t * K + kn) * 16);
      }
    }
  };
  for (int l = 0; l < depth; ++l) {
    const LayerDesc L = layers[l];
    const int f0 = wave * (16 * FT);
    f32x4 acc[FT][RT];
    product(Wf + bf_off[l], L.in, f0, acc);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < FT; ++t) {
      const int f = f0 + 16 * t + (lane >> 4) * 4;
      float bias[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[q] = w[L.b_off + f + q];
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        bf16x4 h;
        float z[4], s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) z[q] = acc[t][r][q] + bias[q];
        sigm4(z, s);
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] = (bf16)(z[q] * s[q]);
        *reinterpret_cast<bf16x4*>(act + (16 * r + li) * S + f) = h;
      }
    }
    __syncthreads();
  }
  // the output layer, 32 features per wave at a time (its padding ends on one),
  // every gridDim.y-th 256 of them
  const LayerDesc L = layers[depth];
  for (int f0 = (int)blockIdx.y * 256 + wave * 32; f0 < n_out; f0 += 256 * (int)gridDim.y) {
    f32x4 acc[2][RT];
    product(Wf + bf_off[depth], L.in, f0, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int f = f0 + 16 * t + (lane >> 4) * 4;
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const int64_t row = r0 + 16 * r + li;
        if (row >= n) continue;
        if (vec4 && f < n_out) {
          float4 v;
          v.x = acc[t][r][0] + w[L.b_off + f];
          v.y = acc[t][r][1] + w[L.b_off + f + 1];
          v.z = acc[t][r][2] + w[L.b_off + f + 2];
          v.w = acc[t][r][3] + w[L.b_off + f + 3];
          *reinterpret_cast<float4*>(y + row * n_out + f) = v;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (f + q < n_out) y[row * n_out + f + q] = acc[t][r][q] + w[L.b_off + f + q];
        }
      }
    }
  }
}

int g1(int64_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

// ---------------------------------------------------------------- surrogate I/O
// Canonical features of a particle: one-hot(model) and its rates per bin,
// [kon(nb), koff, alpha(nb), gamma(nb), lambda, splice] in log10 / 3, with
// constant rates repeated over the bins (layout of scripts/model.jl:30-43).
__global__ void features_kernel(int model, int64_t n, const double* __restrict__ theta, int nb,
                                float* __restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int nk = model == 3 ? nb : 1, na = model == 4 ? nb : 1, ng = model == 5 ? nb : 1;
  const int ok = 0, ooff = nk, oa = nk + 1, og = oa + na, ol = og + ng, os = ol + 1;
  const int nin = 5 + 3 * nb + 3;
  float* r = x + i * nin;
  for (int q = 0; q < 5; ++q) r[q] = (q == model - 1) ? 1.0f : 0.0f;
  int c = 5;
  for (int j = 0; j < nb; ++j) r[c++] = (float)(theta[i + n * (ok + (nk > 1 ? j : 0))] / 3.0);
  r[c++] = (float)(theta[i + n * ooff] / 3.0);
  for (int j = 0; j < nb; ++j) r[c++] = (float)(theta[i + n * (oa + (na > 1 ? j : 0))] / 3.0);
  for (int j = 0; j < nb; ++j) r[c++] = (float)(theta[i + n * (og + (ng > 1 ? j : 0))] / 3.0);
  r[c++] = (float)(theta[i + n * ol] / 3.0);
  r[c++] = (float)(theta[i + n * os] / 3.0);
}

// Targets: standardised asinh of every statistic (stats n x K column-major).
__global__ void targets_kernel(int64_t n, const double* __restrict__ stats, int K,
                               const float* __restrict__ mean, const float* __restrict__ sd,
                               float* __restrict__ t) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n * K) return;
  const int64_t i = q / K;
  const int k = (int)(q % K);
  const double s = stats[i + n * k];
  float v = 0.0f;
  if (s == s && fabs(s) < 1e300) v = (float)((asinh(s) - (double)mean[k]) / (double)sd[k]);
  t[q] = v;
}

// Screen: the surrogate gives, per statistic, y ~ N(mu, sigma^2) in the
// standardised asinh space, s = sinh(mean_k + sd_k y).  Its central moments
// (E s, c2, c3, c4) come from 7-point Gauss-Hermite quadrature.  The
// statistics of different (bin, condition) groups come from disjoint cells,
// so the error err_g = sum_k W_gk (d_gk - s_k)^2 concentrates around
//   E err = sum W (delta^2 + c2),  Var err = sum W^2 (4 delta^2 c2 - 4 delta c3 + c4 - c2^2)
// with delta = d - E s.  A particle passes when E err - z sd err can reach a
// gene's threshold (or when its prediction is not finite).  Genes whose data
// are not finite have NaN errors and accept nobody.
//
// A workgroup holds the moments of PT particles in LDS; a lane scores genes g
// and g + 256 against all of them.  A (particle, statistic, gene) term is 13
// FP32 instructions, and one 16-byte and a quarter of a 16-byte LDS read serve
// two: the reference expression
//   4 delta delta c2 - 4 delta c3 + c4 - c2 c2  (16, four 4-byte LDS reads)
// with the powers of two moved to c4 / 4, c2 c2 / 4 and 4 W^2, which changes no
// bit while nothing overflows and no product is subnormal: moments and data
// inside screen_safe's and SCREEN_BIG's ranges.  A workgroup that holds a
// moment outside them, and a gene with such a datum, are scored with the
// expression as it stands.  VALU issue bounds it: 40,000 particles, 2,000 genes,
// 90 statistics in 2.0 ms with the moments and the normal integrals (2.5 ms
// with 16 particles of one gene a lane and the expression as it stands; 7.2e9
// terms of 13 instructions take 1.8 ms at the 3 cycles each that FP32
// reaches).  500 particles: 0.28 ms for 1.04, as 8 particles a workgroup fill
// more of the chip.  Four waves per SIMD: with five or six the sums spill (2.3
// and 2.5 ms).
#define SCREEN_BIG 0x1p30f
ABC_DEV bool screen_safe(float e, float v2, float v3, float v4) {
  // |delta| is 0 or at least 2^-44 then, and every product at least 2^-126
  const float ae = fabsf(e), a3 = fabsf(v3);
  return ae >= 0x1p-20f && ae <= SCREEN_BIG && v2 >= 0x1p-38f && v2 <= SCREEN_BIG &&
         a3 >= 0x1p-80f && a3 <= 0x1p45f && v4 >= 0x1p-100f && v4 <= 0x1p60f;
}

template <bool SCORE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void screen_kernel(const float* __restrict__ y, int64_t n, int K,
                                                     const float* __restrict__ mean,
                                                     const float* __restrict__ sd, float z,
                                                     const float* __restrict__ Wf,
                                                     const double* __restrict__ data, int64_t G,
                                                     const double* __restrict__ thr, float margin,
                                                     double clamp, uint8_t* __restrict__ pass,
                                                     float* __restrict__ score) {
  constexpr int PT = ABC_SCREEN_PT;
  __shared__ float4 mo[ABC_MAX_STATS / 2][PT];  // E s, c2, c3, c4 (plain: c4 / 4)
  __shared__ __attribute__((aligned(16))) float qv[ABC_MAX_STATS / 2][PT];  // c2 c2 / 4
  __shared__ int hit[PT], bad[PT], general;
  __shared__ float s_sum[4][PT], s_max[4][PT];  // per wave: expected pairs, largest margin
  const double gx[7] = {-3.7504397177257425, -2.366759410734541, -1.1544053947399682, 0.0,
                        1.1544053947399682, 2.366759410734541, 3.7504397177257425};
  const double gw[7] = {0.000548268855972217, 0.03075712396758652, 0.2401231786050127,
                        0.45714285714285724, 0.2401231786050127, 0.03075712396758652,
                        0.000548268855972217};
  const int64_t i0 = (int64_t)blockIdx.x * PT;
  if (threadIdx.x < PT) {
    hit[threadIdx.x] = (i0 + threadIdx.x < n) ? 0 : 1;
    bad[threadIdx.x] = 0;
  }
  if (threadIdx.x == 0) general = 0;
  __syncthreads();
  for (int q = threadIdx.x; q < PT * K; q += blockDim.x) {
    const int p = q / K, k = q % K;
    const int64_t i = i0 + p;
    double m1 = 1.0, v2 = 1.0, v3 = 1.0, v4 = 1.0;  // past n: anything in range
    if (i < n) {
      m1 = v2 = v3 = v4 = 0.0;
      const double mu = y[i * 2 * K + k];
      const double lv = fmin(fmax((double)y[i * 2 * K + K + k], -12.0), 12.0);
      const double s = exp(0.5 * lv);
      double sv[7];
      for (int r = 0; r < 7; ++r) {
        sv[r] = sinh((double)mean[k] + (double)sd[k] * (mu + s * gx[r]));
        m1 += gw[r] * sv[r];
      }
      for (int r = 0; r < 7; ++r) {
        const double e = sv[r] - m1, e2 = e * e;
        v2 += gw[r] * e2;
        v3 += gw[r] * e2 * e;
        v4 += gw[r] * e2 * e2;
      }
      if (!(fabs(m1) < 1e30) || !(v4 < 1e300)) hit[p] = bad[p] = 1;
    }
    const float4 m = {(float)m1, (float)v2, (float)v3, (float)v4};
    mo[k][p] = m;
    qv[k][p] = m.y * m.y * 0.25f;
    if (!screen_safe(m.x, m.y, m.z, m.w)) general = 1;  // benign race: every writer stores 1
  }
  __syncthreads();
  const bool plain = general == 0;  // the whole workgroup
  if (plain) {
    for (int q = threadIdx.x; q < PT * K; q += blockDim.x) mo[q / PT][q % PT].w *= 0.25f;
    __syncthreads();
  }
  // per particle over this thread's genes: sum of P(err <= t) under the
  // Gaussian approximation, and the largest standardised margin (t - E) / sd
  float psum[PT], pmax[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) { psum[p] = 0.f; pmax[p] = -HUGE_VALF; }
  auto finish = [&](float t, const float (&em)[PT], const float (&ev)[PT]) {
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const float sdv = sqrtf(ev[p]);
      if (em[p] - z * sdv <= t) hit[p] = 1;  // benign race: every writer stores 1
      if (SCORE) {
        const float d = t - em[p];
        const float u = sdv > 0.f ? d / sdv : (d >= 0.f ? HUGE_VALF : -HUGE_VALF);
        psum[p] += normcdff(u);
        pmax[p] = fmaxf(pmax[p], u);
      }
    }
  };
  // gene g by the expression as it stands
  auto gene = [&](int64_t g, float t) {
    const float back = plain ? 4.f : 1.f;  // c4 from mo
    float em[PT], ev[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) { em[p] = 0.f; ev[p] = 0.f; }
    for (int k = 0; k < K; ++k) {
      const float d = (float)data[g + G * k];
      const float w = Wf[g + G * k];
      const float w2 = w * w;
#pragma unroll
      for (int p = 0; p < PT; ++p) {
        const float4 m = mo[k][p];
        const float dl = d - m.x;
        em[p] += w * (dl * dl + m.y);
        ev[p] += w2 * fmaxf(4.f * dl * dl * m.y - 4.f * dl * m.z + back * m.w - m.y * m.y, 0.f);
      }
    }
    finish(t, em, ev);
  };
  for (int64_t g = threadIdx.x; g < G; g += 512) {
    float t[2];
    bool run[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t gh = g + 256 * h;
      const double tg = gh < G ? thr[gh] : 0.0;
      // a clamped threshold is every clamped error's: nobody may be skipped
      run[h] = gh < G && !(tg >= clamp);
      t[h] = (float)(tg * (1.0 + (double)margin));
    }
    float em0[PT], ev0[PT], em1[PT], ev1[PT], big = 0.f, big1 = 0.f;
    const bool both = plain && (run[0] || run[1]);
    if (both) {
      const int64_t ga = run[0] ? g : g + 256, gb = run[1] ? g + 256 : g;
#pragma unroll
      for (int p = 0; p < PT; ++p) em0[p] = ev0[p] = em1[p] = ev1[p] = 0.f;
      for (int k = 0; k < K; ++k) {
        const float d0 = (float)data[ga + G * k], d1 = (float)data[gb + G * k];
        const float w0 = Wf[ga + G * k], w1 = Wf[gb + G * k];
        big = fmaxf(fmaxf(big, fabsf(d0)), w0);
        big1 = fmaxf(fmaxf(big1, fabsf(d1)), w1);
        const float x0 = 4.f * (w0 * w0), x1 = 4.f * (w1 * w1);
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          const float4 m = mo[k][p];
          const float q = qv[k][p];
          const float a = d0 - m.x, b = d1 - m.x;
          const float aa = a * a, bb = b * b;
          em0[p] += w0 * (aa + m.y);
          em1[p] += w1 * (bb + m.y);
          ev0[p] += x0 * fmaxf(aa * m.y - a * m.z + m.w - q, 0.f);
          ev1[p] += x1 * fmaxf(bb * m.y - b * m.z + m.w - q, 0.f);
        }
      }
    }
#pragma unroll 1
    for (int h = 0; h < 2 && g + 256 * h < G; ++h) {  // one copy of the code
      if (!run[0]) {
        for (int p = 0; p < PT; ++p) {
          hit[p] = 1;
          psum[p] += 1.f;
          pmax[p] = HUGE_VALF;
        }
      } else if (both && big <= SCREEN_BIG) {
        finish(t[0], em0, ev0);
      } else {
        gene(g + 256 * h, t[0]);
      }
#pragma unroll
      for (int p = 0; p < PT; ++p) { em0[p] = em1[p]; ev0[p] = ev1[p]; }
      run[0] = run[1];
      t[0] = t[1];
      big = big1;
    }
  }
  if (SCORE) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      float a = psum[p], b = pmax[p];
      for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b = fmaxf(b, __shfl_xor(b, o));
      }
      if (lane == 0) { s_sum[wave][p] = a; s_max[wave][p] = b; }
    }
  }
  __syncthreads();
  if (threadIdx.x < PT && i0 + threadIdx.x < n) {
    const int p = threadIdx.x;
    pass[i0 + p] = (uint8_t)hit[p];
    if (SCORE) {
      // a prediction that is not finite passes whatever the threshold
      float a = 0.f, b = -HUGE_VALF;
      for (int w = 0; w < 4; ++w) { a += s_sum[w][p]; b = fmaxf(b, s_max[w][p]); }
      score[2 * (i0 + p)] = bad[p] ? HUGE_VALF : a;
      score[2 * (i0 + p) + 1] = bad[p] ? HUGE_VALF : b;
    }
  }
}
template __global__ void screen_kernel<false>(const float*, int64_t, int, const float*,
                                              const float*, float, const float*, const double*,
                                              int64_t, const double*, float, double, uint8_t*,
                                              float*);
template __global__ void screen_kernel<true>(const float*, int64_t, int, const float*,
                                             const float*, float, const float*, const double*,
                                             int64_t, const double*, float, double, uint8_t*,
                                             float*);

struct abc_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  bool own_stream = true;
  int n_in = 0, in_pad = 0, width = 0, depth = 0, n_out = 0, out_pad = 0, ns = 0, max_batch = 0;
  int n_cnt = 0;  // leading count statistics (Poisson loss on a log-rate output)
  int tile_rows = 0;  // GEMM workgroup rows: 0 = by shape, else 64 or 128
  int tile_cols = 0;  // GEMM workgroup columns: 0 = by shape, else 64 or 128
  int64_t n_par = 0, n_bf = 0;
  int w_tiles = 0, n_bias = 0;  // 64 x 64 weight tiles and biases over all layers
  std::vector<LayerDesc> layers;
  std::vector<int64_t> bf_off;
  LayerDesc* d_layers = nullptr;
  int64_t* d_bf_off = nullptr;
  float *w = nullptr, *m = nullptr, *v = nullptr, *g = nullptr;
  bf16 *Wb = nullptr, *WbT = nullptr, *Wf = nullptr;  // Wf: fragment order
  // activations (max_batch rows, padded to 128)
  bf16 *X = nullptr, *XT = nullptr;
  std::vector<float*> Z;
  std::vector<bf16*> H, HT;
  float* O = nullptr;
  bf16 *dA = nullptr, *dAT = nullptr, *dB = nullptr, *dBT = nullptr;
  float *loss = nullptr, *loss_parts = nullptr;  // loss_parts: one per tile of nll_kernel
  float* parts = nullptr;      // partial sums of the gradient (GradParts)
  std::vector<int64_t> part_off;  // per layer
  int64_t step = 0;
  std::string msg;
};

namespace {

int mfail(abc_mlp* p, int code, const std::string& s) {
  if (p) p->msg = s;
  return code;
}

#define MCHK(p, expr)                                                                        \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess) return mfail(p, ABC_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Sums that a weight gradient (M, N = layer widths, K = batch) is split into to
// fill the machine: chunks of whole stages, the last shorter or, past the end,
// empty (a sum of zeros).  With equal chunks only, a batch of 8,064 was split in
// two and a step took 349 us, 209 so; 1,000 samples 139 and 109.
int splitk_for(int M, int N, int K) {
  // counted in 64-row tiles, so the split does not depend on the tile rows
  // chosen below (results do not depend on them either)
  const int tiles = (M / 64) * (N / (N % 128 == 0 ? 128 : 64));
  int S = 1;
  while (tiles * S < 256 && K / (2 * S) >= 256) S *= 2;
  return S;
}
int splitk_chunk(int K, int S) {
  return (K / kDwChunk + S - 1) / S * kDwChunk;  // K, the padded batch, is a multiple of it
}

// Workgroup tile rows: 64 when 128-row tiles would leave fewer than two
// workgroups per CU (one wave per SIMD cannot hide the load and LDS latency).
int tile_rows(int M, int N, int S) {
  const int tiles = (M / 128) * (N / (N % 128 == 0 ? 128 : 64)) * S;
  return (tiles < 512 && M % 64 == 0) ? 64 : 128;
}

// Workgroup tile columns (N % 128 == 0): 64 when 128-column tiles would leave
// fewer than four workgroups per CU.
int tile_cols(int M, int N, int S, int bm) {
  return (M / bm) * (N / 128) * S < 1024 ? 64 : 128;
}

struct Tile {
  int bm, bn;
};
Tile tile_for(const abc_mlp* p, int M, int N, int S) {
  const int bm = p->tile_rows ? p->tile_rows : tile_rows(M, N, S);
  const int bn = N % 128 != 0 ? 64 : (p->tile_cols ? p->tile_cols : tile_cols(M, N, S, bm));
  return Tile{bm, bn};
}

// the product of g (whose K is that of one of its S sums)
template <int EPI>
void gemm(abc_mlp* p, const GemmArgs& g, int S = 1) {
  const Tile t = tile_for(p, g.M, g.N, S);
  const dim3 grid = EPI == EPI_DW ? dim3(S, g.M / t.bm, g.N / t.bn) : dim3(g.M / t.bm, g.N / t.bn);
  if (t.bn == 128 && t.bm == 128)
    hipLaunchKernelGGL((gemm_nt_kernel<128, 128, EPI>), grid, dim3(256), 0, p->stream, g.A, g.B, g.M,
                       g.N, g.K, g.ld, g.bias, g.Cf, g.Cb, g.CbT, g.Zprev, g.Zout);
  else if (t.bn == 128)
    hipLaunchKernelGGL((gemm_nt_kernel<64, 128, EPI>), grid, dim3(256), 0, p->stream, g.A, g.B, g.M,
                       g.N, g.K, g.ld, g.bias, g.Cf, g.Cb, g.CbT, g.Zprev, g.Zout);
  else if (t.bm == 128)
    hipLaunchKernelGGL((gemm_nt_kernel<128, 64, EPI>), grid, dim3(256), 0, p->stream, g.A, g.B, g.M,
                       g.N, g.K, g.ld, g.bias, g.Cf, g.Cb, g.CbT, g.Zprev, g.Zout);
  else
    hipLaunchKernelGGL((gemm_nt_kernel<64, 64, EPI>), grid, dim3(256), 0, p->stream, g.A, g.B, g.M,
                       g.N, g.K, g.ld, g.bias, g.Cf, g.Cb, g.CbT, g.Zprev, g.Zout);
}

int forward(abc_mlp* p, int64_t Bn, const float* x_dev) {
  const int Bpad = (int)((Bn + 127) / 128 * 128);
  hipLaunchKernelGGL(cast_input_kernel, dim3(Bpad / 64, p->in_pad / 64), dim3(256), 0, p->stream,
                     x_dev, (int)Bn, Bpad, p->n_in, p->in_pad, p->X, p->XT);
  const bf16* in = p->X;
  for (int l = 0; l < p->depth; ++l) {
    const LayerDesc& L = p->layers[l];
    gemm<EPI_SILU>(p, GemmArgs{in, p->Wb + p->bf_off[l], Bpad, L.out, L.in, L.in, p->w + L.b_off,
                               nullptr, p->H[l], p->HT[l], nullptr, p->Z[l]});
    in = p->H[l];
  }
  const LayerDesc& L = p->layers[p->depth];
  gemm<EPI_F32>(p, GemmArgs{in, p->Wb + p->bf_off[p->depth], Bpad, L.out, L.in, L.in,
                            p->w + L.b_off, p->O, nullptr, nullptr, nullptr, nullptr});
  MCHK(p, hipGetLastError());
  return ABC_OK;
}

// One launch for all n rows where a layer's outputs fit a workgroup's registers
// and LDS (width up to 512); false: not launched.  Rows per workgroup: 16 while
// those give at most one workgroup per CU, 32 up to two, 64 above, two of which
// share a CU and overlap one's MFMAs with the other's activations (with 128, one
// a CU, they do not).  Outputs beyond 256 are shared by as many workgroups per
// row tile as leave at most one per CU, each with the hidden layers of its own:
// 100 rows, 512 units, one layer, 2,048 outputs 44 us by one, 23 so (32 layer by
// layer).  16 / 32 / 64 / 128 rows, us: n = 77 39 / 43 / 60 / 86, 8,192
// 60 / 51 / 65 / 96, 16,384 97 / 70 / 69 / 101, 40,000 212 / 143 / 131 / 186.
template <int RT, int FT>
bool infer_launch(abc_mlp* p, int64_t n, const float* x, float* y) {
  const size_t lds = (size_t)16 * RT * ((size_t)std::max(p->in_pad, 128 * FT) + kInferPad) * 2;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(infer_kernel<RT, FT>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  const int64_t tiles = (n + 16 * RT - 1) / (16 * RT);
  const int64_t parts = std::max<int64_t>(1, std::min<int64_t>((p->n_out + 255) / 256, 256 / tiles));
  hipLaunchKernelGGL((infer_kernel<RT, FT>), dim3((unsigned)tiles, (unsigned)parts), dim3(512),
                     lds, p->stream, x, n, p->n_in, p->d_layers, p->depth, p->d_bf_off, p->Wf, p->w,
                     p->n_out,
                     (int)(p->n_out % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0), y);
  return true;
}

template <int FT>
bool infer_width(abc_mlp* p, int64_t n, const float* x, float* y) {
  if (n <= 4096) return infer_launch<1, FT>(p, n, x, y);
  if (n <= 16384) return infer_launch<2, FT>(p, n, x, y);
  return infer_launch<4, FT>(p, n, x, y);
}

bool infer(abc_mlp* p, int64_t n, const float* x, float* y) {
  if (n > (int64_t)1 << 30) return false;
  switch (p->width) {
    case 128: return infer_width<1>(p, n, x, y);
    case 256: return infer_width<2>(p, n, x, y);
    case 384: return infer_width<3>(p, n, x, y);
    case 512: return infer_width<4>(p, n, x, y);
    default: return false;
  }
}

// nll_kernel's workgroups for a batch of Bn
int loss_tiles(const abc_mlp* p, int64_t Bn) {
  return (int)((Bn + 127) / 128 * 128 / 64) * (p->out_pad / 64);
}

// fwd + loss + bwd into p->parts, described by P; shares of the loss (mean NLL)
// in p->loss_parts
int grad(abc_mlp* p, int64_t Bn, const float* x_dev, const float* t_dev, GradParts& P) {
  int rc = forward(p, Bn, x_dev);
  if (rc) return rc;
  const int Bpad = (int)((Bn + 127) / 128 * 128);
  hipLaunchKernelGGL(nll_kernel, dim3(Bpad / 64, p->out_pad / 64), dim3(256), 0, p->stream,
                     p->O, t_dev, (int)Bn, Bpad, p->ns, p->n_cnt, p->out_pad, p->dA, p->dAT,
                     p->loss_parts);
  // dA / dAT hold dZ of the current layer (output layer first)
  bf16 *cur = p->dA, *curT = p->dAT, *nxt = p->dB, *nxtT = p->dBT;
  for (int l = p->depth; l >= 0; --l) {
    const LayerDesc& L = p->layers[l];
    const bf16* Hin_T = l == 0 ? p->XT : p->HT[l - 1];
    // dW_l = dZ_l^T H_{l-1}: (out x Bpad) . (in x Bpad)^T, and db_l
    const int64_t MN = (int64_t)L.out * L.in;
    int S = splitk_for(L.out, L.in, Bpad);
    // one sum is the gradient itself, which lies in the same order
    float* part = S > 1 ? p->parts + p->part_off[l] : p->g + L.w_off;
    P.S[l] = S;
    P.p[l] = part;
    const GemmArgs w{curT, Hin_T, L.out, L.in, splitk_chunk(Bpad, S), Bpad,
                     nullptr, part, nullptr, nullptr,
                     nullptr, part + S * MN};
    gemm<EPI_DW>(p, w, S);
    if (l > 0) {
      // dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1}); W_l^T copy is (in x out)
      gemm<EPI_DSILU>(p, GemmArgs{cur, p->WbT + p->bf_off[l], Bpad, L.in, L.out, L.out, nullptr,
                                  nullptr, nxt, nxtT, p->Z[l - 1], nullptr});
      std::swap(cur, nxt);
      std::swap(curT, nxtT);
    }
  }
  MCHK(p, hipGetLastError());
  return ABC_OK;
}

}  // namespace

extern "C" {

int32_t abc_mlp_create(abc_mlp** out, int32_t device, int32_t n_in, int32_t width, int32_t depth,
                       int32_t n_stats, int32_t max_batch, uint64_t seed) {
  if (!out || n_in < 1 || n_in > 256 || width < 64 || width % 128 || depth < 1 || depth > 16 ||
      n_stats < 1 || n_stats > 1024 || max_batch < 1)
    return ABC_E_ARG;
  *out = nullptr;
  abc_mlp* p = new abc_mlp();
  p->device = device;
  if (hipSetDevice(device) != hipSuccess) { delete p; return ABC_E_HIP; }
  p->n_in = n_in;
  p->in_pad = (n_in + 63) / 64 * 64;
  p->width = width;
  p->depth = depth;
  p->ns = n_stats;
  p->n_out = 2 * n_stats;
  p->out_pad = (p->n_out + 127) / 128 * 128;  // rows of dW_out are tiled by 128
  p->max_batch = (max_batch + 127) / 128 * 128;
  int64_t off = 0, boff = 0;
  for (int l = 0; l <= depth; ++l) {
    LayerDesc L;
    L.in = l == 0 ? p->in_pad : width;
    L.out = l == depth ? p->out_pad : width;
    L.w_off = off;
    off += (int64_t)L.in * L.out;
    L.b_off = off;
    off += L.out;
    p->layers.push_back(L);
    p->bf_off.push_back(boff);
    boff += (int64_t)L.in * L.out;
  }
  p->n_par = off;
  p->n_bf = boff;
  // He-uniform initial weights on the real (unpadded) block, zeros elsewhere
  std::vector<float> w0(off, 0.0f);
  std::mt19937_64 rng(seed);
  for (int l = 0; l <= depth; ++l) {
    const LayerDesc& L = p->layers[l];
    const int rin = l == 0 ? n_in : width, rout = l == depth ? p->n_out : width;
    const float a = std::sqrt(3.0f / (float)rin);
    std::uniform_real_distribution<float> U(-a, a);
    for (int o = 0; o < rout; ++o)
      for (int i = 0; i < rin; ++i) w0[L.w_off + (int64_t)o * L.in + i] = U(rng);
  }
  const int64_t Bp = p->max_batch;
  bool ok = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking) == hipSuccess;
  auto A = [&](auto** ptr, size_t bytes) {
    if (ok && hipMalloc((void**)ptr, bytes) != hipSuccess) ok = false;
  };
  A(&p->w, 4 * off); A(&p->m, 4 * off); A(&p->v, 4 * off); A(&p->g, 4 * off);
  A(&p->Wb, 2 * boff); A(&p->WbT, 2 * boff); A(&p->Wf, 2 * boff);
  A(&p->d_layers, sizeof(LayerDesc) * p->layers.size());
  A(&p->d_bf_off, sizeof(int64_t) * p->bf_off.size());
  A(&p->X, 2 * Bp * p->in_pad); A(&p->XT, 2 * Bp * p->in_pad);
  p->Z.assign(depth, nullptr); p->H.assign(depth, nullptr); p->HT.assign(depth, nullptr);
  for (int l = 0; l < depth; ++l) {
    A(&p->Z[l], 4 * Bp * width); A(&p->H[l], 2 * Bp * width); A(&p->HT[l], 2 * Bp * width);
  }
  const int64_t dmax = std::max<int64_t>(width, p->out_pad);
  A(&p->O, 4 * Bp * p->out_pad);
  A(&p->dA, 2 * Bp * dmax); A(&p->dAT, 2 * Bp * dmax);
  A(&p->dB, 2 * Bp * dmax); A(&p->dBT, 2 * Bp * dmax);
  A(&p->loss, 64); A(&p->loss_parts, 4 * (Bp / 64) * (p->out_pad / 64));
  // partial sums of the gradients: as many as any batch up to max_batch splits into
  int64_t n_part = 0;
  for (const LayerDesc& L : p->layers) {
    int S = 1;
    for (int64_t K = 128; K <= Bp; K += 128) S = std::max(S, splitk_for(L.out, L.in, (int)K));
    p->part_off.push_back(n_part);
    if (S > 1) n_part += (int64_t)S * (L.out * (int64_t)L.in + L.out);
  }
  A(&p->parts, 4 * std::max<int64_t>(n_part, 4));
  if (!ok) { abc_mlp_destroy(p); return ABC_E_OOM; }
  std::vector<float> zeros(off, 0.0f);
  if (hipMemcpy(p->w, w0.data(), 4 * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->m, zeros.data(), 4 * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->v, zeros.data(), 4 * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->d_layers, p->layers.data(), sizeof(LayerDesc) * p->layers.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->d_bf_off, p->bf_off.data(), sizeof(int64_t) * p->bf_off.size(), hipMemcpyHostToDevice) != hipSuccess) {
    abc_mlp_destroy(p);
    return ABC_E_HIP;
  }
  for (const LayerDesc& L : p->layers) {
    p->w_tiles += (L.in / 64) * (L.out / 64);
    p->n_bias += L.out;
  }
  hipLaunchKernelGGL(refresh_bf16_kernel, dim3(p->w_tiles), dim3(256), 0, p->stream, p->w,
                     p->d_layers, (int)p->layers.size(), p->d_bf_off, p->Wb, p->WbT, p->Wf);
  if (hipStreamSynchronize(p->stream) != hipSuccess) { abc_mlp_destroy(p); return ABC_E_HIP; }
  *out = p;
  return ABC_OK;
}

int32_t abc_mlp_destroy(abc_mlp* p) {
  if (!p) return ABC_OK;
  if (p->stream) hipStreamSynchronize(p->stream);
  void* bufs[] = {p->w, p->m, p->v, p->g, p->Wb, p->WbT, p->Wf, p->d_layers, p->d_bf_off, p->X, p->XT,
                  p->O, p->dA, p->dAT, p->dB, p->dBT, p->loss, p->loss_parts, p->parts};
  for (void* b : bufs)
    if (b) hipFree(b);
  for (auto* z : p->Z) if (z) hipFree(z);
  for (auto* h : p->H) if (h) hipFree(h);
  for (auto* h : p->HT) if (h) hipFree(h);
  if (p->stream && p->own_stream) hipStreamDestroy(p->stream);
  delete p;
  return ABC_OK;
}

const char* abc_mlp_last_error(const abc_mlp* p) { return p ? p->msg.c_str() : "null model"; }

int64_t abc_mlp_n_params(const abc_mlp* p) { return p ? p->n_par : ABC_E_ARG; }

int32_t abc_mlp_set_tile_rows(abc_mlp* p, int32_t rows) {
  if (!p || (rows != 0 && rows != 64 && rows != 128)) return ABC_E_ARG;
  p->tile_rows = rows;
  return ABC_OK;
}

int32_t abc_mlp_set_tile_cols(abc_mlp* p, int32_t cols) {
  if (!p || (cols != 0 && cols != 64 && cols != 128)) return ABC_E_ARG;
  p->tile_cols = cols;
  return ABC_OK;
}

int32_t abc_mlp_set_count_outputs(abc_mlp* p, int32_t n_counts) {
  if (!p || n_counts < 0 || n_counts > p->ns) return ABC_E_ARG;
  p->n_cnt = n_counts;
  return ABC_OK;
}

int32_t abc_mlp_set_stream(abc_mlp* p, void* s) {
  if (!p) return ABC_E_ARG;
  hipStreamSynchronize(p->stream);
  if (p->own_stream) hipStreamDestroy(p->stream);
  if (s) {
    p->stream = (hipStream_t)s;
    p->own_stream = false;
  } else {
    if (hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking) != hipSuccess) return ABC_E_HIP;
    p->own_stream = true;
  }
  return ABC_OK;
}

int32_t abc_mlp_get_params(abc_mlp* p, float* host) {
  if (!p || !host) return ABC_E_ARG;
  MCHK(p, hipStreamSynchronize(p->stream));
  MCHK(p, hipMemcpy(host, p->w, 4 * p->n_par, hipMemcpyDeviceToHost));
  return ABC_OK;
}

int32_t abc_mlp_set_params(abc_mlp* p, const float* host) {
  if (!p || !host) return ABC_E_ARG;
  MCHK(p, hipStreamSynchronize(p->stream));
  MCHK(p, hipMemcpy(p->w, host, 4 * p->n_par, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(refresh_bf16_kernel, dim3(p->w_tiles), dim3(256), 0, p->stream, p->w,
                     p->d_layers, (int)p->layers.size(), p->d_bf_off, p->Wb, p->WbT, p->Wf);
  MCHK(p, hipStreamSynchronize(p->stream));
  return ABC_OK;
}

int32_t abc_mlp_forward_dev(abc_mlp* p, int64_t n, const float* x_dev, float* y_dev) {
  if (!p || n < 0 || (n > 0 && (!x_dev || !y_dev))) return ABC_E_ARG;
  if (n > 0 && infer(p, n, x_dev, y_dev)) {
    MCHK(p, hipGetLastError());
    return ABC_OK;
  }
  for (int64_t o = 0; o < n; o += p->max_batch) {
    const int64_t b = std::min<int64_t>(p->max_batch, n - o);
    int rc = forward(p, b, x_dev + o * p->n_in);
    if (rc) return rc;
    hipLaunchKernelGGL(gather_out_kernel, dim3(g1(b * p->n_out, 256)), dim3(256), 0, p->stream,
                       p->O, (int)b, p->ns, p->out_pad, y_dev + o * p->n_out);
  }
  MCHK(p, hipGetLastError());
  return ABC_OK;
}

int32_t abc_mlp_grad_dev(abc_mlp* p, int64_t n, const float* x_dev, const float* t_dev,
                         float* grad_host, float* loss_host) {
  if (!p || n < 1 || n > p->max_batch || !x_dev || !t_dev) return ABC_E_ARG;
  GradParts P;
  int rc = grad(p, n, x_dev, t_dev, P);
  if (rc) return rc;
  hipLaunchKernelGGL(grad_sum_kernel, dim3(p->w_tiles + g1(p->n_bias, 256)), dim3(256), 0,
                     p->stream, P, p->d_layers, (int)p->layers.size(), p->g, p->loss_parts,
                     loss_tiles(p, n), p->loss);
  MCHK(p, hipStreamSynchronize(p->stream));
  if (grad_host) MCHK(p, hipMemcpy(grad_host, p->g, 4 * p->n_par, hipMemcpyDeviceToHost));
  if (loss_host) MCHK(p, hipMemcpy(loss_host, p->loss, 4, hipMemcpyDeviceToHost));
  return ABC_OK;
}

int32_t abc_mlp_train_step_dev(abc_mlp* p, int64_t n, const float* x_dev, const float* t_dev,
                               float lr, float beta1, float beta2, float eps, float weight_decay,
                               float* loss_dev_or_null) {
  if (!p || n < 1 || n > p->max_batch || !x_dev || !t_dev) return ABC_E_ARG;
  GradParts P;
  int rc = grad(p, n, x_dev, t_dev, P);
  if (rc) return rc;
  p->step++;
  const float c1 = 1.0f - std::pow(beta1, (float)p->step);
  const float c2 = 1.0f - std::pow(beta2, (float)p->step);
  hipLaunchKernelGGL(adam_kernel, dim3(p->w_tiles + g1(p->n_bias, 256)), dim3(256), 0, p->stream,
                     p->w, p->m, p->v, P, lr, beta1, beta2, eps, weight_decay, c1, c2,
                     p->d_layers, (int)p->layers.size(), p->d_bf_off, p->Wb, p->WbT, p->Wf,
                     p->loss_parts, loss_tiles(p, n), p->loss, loss_dev_or_null);
  MCHK(p, hipGetLastError());
  return ABC_OK;
}

int32_t abc_mlp_synchronize(abc_mlp* p) {
  if (!p) return ABC_E_ARG;
  MCHK(p, hipStreamSynchronize(p->stream));
  return ABC_OK;
}

int32_t abc_mlp_n_stats(const abc_mlp* p) { return p ? p->ns : ABC_E_ARG; }

int32_t abc_features_dev(int32_t model, int64_t n, const double* theta_dev, int32_t n_bins,
                         float* x_dev, void* stream) {
  if (model < 1 || model > 5 || n < 0 || n_bins < 1 || n_bins > ABC_MAX_BINS ||
      (n > 0 && (!theta_dev || !x_dev)))
    return ABC_E_ARG;
  if (n == 0) return ABC_OK;
  hipLaunchKernelGGL(features_kernel, dim3(g1(n, 256)), dim3(256), 0, (hipStream_t)stream, model,
                     n, theta_dev, n_bins, x_dev);
  return hipGetLastError() == hipSuccess ? ABC_OK : ABC_E_HIP;
}

int32_t abc_targets_dev(int64_t n, const double* stats_dev, int32_t K, const float* mean_dev,
                        const float* sd_dev, float* t_dev, void* stream) {
  if (n < 0 || K < 1 || (n > 0 && (!stats_dev || !mean_dev || !sd_dev || !t_dev))) return ABC_E_ARG;
  if (n == 0) return ABC_OK;
  hipLaunchKernelGGL(targets_kernel, dim3(g1(n * K, 256)), dim3(256), 0, (hipStream_t)stream, n,
                     stats_dev, K, mean_dev, sd_dev, t_dev);
  return hipGetLastError() == hipSuccess ? ABC_OK : ABC_E_HIP;
}

}  // extern "C"
