// plg_mlp.hip -- the learned part: a small multilayer perceptron with BF16
// weights and activations and FP32 accumulation, trained and evaluated on
// gfx950 by the kernels of this file (no library GEMM, no autograd).
//
// The network (no counterpart in the reference) maps cheap per-source inputs
// (zero-momentum correlators) to expensive outputs (high-momentum nucleon
// correlators):  x -> [Linear -> SiLU] x (L-1) -> Linear -> y.
//
// Rounding points (a CPU restatement mirrors them exactly):
//   forward   X_0 = bf16(x);  Z_l = X_l W_l^T + b_l  (bf16 x bf16 products,
//             FP32 sums);  X_{l+1} = bf16(silu(Z_l));  y = Z_{L-1}
//   loss      mean squared error over batch x outputs, dY = 2 (y - t) / (B N)
//   backward  dW_l = bf16(dZ_l)^T X_l,  db_l = sum_b dZ_l,
//             dX_l = bf16(dZ_l) W_l,  dZ_{l-1} = dX_l * silu'(Z_{l-1})
//   update    Adam on FP32 master weights, bf16 copies rewritten each step
// Every product is a v_mfma_f32_16x16x32_bf16 tile.
//
// Networks whose widths are all below 512 (the learned workload's 17-256-256-11)
// train in two launches a step, k_mlp_rows (forward, loss gradient and the
// chain of dX, which never leave a block of 16 rows) and k_mlp_update (weight
// and bias gradients and their Adam update); wider ones, whose products sum
// over K in split ranges, in one launch per product.  Both sum in the same order.
#include "plg_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

namespace plg {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr int MG_THREADS = 256;  // 4 waves, a 32 x 32 tile of C, 16 x 16 per wave

// C[m][n] (+ bias[n]) = sum_k A(m, k) B(k, n) with A(m, k) = A[m sam + k sak],
// B(k, n) = B[k sbk + n sbn] (bf16 bit patterns), FP32 accumulation.
// Optional epilogue: C (FP32, row stride ldc) and Cb = bf16(act(C)).
struct GemmArgs {
  int M, N, K;
  const uint16_t *A;
  int64_t sam, sak;
  const uint16_t *B;
  int64_t sbk, sbn;
  float *C;
  int64_t ldc;
  uint16_t *Cb;
  const float *bias;
  int silu;  // Cb = bf16(silu(C)) when set, else bf16(C)
  // split K: ks > 1 workgroup layers (blockIdx.z) sum K ranges of kper into
  // Cs[z][m][n]; k_gemm_reduce adds them and applies the epilogue
  int ks, kper;
  float *Cs;
};

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_grad(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

__global__ __launch_bounds__(MG_THREADS) void k_gemm_bf16(GemmArgs g) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * 32 + (wave >> 1) * 16;
  const int n0 = blockIdx.x * 32 + (wave & 1) * 16;
  // operand fragments of 16x16x32: lane l holds A[m0 + l%16][k0 + 8(l/16) + i]
  // and B[k0 + 8(l/16) + i][n0 + l%16], i < 8
  const int am = m0 + (lane & 15), bn = n0 + (lane & 15);
  const int kq = 8 * (lane >> 4);
  const int kb = blockIdx.z * g.kper, ke = min(g.K, kb + g.kper);
  f4 acc = {0, 0, 0, 0};
  for (int k0 = kb; k0 < ke; k0 += 32) {
    u16x8 a, b;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k = k0 + kq + i;
      a[i] = (am < g.M && k < ke) ? g.A[am * g.sam + k * g.sak] : (uint16_t)0;
      b[i] = (bn < g.N && k < ke) ? g.B[k * g.sbk + bn * g.sbn] : (uint16_t)0;
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), acc,
                                                 0, 0, 0);
  }
  // D of 16x16x32 (f32): lane l, value v -> row 4 (l/16) + v, column l % 16
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int m = m0 + 4 * (lane >> 4) + v, n = n0 + (lane & 15);
    if (g.ks > 1) {
      if (m < g.M && n < g.N) g.Cs[((int64_t)blockIdx.z * g.M + m) * g.N + n] = acc[v];
      continue;
    }
    if (m < g.M && n < g.N) {
      float z = acc[v] + (g.bias ? g.bias[n] : 0.0f);
      if (g.C) g.C[m * g.ldc + n] = z;
      if (g.Cb) g.Cb[m * g.ldc + n] = bf16_rne(g.silu ? silu(z) : z);
    }
  }
}

// the split-K partials summed in order of z, then the GEMM's epilogue
__global__ void k_gemm_reduce(GemmArgs g) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)g.M * g.N) return;
  const int m = (int)(e / g.N), n = (int)(e % g.N);
  float z = 0;
  for (int k = 0; k < g.ks; k++) z += g.Cs[(int64_t)k * g.M * g.N + e];
  z += g.bias ? g.bias[n] : 0.0f;
  if (g.C) g.C[m * g.ldc + n] = z;
  if (g.Cb) g.Cb[m * g.ldc + n] = bf16_rne(g.silu ? silu(z) : z);
}

__global__ void k_to_bf16(const float *__restrict__ x, uint16_t *__restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = bf16_rne(x[i]);
}

// dY = 2 (y - t) / (B N) (FP32 and bf16), per-block partial sums of (y - t)^2
__global__ void k_mse(const float *__restrict__ y, const float *__restrict__ t, float *__restrict__ dy,
                      uint16_t *__restrict__ dyb, float *__restrict__ part, int64_t n, float scale) {
  __shared__ float red[256];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float e2 = 0;
  if (i < n) {
    const float e = y[i] - t[i];
    const float d = 2.0f * e * scale;
    dy[i] = d;
    dyb[i] = bf16_rne(d);
    e2 = e * e;
  }
  red[threadIdx.x] = e2;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// dZ = dX * silu'(Z), FP32 and bf16
__global__ void k_silu_back(const float *__restrict__ dx, const float *__restrict__ z, float *__restrict__ dz,
                            uint16_t *__restrict__ dzb, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const float d = dx[i] * silu_grad(z[i]);
    dz[i] = d;
    dzb[i] = bf16_rne(d);
  }
}

// db[n] = sum_b dZ[b][n] in two deterministic stages.  k_bias_part: block
// (column group cx, row block rb) sums the rows [rb*rpb, (rb+1)*rpb) of 16
// columns; thread (row lane r, column j) takes the rows r, r + 16, ... with
// four independent accumulators (loads in flight together), and the 16 row
// lanes are added in LDS in a fixed order into part[rb][n].  k_bias_sum adds
// the row blocks' partials in order.  (One block per 16 columns walking all
// rows took about 35 us per call at B = 2048, most of a training step.)
constexpr int MG_BROWS = 16;  // row blocks of the bias gradient
__global__ __launch_bounds__(256) void k_bias_part(const float *__restrict__ dz, float *__restrict__ part, int B,
                                                   int N, int rpb) {
  __shared__ float red[16][17];
  const int j = threadIdx.x & 15, r = threadIdx.x >> 4;
  const int n = blockIdx.x * 16 + j;
  const int b0 = blockIdx.y * rpb, b1 = min(B, b0 + rpb);
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (n < N) {
    int b = b0 + r;
    for (; b + 48 < b1; b += 64)
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] += dz[(int64_t)(b + 16 * u) * N + n];
    for (int u = 0; b < b1; b += 16, u++) s[u & 3] += dz[(int64_t)b * N + n];
  }
  red[r][j] = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  if (r == 0 && n < N) {
    float t = 0;
    for (int k = 0; k < 16; k++) t += red[k][j];
    part[(int64_t)blockIdx.y * N + n] = t;
  }
}
__global__ void k_bias_sum(const float *__restrict__ part, float *__restrict__ db, int nrb, int N) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  float t = 0;
  for (int k = 0; k < nrb; k++) t += part[(int64_t)k * N + n];
  db[n] = t;
}

// the Adam step counter and its bias corrections 1 / (1 - b^step), on the
// device so that a captured training step replays unchanged
__global__ void k_adam_step(int *__restrict__ step, float *__restrict__ coef, float b1, float b2) {
  const int s = ++step[0];
  coef[0] = 1.0f / (1.0f - powf(b1, (float)s));
  coef[1] = 1.0f / (1.0f - powf(b2, (float)s));
}
// one parameter's Adam update, with the roundings spelled out (the two forms
// of a step leave the same bits)
__device__ __forceinline__ void adam_update(float &w, float &m, float &v, float g, float lr, float b1, float b2, float eps,
                                            float c1, float c2) {
#pragma clang fp contract(off)
  m = fmaf(1.0f - b1, g, b1 * m);
  v = fmaf(g, (1.0f - b2) * g, b2 * v);
  w = w - lr * (m * c1) / (sqrtf(v * c2) + eps);
}
// Adam (Kingma & Ba 2015) on FP32 master weights; wb: bf16 copy (NULL for biases)
__global__ void k_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                       const float *__restrict__ g, uint16_t *__restrict__ wb, int64_t n, float lr, float b1,
                       float b2, float eps, const float *__restrict__ coef) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float wi = w[i], mi = m[i], vi = v[i];
  adam_update(wi, mi, vi, g[i], lr, b1, b2, eps, coef[0], coef[1]);
  m[i] = mi;
  v[i] = vi;
  w[i] = wi;
  if (wb) wb[i] = bf16_rne(wi);
}

// ------------------------------------------------------------------ two-launch training step
constexpr int MF_WIDTH = 511;   // widest layer (products below 512 terms are one MFMA chain)
constexpr int MF_MAXL = 16;
constexpr int MF_THREADS = 1024, MF_WAVES = MF_THREADS / 64;
constexpr int MF_ZL = 2;        // hidden layers whose Z stays in LDS for the backward pass
// columns of the activations in LDS of a block of nw waves
__host__ __device__ constexpr int mlp_cols(int nw) { return nw == 1 ? 32 : nw == 4 ? 64 : nw == 8 ? 192 : 512; }
__host__ __device__ __forceinline__ int pad16(int n) { return (n + 15) / 16 * 16; }
__host__ __device__ __forceinline__ int pad32(int n) { return (n + 31) / 32 * 32; }

// An operand in fragment order: the 16 columns of a tile and 32 terms k that one
// MFMA reads are 1 KB in the order of the lanes (lane 16 (k % 32 / 8) + column,
// eight terms each), KS such blocks a tile.  Rows of a plain matrix, 512 bytes
// apart, took 4.6 us for a 256 x 256 layer.
__host__ __device__ __forceinline__ int64_t frag_idx(int col, int k, int KS) {
  return (((int64_t)(col >> 4) * KS + (k >> 5)) * 64 + ((k >> 3) & 3) * 16 + (col & 15)) * 8 + (k & 7);
}
// Device arrays of such a network.  The operands are padded to whole fragments
// with zeros, so the products run without bounds.
struct MlpDev {
  int L, B, BT;  // layers, rows of this call, rows of the arrays (a multiple of 32)
  int dims[MF_MAXL + 1];
  int64_t w_off[MF_MAXL], b_off[MF_MAXL];
  float *p, *g, *m, *v;
  uint16_t *wf[MF_MAXL];   // W_l, columns out, terms in
  uint16_t *wt[MF_MAXL];   // W_l, columns in, terms out
  uint16_t *xt[MF_MAXL];   // X_l, columns in, terms rows
  uint16_t *dzt[MF_MAXL];  // bf16(dZ_l), columns out, terms rows
  f4 *dzf[MF_MAXL];        // dZ_l: four rows of a column, [tile][row / 4][16 columns]
  float *zs[MF_MAXL];      // hidden Z_l: a lane's rows of its column, [row block][tile][lane]
};

// parameter copies in the layouts of the products
__device__ __forceinline__ void mlp_put_weight(const MlpDev &d, int l, int o, int i, float w) {
  const uint16_t b = bf16_rne(w);
  d.wf[l][frag_idx(o, i, pad32(d.dims[l]) / 32)] = b;
  d.wt[l][frag_idx(i, o, pad32(d.dims[l + 1]) / 32)] = b;
}
__global__ void k_mlp_pack(MlpDev d) {
  const int l = blockIdx.y, Ni = d.dims[l], n = Ni * d.dims[l + 1];
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) mlp_put_weight(d, l, e / Ni, e % Ni, d.p[d.w_off[l] + e]);
}

// barrier over the workgroup's LDS only: stores to memory stay in flight (a
// __syncthreads would wait for them at every layer)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The rows [4 Q blockIdx.x, + 4 Q) through the whole network (Q rows a lane, 4 or
// 2; NW waves): every layer's outputs are column tiles of 16, one per wave in turn,
// the activations stay in LDS.  BACK: the loss gradient 2 (y - t) scale and the chain of dX as well, with
// the transposed operands of the weight gradients for k_mlp_update.  y (may be
// NULL): outputs, [B][out].  coef (may be NULL): the step counter is advanced
// and its bias corrections are written.
// Bound by the chain of layers: eight rows a block (Q = 2, half of each MFMA's
// rows unused) spread the learned workload's 2 048 rows over 256 CUs and halve
// the activations' vector instructions of a wave (a 256-wide layer 2.6 -> 2.2
// us); 16 rows where the batch fills the CUs.  There a block has as many waves as
// the widest layer has column tiles (two tiles a wave from 129 to 192 columns),
// so that idle waves leave the CUs to other blocks: forward passes of 131 072
// rows, 16 waves a block always / so, us: 17-11 47 / 12, 17-64-11 83 / 28,
// 17-129-11 98 / 69 (launch by product 19, 75, 95).  A wave loads the weights of
// its first tile of the next layer before this layer's stores.
// 17-256-256-11 at 2 048 rows: 17 us (a 256 x 256 layer streams its 131 KB of
// weights through the CU in about 2 us; the transposed outputs' stores are
// 4 us), k_mlp_update 6 us; a step takes 26 us against 153 us in 23 launches.
template <bool BACK, int Q, int NW>
__global__ __launch_bounds__(64 * NW) void k_mlp_rows(MlpDev d, const float *__restrict__ x, const float *__restrict__ t,
                                                         float scale, float *__restrict__ y, int *__restrict__ step,
                                                         float *__restrict__ coef, float b1, float b2) {
  constexpr int LD = mlp_cols(NW) + 8;  // the 16 rows of a fragment read start on distinct banks
  __shared__ __align__(16) uint16_t act[2][16][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * 4 * Q, lc = lane & 15, lk = 8 * (lane >> 4);
  // the lane's rows: of the block, and of act (and of the MFMA)
  const int rq = Q * (lane >> 4), r4 = 4 * (lane >> 4);
  __shared__ float zl_[MF_ZL][64 * NW * Q];  // Z of the waves' first tiles of the first hidden layers
  // eight fragments (256 terms) of rows [16 tile, + 16) of a padded matrix
  u16x8 w8[8];
  auto load = [&](const uint16_t *w, int KP, int tile, int k0) {
    const u16x8 *wr = (const u16x8 *)w + ((int64_t)tile * (KP / 32) + k0 / 32) * 64 + lane;
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (k0 + 32 * i < KP) w8[i] = wr[i * 64];
  };
  // rows of act[cur] times them: K in order; the first fragments of the
  // wave's first tile are loaded already
  auto product = [&](const uint16_t *w, int KP, int tile, int cur) {
    f4 acc = {0, 0, 0, 0};
    for (int k0 = 0; k0 < KP; k0 += 256) {
      if (k0 > 0 || tile != wave) load(w, KP, tile, k0);
      if (k0 + 256 <= KP) {
        u16x8 a[8];
#pragma unroll
        for (int i = 0; i < 8; i++) a[i] = *(const u16x8 *)&act[cur][lc][k0 + 32 * i + lk];
#pragma unroll
        for (int i = 0; i < 8; i++)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a[i]), __builtin_bit_cast(bf8, w8[i]), acc, 0, 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (k0 + 32 * i < KP) {
            const u16x8 a = *(const u16x8 *)&act[cur][lc][k0 + 32 * i + lk];
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, w8[i]), acc, 0, 0, 0);
          }
      }
    }
    return acc;
  };
  // the lane's four rows of a column as bf16: to the next product's LDS rows
  // and to a transposed array (rows past the batch zero)
  typedef uint16_t hv __attribute__((ext_vector_type(Q)));
  typedef float fv __attribute__((ext_vector_type(Q)));
  auto put = [&](const hv &h, int n, int N, int nxt, uint16_t *tr) {
#pragma unroll
    for (int q = 0; q < Q; q++) act[nxt][r4 + q][n] = h[q];
    if (tr && n < N) *(hv *)(tr + frag_idx(n, row0 + rq, d.BT / 32)) = h;
  };
  auto put_dz = [&](int l, int tile, const fv &dz) {
    *(fv *)((float *)(d.dzf[l] + ((int64_t)tile * (d.BT / 4) + (row0 + rq) / 4) * 16 + lc) + ((row0 + rq) & 3)) = dz;
  };
  auto bias_of = [&](int l, int n) { return l < d.L && n < d.dims[l + 1] ? d.p[d.b_off[l] + n] : 0.0f; };
  auto row_in = [&](int q) { return row0 + rq + q < d.B; };
  auto targets = [&](int n, float (&tv)[Q]) {
    const int No = d.dims[d.L];
#pragma unroll
    for (int q = 0; q < Q; q++) tv[q] = n < No && row_in(q) ? t[(int64_t)(row0 + rq + q) * No + n] : 0.0f;
  };
  float bias0 = bias_of(0, wave * 16 + lc), tv0[Q] = {};
  if (wave * 16 < d.dims[1]) load(d.wf[0], pad32(d.dims[0]), wave, 0);
  if (BACK) targets(wave * 16 + lc, tv0);
  if (wave < 4 * Q) {  // 64 lanes a row, the wave's rows loaded together
    constexpr int RW = (4 * Q + NW - 1) / NW;
    const int Ni = d.dims[0], KP = pad32(Ni);
    for (int i = lane; i < KP; i += 64) {
      uint16_t b[RW];
#pragma unroll
      for (int k = 0; k < RW; k++) {
        const int r = wave + k * NW;
        b[k] = (i < Ni && row0 + r < d.B) ? bf16_rne(x[(int64_t)(row0 + r) * Ni + i]) : (uint16_t)0;
      }
#pragma unroll
      for (int k = 0; k < RW; k++) {
        const int r = wave + k * NW;
        act[0][r / Q * 4 + r % Q][i] = b[k];
        if (BACK && i < Ni) d.xt[0][frag_idx(i, row0 + r, d.BT / 32)] = b[k];
      }
    }
  }
  if (BACK && coef && blockIdx.x == 0 && tid == 0) {
    const int s = ++step[0];
    coef[0] = 1.0f / (1.0f - powf(b1, (float)s));
    coef[1] = 1.0f / (1.0f - powf(b2, (float)s));
  }
  lds_barrier();
  int cur = 0;
  for (int l = 0; l < d.L; l++) {
    const int Ni = d.dims[l], No = d.dims[l + 1], NT = pad16(No) / 16;
    const bool last = l == d.L - 1;
    const uint16_t *wl = d.wf[l];
    f4 acc = {0, 0, 0, 0};
    if (wave < NT) acc = product(wl, pad32(Ni), wave, cur);
    float bias = bias0;
    // the wave's first operands of the next product, ahead of this layer's
    // stores (a wait for later loads would be a wait for the stores too)
    bias0 = bias_of(l + 1, wave * 16 + lc);
    if (!last) {
      if (wave * 16 < d.dims[l + 2]) load(d.wf[l + 1], pad32(No), wave, 0);
    } else if (BACK && l > 0) {
      if (wave * 16 < Ni) load(d.wt[l], pad32(No), wave, 0);
    }
    for (int tile = wave; tile < pad32(No) / 16; tile += NW) {
      const int n = tile * 16 + lc;
      hv h = {};
      if (tile < NT) {
        float tv[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) tv[q] = tv0[q];
        if (tile != wave) {
          bias = bias_of(l, n);
          if (BACK && last) targets(n, tv);
          acc = product(wl, pad32(Ni), tile, cur);
        }
        fv z, dz = {};
#pragma unroll
        for (int q = 0; q < Q; q++) {
          z[q] = acc[q] + bias;
          const bool in = n < No && row_in(q);
          if (!last) {
            h[q] = in ? bf16_rne(silu(z[q])) : (uint16_t)0;
          } else if (in) {
            if (y) y[(int64_t)(row0 + rq + q) * No + n] = z[q];
            if (BACK) {
              const float df = z[q] - tv[q];
              dz[q] = 2.0f * df * scale;
              h[q] = bf16_rne(dz[q]);
            }
          }
        }
        if (BACK && !last) {
          if (tile == wave && l < MF_ZL) ((fv *)zl_[l])[tid] = z;
          else ((fv *)d.zs[l])[((int64_t)blockIdx.x * NT + tile) * 64 + lane] = z;
        }
        if (BACK && last && n < No) put_dz(l, tile, dz);
      }
      if (!last || BACK) put(h, n, No, cur ^ 1, BACK ? (last ? d.dzt[l] : d.xt[l + 1]) : nullptr);
    }
    // (waves of several tiles have overwritten their prefetched weights)
    if (wave + NW < NT) {
      if (!last) {
        if (wave * 16 < d.dims[l + 2]) load(d.wf[l + 1], pad32(No), wave, 0);
      } else if (BACK && l > 0) {
        if (wave * 16 < Ni) load(d.wt[l], pad32(No), wave, 0);
      }
    }
    cur ^= 1;
    lds_barrier();
  }
  if (!BACK) return;
  for (int l = d.L - 1; l > 0; l--) {
    const int Ni = d.dims[l], No = d.dims[l + 1], NT = pad16(Ni) / 16;
    const uint16_t *wl = d.wt[l];
    f4 dx = {0, 0, 0, 0};
    if (wave < NT) dx = product(wl, pad32(No), wave, cur);
    if (l > 1 && wave * 16 < d.dims[l - 1]) load(d.wt[l - 1], pad32(Ni), wave, 0);
    for (int tile = wave; tile < pad32(Ni) / 16; tile += NW) {
      const int n = tile * 16 + lc;
      hv h = {};
      if (tile < NT) {
        const fv z = tile == wave && l <= MF_ZL ? ((const fv *)zl_[l - 1])[tid]
                                                : ((const fv *)d.zs[l - 1])[((int64_t)blockIdx.x * NT + tile) * 64 + lane];
        if (tile != wave) dx = product(wl, pad32(No), tile, cur);
        fv dz;
#pragma unroll
        for (int q = 0; q < Q; q++) {
          const float v = dx[q] * silu_grad(z[q]);
          dz[q] = n < Ni && row_in(q) ? v : 0.0f;
          h[q] = bf16_rne(dz[q]);
        }
        if (n < Ni) put_dz(l - 1, tile, dz);
      }
      put(h, n, Ni, cur ^ 1, d.dzt[l - 1]);
    }
    if (l > 1 && wave + NW < NT && wave * 16 < d.dims[l - 1]) load(d.wt[l - 1], pad32(Ni), wave, 0);
    cur ^= 1;
    lds_barrier();
  }
}

// Weight and bias gradients and their update.  A block takes a 32 x 32 tile of
// dW_l = dZ_l^T X_l, wave z the z-th K range (kper rows, the split of
// gemm_ksplit), and the ranges are added in order of z; or four columns of a bias,
// summed as k_bias_part and k_bias_sum do.  ADAM: the parameters are updated in
// place with their padded bf16 copies, else the gradient is written to g.
// Bound by the latency of one pass of operand loads (all of a wave's range in
// flight); no partial sum leaves the block.
template <bool ADAM>
__global__ __launch_bounds__(MF_THREADS) void k_mlp_update(MlpDev d, int ks, int kper, float lr, float b1, float b2,
                                                           float eps, const float *__restrict__ coef) {
  __shared__ float part[MF_WAVES][32][33];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  struct Param {
    float w, m, v;
  };
  auto fetch = [&](int64_t e) { return ADAM ? Param{d.p[e], d.m[e], d.v[e]} : Param{}; };
  const float c1 = ADAM ? coef[0] : 0.0f, c2 = ADAM ? coef[1] : 0.0f;
  auto apply = [&](int64_t e, Param a, float gi) {
    if (ADAM) {
      adam_update(a.w, a.m, a.v, gi, lr, b1, b2, eps, c1, c2);
      d.p[e] = a.w;
      d.m[e] = a.m;
      d.v[e] = a.v;
      return a.w;
    }
    d.g[e] = gi;
    return 0.0f;
  };
  // the block's tile (weight tiles of every layer, then the bias groups)
  int id = blockIdx.x, l = 0, nt = 0;
  for (; l < d.L; l++) {
    nt = (pad32(d.dims[l + 1]) / 32) * (pad32(d.dims[l]) / 32);
    if (id < nt) break;
    id -= nt;
  }
  if (l < d.L) {
    const int Ni = d.dims[l], No = d.dims[l + 1], tn = pad32(Ni) / 32;
    const int m0 = id / tn * 32, n0 = id % tn * 32, lc = lane & 15;
    const int o = m0 + tid / 32, i = n0 + tid % 32;
    const bool in = o < No && i < Ni;
    const int64_t e = d.w_off[l] + (int64_t)o * Ni + i;
    const Param own = in ? fetch(e) : Param{};  // in flight beside the operands
    if (wave < ks) {
      const int kb = wave * kper, ke = min(d.B, kb + kper);
      const int KS = d.BT / 32;
      const u16x8 *A = (const u16x8 *)d.dzt[l] + (int64_t)(m0 / 16) * KS * 64 + lane;
      const u16x8 *X = (const u16x8 *)d.xt[l] + (int64_t)(n0 / 16) * KS * 64 + lane;
      f4 acc[2][2] = {{{0, 0, 0, 0}, {0, 0, 0, 0}}, {{0, 0, 0, 0}, {0, 0, 0, 0}}};
      // halves of the tile that are padding alone are not read: a batch of
      // many rows and a small layer are bound by one CU's reads (17-11 at 1 M
      // rows: a training step 2.29 -> 1.61 ms)
      const bool a2 = m0 + 16 < No, b2 = n0 + 16 < Ni;
      for (int k0 = kb; k0 < ke; k0 += 128) {
        u16x8 a[4][2] = {}, b[4][2] = {};
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (k0 + 32 * i < ke)
#pragma unroll
            for (int q = 0; q < 2; q++) {
              if (q == 0 || a2) a[i][q] = A[(int64_t)(q * KS + k0 / 32 + i) * 64];
              if (q == 0 || b2) b[i][q] = X[(int64_t)(q * KS + k0 / 32 + i) * 64];
            }
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (k0 + 32 * i < ke)
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
              for (int r = 0; r < 2; r++)
                acc[q][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a[i][q]),
                                                                    __builtin_bit_cast(bf8, b[i][r]), acc[q][r], 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
          for (int v = 0; v < 4; v++) part[wave][16 * q + 4 * (lane >> 4) + v][16 * r + lc] = acc[q][r][v];
    }
    __syncthreads();
    if (in) {
      float gi = 0;
      for (int z = 0; z < ks; z++) gi += part[z][tid / 32][tid % 32];
      const float w = apply(e, own, gi);
      if (ADAM) mlp_put_weight(d, l, o, i, w);
    }
    return;
  }
  for (l = 0; l < d.L; l++) {
    nt = (d.dims[l + 1] + 3) / 4;
    if (id < nt) break;
    id -= nt;
  }
  if (l >= d.L) return;
  // thread: row lane r, column j, row block rb
  const int No = d.dims[l + 1], rpb = (d.B + MG_BROWS - 1) / MG_BROWS;
  const int r = tid & 15, j = tid >> 4 & 3, rb = tid >> 6, n = id * 4 + j;
  float(*red)[4][17] = reinterpret_cast<float(*)[4][17]>(&part[0][0][0]);  // [row block][column][row lane]
  {
    const int r0 = rb * rpb, r1 = min(d.B, r0 + rpb);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (n < No) {
      const float *dzl = (const float *)d.dzf[l] + ((int64_t)(n >> 4) * (d.BT / 4) * 16 + (n & 15)) * 4;
      auto dz = [&](int b) { return dzl[(int64_t)(b >> 2) * 64 + (b & 3)]; };
      int b = r0 + r;
      for (; b + 48 < r1; b += 64)
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] += dz(b + 16 * u);
#pragma unroll
      for (int u = 0; u < 4; u++, b += 16)
        if (b < r1) s[u] += dz(b);
    }
    red[rb][j][r] = (s[0] + s[1]) + (s[2] + s[3]);
  }
  __syncthreads();
  float t = 0;
  if (tid < 4 * MG_BROWS)  // thread: column tid / 16, row block tid % 16
    for (int k = 0; k < 16; k++) t += red[tid & 15][tid >> 4][k];
  __syncthreads();
  float *bp = &part[0][0][0];
  if (tid < 4 * MG_BROWS) bp[tid] = t;
  __syncthreads();
  if (tid < 4 && id * 4 + tid < No) {
    float db = 0;
    for (int k = 0; k < MG_BROWS; k++) db += bp[tid * 16 + k];
    const int64_t e = d.b_off[l] + id * 4 + tid;
    apply(e, fetch(e), db);
  }
}

static int blocks(int64_t n, int t = 256) { return (int)((n + t - 1) / t); }
constexpr float MG_B1 = 0.9f, MG_B2 = 0.999f, MG_EPS = 1e-8f;  // Adam

}  // namespace plg

using namespace plg;

// ------------------------------------------------------------------ the network object
struct plg_mlp_s {
  std::vector<int> dims;  // dims[0] = inputs, dims[L] = outputs
  int L = 0, max_batch = 0;
  int64_t nparams = 0;
  std::vector<int64_t> w_off, b_off;  // offsets of W_l [out][in] and b_l [out] in the parameter vector
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  uint16_t *pb = nullptr;  // bf16 copy, same offsets (biases unused)
  // activations, per layer l: X_l (bf16, [B][dims[l]]), Z_l (FP32, [B][dims[l+1]])
  std::vector<uint16_t *> X;
  std::vector<float *> Z;
  float *dz = nullptr, *dx = nullptr, *part = nullptr;
  float *bpart = nullptr;  // bias-gradient partials [MG_BROWS][widest]
  uint16_t *dzb = nullptr;
  int64_t step = 0;
  float *ksw = nullptr;     // split-K partials of the products
  int *d_step = nullptr;    // Adam step on the device
  float *d_coef = nullptr;  // its bias corrections
  // one training step captured as a graph, for the arguments it was captured with
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  const float *gx = nullptr, *gt = nullptr;
  int gB = 0;
  float glr = 0;
  // widths below 512: the two-launch step on padded and transposed arrays
  bool rows = false;
  MlpDev dev{};
  std::vector<void *> allocs;
  ~plg_mlp_s() {
    if (exec) hipGraphExecDestroy(exec);
    if (graph) hipGraphDestroy(graph);
    if (cap) hipStreamDestroy(cap);
    for (void *q : allocs) hipFree(q);
  }
};

static int mlp_alloc(plg_mlp_s *net, void **dst, size_t bytes) {
  if (hipMalloc(dst, bytes) != hipSuccess) return fail(PLG_ERR_ALLOC, "MLP device allocation failed");
  net->allocs.push_back(*dst);
  return PLG_OK;
}

// K split for long, narrow products (the weight gradients sum over the
// batch): up to MG_KSPLIT ranges of at least 128, when the tile grid is small
constexpr int MG_KSPLIT = 16;
static int gemm_ksplit(int M, int N, int K) {
  const int64_t tiles = (int64_t)((N + 31) / 32) * ((M + 31) / 32);
  if (K < 512 || tiles >= 512) return 1;
  return std::max(1, std::min(MG_KSPLIT, K / 128));
}
static void gemm(GemmArgs a, float *ws, hipStream_t st) {
  a.ks = ws ? gemm_ksplit(a.M, a.N, a.K) : 1;
  a.kper = a.ks > 1 ? ((a.K + a.ks - 1) / a.ks + 31) / 32 * 32 : a.K;
  a.ks = a.ks > 1 ? (a.K + a.kper - 1) / a.kper : 1;
  a.Cs = ws;
  dim3 grid((unsigned)((a.N + 31) / 32), (unsigned)((a.M + 31) / 32), (unsigned)a.ks);
  k_gemm_bf16<<<grid, MG_THREADS, 0, st>>>(a);
  if (a.ks > 1) k_gemm_reduce<<<blocks((int64_t)a.M * a.N), 256, 0, st>>>(a);
}

// the arrays of a call with B rows
static MlpDev rows_dev(const plg_mlp_s *net, int B) {
  MlpDev d = net->dev;
  d.B = B;
  return d;
}
// forward (outputs y, may be NULL with t) and, with t, the loss gradient and
// everything the weight gradients read; count: advance the Adam step
static int rows_pass(plg_mlp_s *net, const float *x, const float *t, int B, float *y, bool count, hipStream_t st) {
  const MlpDev d = rows_dev(net, B);
  const float scale = 1.0f / (float)((int64_t)B * net->dims[net->L]);
  float *coef = count ? net->d_coef : nullptr;
  auto launch = [&](auto Q, auto NW) {
    const dim3 grid(pad32(B) / (4 * Q.value)), block(64 * NW.value);
    if (t) k_mlp_rows<true, Q.value, NW.value><<<grid, block, 0, st>>>(d, x, t, scale, y, net->d_step, coef, MG_B1, MG_B2);
    else k_mlp_rows<false, Q.value, NW.value><<<grid, block, 0, st>>>(d, x, nullptr, 0.0f, y, nullptr, nullptr, MG_B1, MG_B2);
  };
  // eight rows a block while 16 would leave CUs of the 256 without one; the
  // waves of the blocks of 16 by the widest layer (k_mlp_rows has the times)
  const int out = *std::max_element(net->dims.begin() + 1, net->dims.end()), all = std::max(out, net->dims[0]);
  if (pad32(B) / 8 <= 256) launch(ic<2>{}, ic<16>{});
  else if (out <= 16 && all <= mlp_cols(1)) launch(ic<4>{}, ic<1>{});
  else if (out <= 64 && all <= mlp_cols(4)) launch(ic<4>{}, ic<4>{});
  else if (out <= 192 && all <= mlp_cols(8)) launch(ic<4>{}, ic<8>{});
  else launch(ic<4>{}, ic<16>{});
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP rows launch failed");
}
// gradients of the last rows_pass: into net->g, or (adam) applied
static int rows_update(plg_mlp_s *net, int B, bool adam, float lr, hipStream_t st) {
  const MlpDev d = rows_dev(net, B);
  int grid = 0;
  for (int l = 0; l < net->L; l++)
    grid += (pad32(d.dims[l + 1]) / 32) * (pad32(d.dims[l]) / 32) + (d.dims[l + 1] + 3) / 4;
  // the K ranges of gemm_ksplit (a layer has at most 256 tiles here)
  int ks = gemm_ksplit(32, 32, B), kper = B;
  if (ks > 1) {
    kper = pad32((B + ks - 1) / ks);
    ks = (B + kper - 1) / kper;
  }
  if (adam) k_mlp_update<true><<<grid, MF_THREADS, 0, st>>>(d, ks, kper, lr, MG_B1, MG_B2, MG_EPS, net->d_coef);
  else k_mlp_update<false><<<grid, MF_THREADS, 0, st>>>(d, ks, kper, 0.0f, MG_B1, MG_B2, MG_EPS, nullptr);
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP update launch failed");
}
// loss partials (net->part) of outputs in net->Z.back()
static int rows_loss(plg_mlp_s *net, const float *t, int B, hipStream_t st) {
  const int64_t ny = (int64_t)B * net->dims[net->L];
  k_mse<<<blocks(ny), 256, 0, st>>>(net->Z[net->L - 1], t, net->dz, net->dzb, net->part, ny, 1.0f / (float)ny);
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP loss launch failed");
}

static int mlp_forward(plg_mlp_s *net, const float *x, int B, hipStream_t st) {
  const int64_t n0 = (int64_t)B * net->dims[0];
  k_to_bf16<<<blocks(n0), 256, 0, st>>>(x, net->X[0], n0);
  for (int l = 0; l < net->L; l++) {
    const int Ni = net->dims[l], No = net->dims[l + 1];
    const bool last = l == net->L - 1;
    GemmArgs a{};
    a.M = B; a.N = No; a.K = Ni;
    a.A = net->X[l]; a.sam = Ni; a.sak = 1;              // X_l [b][i]
    a.B = net->pb + net->w_off[l]; a.sbk = 1; a.sbn = Ni;  // W_l^T: (i, o) -> W[o][i]
    a.C = net->Z[l]; a.ldc = No;
    a.Cb = last ? nullptr : net->X[l + 1];
    a.bias = net->p + net->b_off[l];
    a.silu = 1;
    gemm(a, net->ksw, st);
  }
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP forward launch failed");
}

// loss partials + full backward into net->g
static int mlp_backward(plg_mlp_s *net, const float *t, int B, hipStream_t st) {
  const int Lx = net->L;
  const int64_t ny = (int64_t)B * net->dims[Lx];
  k_mse<<<blocks(ny), 256, 0, st>>>(net->Z[Lx - 1], t, net->dz, net->dzb, net->part, ny,
                                   1.0f / (float)ny);
  for (int l = Lx - 1; l >= 0; l--) {
    const int Ni = net->dims[l], No = net->dims[l + 1];
    // dW_l[o][i] = sum_b dZ[b][o] X_l[b][i]
    GemmArgs a{};
    a.M = No; a.N = Ni; a.K = B;
    a.A = net->dzb; a.sam = 1; a.sak = No;
    a.B = net->X[l]; a.sbk = Ni; a.sbn = 1;
    a.C = net->g + net->w_off[l]; a.ldc = Ni;
    gemm(a, net->ksw, st);
    {
      const int rpb = (B + MG_BROWS - 1) / MG_BROWS;
      k_bias_part<<<dim3(blocks(No, 16), MG_BROWS), 256, 0, st>>>(net->dz, net->bpart, B, No, rpb);
      k_bias_sum<<<blocks(No), 256, 0, st>>>(net->bpart, net->g + net->b_off[l], MG_BROWS, No);
    }
    if (l > 0) {
      // dX_l[b][i] = sum_o dZ[b][o] W_l[o][i], then dZ_{l-1} = dX_l silu'(Z_{l-1})
      GemmArgs d{};
      d.M = B; d.N = Ni; d.K = No;
      d.A = net->dzb; d.sam = No; d.sak = 1;
      d.B = net->pb + net->w_off[l]; d.sbk = Ni; d.sbn = 1;
      d.C = net->dx; d.ldc = Ni;
      gemm(d, net->ksw, st);
      const int64_t n = (int64_t)B * Ni;
      k_silu_back<<<blocks(n), 256, 0, st>>>(net->dx, net->Z[l - 1], net->dz, net->dzb, n);
    }
  }
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP backward launch failed");
}

static int mlp_loss(plg_mlp_s *net, int B, hipStream_t st, double *loss) {
  const int64_t ny = (int64_t)B * net->dims[net->L];
  const int nb = blocks(ny);
  std::vector<float> h(nb);
  if (hipMemcpyAsync(h.data(), net->part, nb * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return fail(PLG_ERR_HIP, "MLP loss read-back failed");
  double s = 0;
  for (float v : h) s += v;
  *loss = s / (double)ny;
  return PLG_OK;
}

// one Adam step: forward, backward, step counter, updates (no allocation,
// no memset: capturable)
static int train_step(plg_mlp_s *net, const float *x, const float *t, int B, float lr, hipStream_t st) {
  int rc;
  if ((rc = mlp_forward(net, x, B, st)) || (rc = mlp_backward(net, t, B, st))) return rc;
  k_adam_step<<<1, 1, 0, st>>>(net->d_step, net->d_coef, MG_B1, MG_B2);
  // the parameters (W_0, b_0, W_1, ...) are one contiguous array: one update
  // launch for all of them (the biases' bf16 copies are written but unused)
  k_adam<<<blocks(net->nparams), 256, 0, st>>>(net->p, net->m, net->v, net->g, net->pb, net->nparams, lr, MG_B1,
                                               MG_B2, MG_EPS, net->d_coef);
  return hipGetLastError() == hipSuccess ? PLG_OK : fail(PLG_ERR_HIP, "MLP update launch failed");
}

static int check_batch(plg_mlp_s *net, int B) {
  if (!net) return fail(PLG_ERR_INVALID, "null MLP handle");
  if (B <= 0 || B > net->max_batch)
    return fail(PLG_ERR_RANGE, "batch " + std::to_string(B) + " outside 1.." + std::to_string(net->max_batch));
  return PLG_OK;
}

extern "C" {

int plg_mlp_create(const int *dims, int nlayers, int max_batch, plg_mlp *out) {
  if (!dims || !out || nlayers < 1 || nlayers > 16 || max_batch <= 0)
    return fail(PLG_ERR_INVALID, "plg_mlp_create: bad arguments");
  for (int l = 0; l <= nlayers; l++)
    if (dims[l] <= 0 || dims[l] > 65536) return fail(PLG_ERR_INVALID, "plg_mlp_create: bad layer width");
  auto *net = new plg_mlp_s();
  net->dims.assign(dims, dims + nlayers + 1);
  net->L = nlayers;
  net->max_batch = max_batch;
  int64_t off = 0, widest = 0;
  for (int l = 0; l < nlayers; l++) {
    net->w_off.push_back(off);
    off += (int64_t)dims[l] * dims[l + 1];
    net->b_off.push_back(off);
    off += dims[l + 1];
  }
  for (int l = 0; l <= nlayers; l++) widest = std::max<int64_t>(widest, dims[l]);
  net->nparams = off;
  // every array in one zeroed allocation (padding is never written)
  std::vector<std::pair<void **, size_t>> arrays;
  auto want = [&](auto **q, size_t bytes) { arrays.emplace_back((void **)q, bytes); };
  const size_t pbytes = (size_t)off * sizeof(float);
  want(&net->p, pbytes);
  want(&net->g, pbytes);
  want(&net->m, pbytes);
  want(&net->v, pbytes);
  want(&net->pb, (size_t)off * sizeof(uint16_t));
  net->rows = true;
  for (int l = 0; l <= nlayers; l++) net->rows = net->rows && dims[l] <= MF_WIDTH;
  if (net->rows) {
    MlpDev &d = net->dev;
    d.L = nlayers;
    d.BT = pad32(max_batch);
    for (int l = 0; l <= nlayers; l++) d.dims[l] = dims[l];
    for (int l = 0; l < nlayers; l++) {
      const size_t Ni = dims[l], No = dims[l + 1], BT = d.BT;
      d.w_off[l] = net->w_off[l];
      d.b_off[l] = net->b_off[l];
      want(&d.wf[l], (size_t)pad16(No) * pad32(Ni) * sizeof(uint16_t));
      want(&d.wt[l], (size_t)pad16(Ni) * pad32(No) * sizeof(uint16_t));
      want(&d.xt[l], (size_t)pad32(Ni) * BT * sizeof(uint16_t));
      want(&d.dzt[l], (size_t)pad32(No) * BT * sizeof(uint16_t));
      want(&d.dzf[l], (size_t)pad16(No) * BT * sizeof(float));
      want(&d.zs[l], (size_t)pad16(No) * BT * sizeof(float));
    }
  }
  // the launch-per-product form's activations; the outputs and the loss's
  // arrays serve both
  net->X.assign(nlayers, nullptr);
  net->Z.assign(nlayers, nullptr);
  for (int l = 0; l < nlayers; l++) {
    if (!net->rows) want(&net->X[l], (size_t)max_batch * dims[l] * sizeof(uint16_t));
    if (!net->rows || l == nlayers - 1) want(&net->Z[l], (size_t)max_batch * dims[l + 1] * sizeof(float));
  }
  const size_t wb = (size_t)max_batch * (net->rows ? dims[nlayers] : widest);
  want(&net->dz, wb * sizeof(float));
  want(&net->dzb, wb * sizeof(uint16_t));
  want(&net->part, (size_t)blocks((int64_t)wb) * sizeof(float));
  if (!net->rows) {
    want(&net->dx, wb * sizeof(float));
    want(&net->bpart, (size_t)MG_BROWS * widest * sizeof(float));
    // split-K partials: a bound of ks x M x N over the network's products
    // at any batch up to max_batch (the split ignoring the tile count)
    size_t kw = 1;
    for (int l = 0; l < nlayers; l++) {
      const int Ni = dims[l], No = dims[l + 1];
      const int64_t shapes[3][3] = {{max_batch, No, Ni}, {No, Ni, max_batch}, {max_batch, Ni, No}};
      for (auto &sh : shapes)
        if (sh[2] >= 512) kw = std::max(kw, (size_t)std::min<int64_t>(MG_KSPLIT, sh[2] / 128) * sh[0] * sh[1]);
    }
    want(&net->ksw, kw * sizeof(float));
  }
  want(&net->d_step, sizeof(int));
  want(&net->d_coef, 2 * sizeof(float));
  size_t total = 0;
  for (auto &q : arrays) total += (q.second + 255) / 256 * 256;
  unsigned char *arena = nullptr;
  int rc = mlp_alloc(net, (void **)&arena, total);
  if (!rc && hipMemset(arena, 0, total) != hipSuccess) rc = fail(PLG_ERR_HIP, "MLP array clear failed");
  if (!rc)
    for (auto &q : arrays) {
      *q.first = arena;
      arena += (q.second + 255) / 256 * 256;
    }
  if (net->rows) {
    net->dev.p = net->p;
    net->dev.g = net->g;
    net->dev.m = net->m;
    net->dev.v = net->v;
  }
  if (rc) {
    delete net;
    return rc;
  }
  *out = net;
  return PLG_OK;
}

int plg_mlp_nparams(plg_mlp net, int64_t *n) {
  if (!net || !n) return fail(PLG_ERR_INVALID, "null argument");
  *n = net->nparams;
  return PLG_OK;
}

// parameters: for each layer, W [out][in] then b [out], FP32.  Resets Adam.
int plg_mlp_set_params(plg_mlp net, const float *host) {
  if (!net || !host) return fail(PLG_ERR_INVALID, "null argument");
  const size_t bytes = (size_t)net->nparams * sizeof(float);
  if (hipMemcpy(net->p, host, bytes, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(net->m, 0, bytes) != hipSuccess || hipMemset(net->v, 0, bytes) != hipSuccess)
    return fail(PLG_ERR_HIP, "MLP parameter upload failed");
  if (net->rows) {
    int most = 0;
    for (int l = 0; l < net->L; l++) most = std::max(most, net->dims[l] * net->dims[l + 1]);
    k_mlp_pack<<<dim3(blocks(most), net->L), 256>>>(net->dev);
  } else {
    k_to_bf16<<<blocks(net->nparams), 256>>>(net->p, net->pb, net->nparams);
  }
  net->step = 0;
  if (hipMemset(net->d_step, 0, sizeof(int)) != hipSuccess) return fail(PLG_ERR_HIP, "MLP step clear failed");
  if (hipDeviceSynchronize() != hipSuccess) return fail(PLG_ERR_HIP, "MLP parameter conversion failed");
  return PLG_OK;
}

int plg_mlp_get_params(plg_mlp net, float *host) {
  if (!net || !host) return fail(PLG_ERR_INVALID, "null argument");
  if (hipDeviceSynchronize() != hipSuccess ||
      hipMemcpy(host, net->p, (size_t)net->nparams * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
    return fail(PLG_ERR_HIP, "MLP parameter read-back failed");
  return PLG_OK;
}

int plg_mlp_forward(plg_mlp net, const float *x, int batch, float *y, void *stream) {
  int rc = check_batch(net, batch);
  if (rc) return rc;
  if (!x || !y) return fail(PLG_ERR_INVALID, "null argument");
  hipStream_t st = (hipStream_t)stream;
  const size_t bytes = (size_t)batch * net->dims[net->L] * sizeof(float);
  if (net->rows) {
    // straight into y, unless y overlaps x (blocks write while others read)
    const uintptr_t xa = (uintptr_t)x, ya = (uintptr_t)y;
    if (ya + bytes <= xa || xa + (size_t)batch * net->dims[0] * sizeof(float) <= ya)
      return rows_pass(net, x, nullptr, batch, y, false, st);
    if ((rc = rows_pass(net, x, nullptr, batch, net->Z[net->L - 1], false, st))) return rc;
  } else if ((rc = mlp_forward(net, x, batch, st))) {
    return rc;
  }
  if (hipMemcpyAsync(y, net->Z[net->L - 1], bytes, hipMemcpyDeviceToDevice, st) != hipSuccess)
    return fail(PLG_ERR_HIP, "MLP output copy failed");
  return PLG_OK;
}

int plg_mlp_gradient(plg_mlp net, const float *x, const float *t, int batch, double *loss, float *grad_host,
                     void *stream) {
  int rc = check_batch(net, batch);
  if (rc) return rc;
  if (!x || !t) return fail(PLG_ERR_INVALID, "null argument");
  hipStream_t st = (hipStream_t)stream;
  if (net->rows) {
    if ((rc = rows_pass(net, x, t, batch, net->Z[net->L - 1], false, st)) || (rc = rows_update(net, batch, false, 0, st)) ||
        (loss && (rc = rows_loss(net, t, batch, st))))
      return rc;
  } else if ((rc = mlp_forward(net, x, batch, st)) || (rc = mlp_backward(net, t, batch, st))) {
    return rc;
  }
  if (loss && (rc = mlp_loss(net, batch, st, loss))) return rc;
  if (grad_host) {
    if (hipMemcpyAsync(grad_host, net->g, (size_t)net->nparams * sizeof(float), hipMemcpyDeviceToHost, st) !=
            hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return fail(PLG_ERR_HIP, "MLP gradient read-back failed");
  }
  return PLG_OK;
}

int plg_mlp_train(plg_mlp net, const float *x, const float *t, int batch, int steps, float lr, double *loss,
                  void *stream) {
  int rc = check_batch(net, batch);
  if (rc) return rc;
  if (!x || !t || steps < 0 || !(lr > 0)) return fail(PLG_ERR_INVALID, "plg_mlp_train: bad arguments");
  hipStream_t st = (hipStream_t)stream;
  // Steps are replayed from a graph of one step (captured again when the
  // inputs, batch or rate change) unless PLG_MLP_EAGER=1 or the call is
  // short; both forms launch the same kernels with the same arguments.
  // A two-launch step is launched as it is.
  const char *ev = std::getenv("PLG_MLP_EAGER");
  const bool eager = steps < 4 || (ev && std::atoi(ev) != 0);
  if (net->rows) {
    for (int s = 0; s < steps; s++)
      if ((rc = rows_pass(net, x, t, batch, nullptr, true, st)) || (rc = rows_update(net, batch, true, lr, st))) return rc;
  } else if (eager) {
    for (int s = 0; s < steps; s++)
      if ((rc = train_step(net, x, t, batch, lr, st))) return rc;
  } else {
    if (!net->exec || net->gx != x || net->gt != t || net->gB != batch || net->glr != lr) {
      if (net->exec) hipGraphExecDestroy(net->exec);
      if (net->graph) hipGraphDestroy(net->graph);
      net->exec = nullptr;
      net->graph = nullptr;
      if (!net->cap && hipStreamCreateWithFlags(&net->cap, hipStreamNonBlocking) != hipSuccess)
        return fail(PLG_ERR_HIP, "MLP capture stream creation failed");
      // the capture stream starts after the work queued on `stream`
      hipEvent_t ev0;
      if (hipEventCreateWithFlags(&ev0, hipEventDisableTiming) != hipSuccess) return fail(PLG_ERR_HIP, "event");
      hipEventRecord(ev0, st);
      hipStreamWaitEvent(net->cap, ev0, 0);
      hipEventDestroy(ev0);
      if (hipStreamBeginCapture(net->cap, hipStreamCaptureModeThreadLocal) != hipSuccess)
        return fail(PLG_ERR_HIP, "MLP step capture failed");
      rc = train_step(net, x, t, batch, lr, net->cap);
      hipGraph_t g = nullptr;
      const hipError_t ce = hipStreamEndCapture(net->cap, &g);
      if (rc) {
        if (g) hipGraphDestroy(g);
        return rc;
      }
      if (ce != hipSuccess || !g || hipGraphInstantiate(&net->exec, g, nullptr, nullptr, 0) != hipSuccess) {
        if (g) hipGraphDestroy(g);
        return fail(PLG_ERR_HIP, "MLP step graph instantiation failed");
      }
      net->graph = g;
      net->gx = x;
      net->gt = t;
      net->gB = batch;
      net->glr = lr;
    }
    for (int s = 0; s < steps; s++)
      if (hipGraphLaunch(net->exec, st) != hipSuccess) return fail(PLG_ERR_HIP, "MLP step graph launch failed");
  }
  net->step += steps;
  if (loss) {
    // loss of the parameters after the last update
    if (net->rows) {
      if ((rc = rows_pass(net, x, nullptr, batch, net->Z[net->L - 1], false, st)) || (rc = rows_loss(net, t, batch, st))) return rc;
    } else if ((rc = mlp_forward(net, x, batch, st)) || (rc = mlp_backward(net, t, batch, st))) {
      return rc;
    }
    if ((rc = mlp_loss(net, batch, st, loss))) return rc;
  }
  return PLG_OK;
}

int plg_mlp_destroy(plg_mlp net) {
  if (!net) return PLG_OK;
  hipDeviceSynchronize();
  delete net;
  return PLG_OK;
}

}  // extern "C"
