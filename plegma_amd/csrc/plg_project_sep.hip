// plg_project_sep.hip -- momentum projection as a separable DFT (gfx950).
//
// The projection of a site-correlator column c(x, y, z) on a momentum
// n = (n_x, n_y, n_z) (lib/kernels/PLEGMA_kernel_utils.cuh:820-860, sign -1)
//   F(n) = sum_{x,y,z} exp(-i 2 pi (n_x x / Lx + n_y y / Ly + n_z z / Lz)) c(x, y, z)
// factorises over the directions.  A createMom list (|n|^2 <= Q) has few
// distinct components, so the sums run direction by direction:
//   G[n_x](y, z) = sum_x exp(-i 2 pi n_x x / Lx) c          (per line)
//   H[n_x, n_y](z) = sum_y exp(-i 2 pi n_y y / Ly) G[n_x]   (per plane)
//   F(n) = sum_z exp(-i 2 pi n_z z / Lz) H[n_x, n_y]        (per column)
// For 257 momenta (|n|^2 <= 16) on 32^3 that is about 25 real FMAs per site
// and column instead of 8 x 129 for the paired phase-matrix GEMM, all in FP64
// (the FP32 site correlator is converted exactly), so the pass is bound by
// reading the site correlator from HBM.
//
//  k_sep_xy  workgroup = 16 columns x one z plane.  The plane is staged in
//            chunks of CHL lines (256 FP32 or 128 FP64 sites per column) in
//            LDS; each line is summed by NPART threads (NPART * CHL = 16),
//            each over W = Lx / NPART sites with the phases of its offset
//            i < W read as uniform (scalar) loads, rotated by the part's
//            phase and combined by DPP row exchanges (the line's parts are
//            neighbouring lanes).  The cos and sin sums of
//            a = |n_x| give both n_x = a and n_x = -a.  Thread (column,
//            n_x residue) then accumulates the plane's cos and sin sums over y
//            for every |n_y| class; the (n_x, n_y) pairs the momenta use are
//            written.
//            Where a line is whole groups of 4 sites and the momenta are few,
//            k_sep_xy_mm does the same without the LDS (below).
//  k_sep_z   lane = column, workgroup row = (n_x, n_y) pair: the sums over
//            z of the pair's momenta, written momentum-major for the
//            finalize kernel.
//
// LDS strides: a chunk element (column c, line l, part p, offset i) sits at
// c RS + l LS + p PS + i; PS = 1 and RS = NPART modulo the lanes of one LDS
// pass (16 for 8-byte reads, 8 for 16-byte reads), so the lanes of a pass
// (consecutive parts, then columns) read distinct banks.
#include "plg_internal.h"
#include "plg_tile.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>

namespace plg {

template <typename T> struct SepT;
template <> struct SepT<float> {
  static constexpr int SCH = 256, UPC = 8, EPU = 2, PASS = 16, ELEMS = 5120;
};
template <> struct SepT<double> {
  static constexpr int SCH = 128, UPC = 16, EPU = 1, PASS = 8, ELEMS = 2560;
};
constexpr int SEP_LDS = 40960;  // bytes: SepT<T>::ELEMS elements of cx<T>

template <typename T, int EPU> struct SepVec;
template <> struct SepVec<float, 2> {
  typedef float v __attribute__((ext_vector_type(4)));
};
template <> struct SepVec<double, 1> {
  typedef double v __attribute__((ext_vector_type(2)));
};

// v += the value of the lanes whose index differs in the low log2(N) bits
template <int N> __device__ __forceinline__ void sep_rowsum(double &v) {
  if (N > 1) v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  if (N > 2) v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  if (N > 4) v += dpp<0x141>(v);  // row_half_mirror
  if (N > 8) v += dpp<0x140>(v);  // row_mirror
}

// small tables: three waves per SIMD
template <typename T, int NPART, int MAXA, int MAXB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MAXA <= 5 ? 3 : 1))) void k_sep_xy(SepGeom s, const cx<T> *__restrict__ c,
                                                cx<double> *__restrict__ H) {
  using Q = SepT<T>;
  typedef typename SepVec<T, Q::EPU>::v vec;
  constexpr int CHL = 16 / NPART;                  // lines per chunk
  constexpr int KU = Q::SCH * Q::UPC / 256;        // 16-byte units per thread and chunk
  __shared__ __align__(16) unsigned char lds[SEP_LDS];
  cx<T> *st = (cx<T> *)lds;              // staged chunk
  cx<double> *gb = (cx<double> *)lds;    // line sums G[n_x] of the chunk (after the staged data is used)
  const int tid = threadIdx.x;
  const int64_t col0 = (int64_t)blockIdx.x * 16;
  const int z = blockIdx.y;
  const int Lx = s.Lx, SCHa = CHL * Lx, NU = SCHa * Q::UPC;

  // staging role: the same column and LDS offsets in every chunk
  const int sc = (tid / Q::UPC) & 15;
  const bool col_ok = col0 + sc < s.ncols;
  uint32_t loff[KU];  // LDS offsets (< 2^16) of the unit's elements, 16 bits each
#pragma unroll
  for (int k = 0; k < KU; k++) {
    const int u = tid + 256 * k, tt = u / (16 * Q::UPC), j = u % Q::UPC;
    loff[k] = 0;
#pragma unroll
    for (int e = 0; e < Q::EPU; e++) {
      const int site = tt * 16 + j * Q::EPU + e, l = site / Lx, x = site - l * Lx, p = x / s.W;
      loff[k] |= (uint32_t)(sc * s.RS + l * s.LS + p * s.PS + (x - p * s.W)) << (16 * e);
    }
  }
  // line role: part p1 of line l1 of column c1
  const int p1 = tid % NPART, c1 = (tid / NPART) & 15, l1 = tid / (NPART * 16);
  const int base1 = c1 * s.RS + l1 * s.LS + p1 * s.PS;
  // plane role: column c2, n_x residue slot j2; cos and sin sums over y for
  // the |n_y| classes b
  const int c2 = tid & 15, j2 = tid >> 4;
  const bool role2 = j2 < s.NXR;
  cx<double> hc[MAXB], hs[MAXB];
#pragma unroll
  for (int b = 0; b < MAXB; b++) hc[b] = hs[b] = cmake<double>(0, 0);

  const int64_t tile_plane = (int64_t)z * (Lx * s.Ly) / 16;
  const int nchunk = s.Ly / CHL;
  // the chunk's 16-byte units (loading the next chunk during the sums holds
  // 32 more registers: two waves per SIMD instead of three, measured slower)
  vec v[KU];
  auto fetch = [&](int q) {
    const int64_t tile0 = tile_plane + (int64_t)q * (SCHa / 16);
#pragma unroll
    for (int k = 0; k < KU; k++) {
      const int u = tid + 256 * k, tt = u / (16 * Q::UPC), j = u % Q::UPC;
      if (u < NU && col_ok)
        v[k] = *(const __attribute__((address_space(1))) vec *)(c + (tile0 + tt) * s.gstride +
                                                               (col0 + sc) * s.cstride + j * Q::EPU);
      else
        v[k] = vec{};
    }
  };
  for (int q = 0; q < nchunk; q++) {
    fetch(q);
    __syncthreads();  // the previous chunk's sums (which share the LDS) are read
#pragma unroll
    for (int k = 0; k < KU; k++) {
      const int u = tid + 256 * k;
      if (u < NU) {
#pragma unroll
        for (int e = 0; e < Q::EPU; e++) st[(loff[k] >> (16 * e)) & 0xffff] = cmake<T>(v[k][2 * e], v[k][2 * e + 1]);
      }
    }
    __syncthreads();
    // sums over the part's sites: C_a = sum cos(2 pi a i / Lx) c, S_a likewise
    cx<double> C[MAXA], S[MAXA];
#pragma unroll
    for (int a = 0; a < MAXA; a++) C[a] = S[a] = cmake<double>(0, 0);
#pragma unroll 2
    for (int i = 0; i < s.W; i++) {
      const cx<T> w = st[base1 + i];
      const double wr = (double)w.re, wi = (double)w.im;
#pragma unroll
      for (int a = 0; a < MAXA; a++) {  // (classes a >= NA have zero phases)
        const cx<double> ph = s.ph1[i * MAXA + a];
        C[a].re += ph.re * wr;
        C[a].im += ph.re * wi;
        S[a].re += ph.im * wr;
        S[a].im += ph.im * wi;
      }
    }
    if (NPART > 1) {
#pragma unroll
      for (int a = 0; a < MAXA; a++) {
        // offset p W: cos(t + u) = cos t cos u - sin t sin u, sin(t + u) = sin t cos u + cos t sin u
        const cx<double> pp = s.ph1p[p1 * MAXA + a];
        const cx<double> c0 = C[a], s0 = S[a];
        C[a] = cmake<double>(pp.re * c0.re - pp.im * s0.re, pp.re * c0.im - pp.im * s0.im);
        S[a] = cmake<double>(pp.im * c0.re + pp.re * s0.re, pp.im * c0.im + pp.re * s0.im);
      }
      // sums over the line's NPART lanes (the low lane bits): quad
      // exchanges, then the other quad, then the other half row
#pragma unroll
      for (int a = 0; a < MAXA; a++) {
        sep_rowsum<NPART>(C[a].re);
        sep_rowsum<NPART>(C[a].im);
        sep_rowsum<NPART>(S[a].re);
        sep_rowsum<NPART>(S[a].im);
      }
    }
    __syncthreads();  // every thread has read its staged sites
    // G[n_x] of the line: a = n_x gives C - i S, a = -n_x (mod Lx) gives C + i S
#pragma unroll
    for (int a = 0; a < MAXA; a++)
      if (a % NPART == p1) {
        const int sp = s.xs[2 * a], sm = s.xs[2 * a + 1];
        if (sp >= 0) gb[(l1 * s.NXR + sp) * 16 + c1] = cmake<double>(C[a].re + S[a].im, C[a].im - S[a].re);
        if (sm >= 0) gb[(l1 * s.NXR + sm) * 16 + c1] = cmake<double>(C[a].re - S[a].im, C[a].im + S[a].re);
      }
    __syncthreads();
    if (role2) {
#pragma unroll 2
      for (int l = 0; l < CHL; l++) {
        const int y = q * CHL + l;
        const cx<double> g = gb[(l * s.NXR + j2) * 16 + c2];
#pragma unroll
        for (int b = 0; b < MAXB; b++) {  // (classes b >= NB have zero phases)
          const cx<double> ph = s.ph2[y * MAXB + b];
          hc[b].re += ph.re * g.re;
          hc[b].im += ph.re * g.im;
          hs[b].re += ph.im * g.re;
          hs[b].im += ph.im * g.im;
        }
      }
    }
  }
  if (role2 && col0 + c2 < s.ncols) {
    // n_y = b: C - i S; n_y = -b (mod Ly): C + i S
#pragma unroll
    for (int b = 0; b < MAXB; b++) {
      const int sp = s.slot[(j2 * MAXB + b) * 2], sm = s.slot[(j2 * MAXB + b) * 2 + 1];
      if (sp >= 0)
        gstore(H + ((int64_t)z * s.NS + sp) * s.ncols + col0 + c2,
               cmake<double>(hc[b].re + hs[b].im, hc[b].im - hs[b].re));
      if (sm >= 0)
        gstore(H + ((int64_t)z * s.NS + sm) * s.ncols + col0 + c2,
               cmake<double>(hc[b].re - hs[b].im, hc[b].im + hs[b].re));
    }
  }
}

// The sums over x and y with the x sums on the matrix cores, where a line is
// whole groups of 4 sites and the tables are small.  A wave owns 16 columns
// and every fourth line of a plane.  A line's sums with the NF cosines and
// sines of the |n_x| classes are 16x16x4 FP64 matrix products, A the functions
// at four sites, B those sites of the 16 columns as the lanes load them (lane
// n + 16 k: column n, sites k EPU ...), so nothing goes through LDS and no
// barrier stands between the loads, which run SEP_PF units ahead.  Row 4 r +
// lane / 16 of the product is in register r: each lane then adds its three
// functions times the NG cosines and sines of the line's y to the plane's
// sums.  The waves' sums meet in LDS, and the (n_x, n_y) pairs are combined
// from them.
// Bound by HBM and, nearly as much, by FP64: 16 columns x 32 sites of a line
// are 4 KB (FP32) of HBM, 16 matrix instructions of 67 cycles and 54 FMAs of a
// SIMD.  A field of 1024 columns on 32^3, 257 momenta, FP32: 98 -> 75 us against
// k_sep_xy's staged lines (55 us with the sums left out); 16
// sources' two-point functions 2.23 -> 1.91 ms.  Three waves per SIMD: two,
// with more loads ahead, 2.2 ms.
constexpr int SEP_PF = 4;
typedef double sep_v4 __attribute__((ext_vector_type(4)));
template <typename T, int EPU> struct SepLoad {
  typedef T v __attribute__((ext_vector_type(2 * EPU)));
};

// RF registers of functions of x (NF <= 4 RF), NG functions of y
template <typename T, int EPU, int RF, int NG>
__global__ __launch_bounds__(256, 3) void k_sep_xy_mm(SepGeom s, const cx<T> *__restrict__ c,
                                                       cx<double> *__restrict__ H) {
  typedef typename SepLoad<T, EPU>::v vec;
  extern __shared__ __align__(16) unsigned char lds_mm[];
  double *pha = (double *)lds_mm;                       // [Lx / 4][64]
  cx<double> *Q = (cx<double> *)(pha + 16 * s.Lx);      // [4 RF][NG][16 columns]
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, k = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t col0 = (int64_t)blockIdx.x * 16;
  const int z = blockIdx.y;
  for (int i = tid; i < 16 * s.Lx; i += 256) pha[i] = s.pha[i];
  __syncthreads();
  // columns past the end repeat the last one and are not stored
  const int64_t col = col0 + n < s.ncols ? col0 + n : s.ncols - 1;
  const cx<T> *cb = c + col * s.cstride + k * EPU;
  const int U = s.Lx / (4 * EPU);  // units of a line: EPU sites of each lane
  const int nl = wave < s.Ly ? (s.Ly - wave + 3) / 4 : 0, NU = nl * U;
  cx<double> acc[RF][NG];
#pragma unroll
  for (int r = 0; r < RF; r++)
#pragma unroll
    for (int j = 0; j < NG; j++) acc[r][j] = cmake<double>(0, 0);
  if (NU > 0) {
    int py = wave, pg = 0, pleft = NU - 1;  // the unit to load next (the last one again at the end)
    auto fetch = [&]() {
      const int64_t site = ((int64_t)z * s.Ly + py) * s.Lx + pg * (4 * EPU);
      const vec v = *(const __attribute__((address_space(1))) vec *)(cb + (site >> 4) * s.gstride + (site & 15));
      if (pleft > 0) {
        pleft--;
        if (++pg == U) {
          pg = 0;
          py += 4;
        }
      }
      return v;
    };
    vec cur[SEP_PF];
#pragma unroll
    for (int u = 0; u < SEP_PF; u++) cur[u] = fetch();
    sep_v4 Dr = (sep_v4)0.0, Di = (sep_v4)0.0;
    int y = wave, g = 0;
    double ph[NG];  // the line's phases, loaded a line ahead
#pragma unroll
    for (int j = 0; j < NG; j++) ph[j] = s.ph2f[y * NG + j];
    for (int u0 = 0; u0 < NU; u0 += SEP_PF) {
      vec next[SEP_PF];
#pragma unroll
      for (int u = 0; u < SEP_PF; u++) next[u] = fetch();
#pragma unroll
      for (int u = 0; u < SEP_PF; u++) {
        if (u0 + u < NU) {
#pragma unroll
          for (int e = 0; e < EPU; e++) {
            const double a = pha[(g * EPU + e) * 64 + lane];
            Dr = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)cur[u][2 * e], Dr, 0, 0, 0);
            Di = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)cur[u][2 * e + 1], Di, 0, 0, 0);
          }
          if (++g == U) {  // the line is whole
            y += 4;
            const int yn = min(y, s.Ly - 1);
#pragma unroll
            for (int j = 0; j < NG; j++) {
              const double p = ph[j];
              ph[j] = s.ph2f[yn * NG + j];
#pragma unroll
              for (int r = 0; r < RF; r++) {
                acc[r][j].re = fma(p, Dr[r], acc[r][j].re);
                acc[r][j].im = fma(p, Di[r], acc[r][j].im);
              }
            }
            Dr = Di = (sep_v4)0.0;
            g = 0;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < SEP_PF; u++) cur[u] = next[u];
    }
  }
  for (int w = 0; w < 4; w++) {
    if (wave == w) {
#pragma unroll
      for (int r = 0; r < RF; r++)
#pragma unroll
        for (int j = 0; j < NG; j++) {
          cx<double> *d = Q + ((4 * r + k) * NG + j) * 16 + n;
          *d = w == 0 ? acc[r][j] : *d + acc[r][j];
        }
    }
    __syncthreads();
  }
  // exp(-i sx a x) exp(-i sy b y) = (C_a - i sx S_a)(C_b - i sy S_b)
  if (col0 + n < s.ncols)
    for (int sl = tid >> 4; sl < s.NS; sl += 16) {
      const int *e = s.slq + sl * 6;
      const int fc = e[0], fs = e[1], gc = e[3], gs = e[4];
      const double sx = e[2], sy = e[5];
      auto at = [&](int f, int j) { return f < 0 || j < 0 ? cmake<double>(0, 0) : Q[(f * NG + j) * 16 + n]; };
      const cx<double> cc = at(fc, gc), ss = at(fs, gs), sc = at(fs, gc), cs = at(fc, gs);
      gstore(H + ((int64_t)z * s.NS + sl) * s.ncols + col0 + n,
             cmake<double>(cc.re - sx * sy * ss.re + sx * sc.im + sy * cs.im,
                           cc.im - sx * sy * ss.im - sx * sc.re - sy * cs.re));
    }
}

// A workgroup holds 64 columns, its four waves every fourth plane each: with
// a thread per column and all its planes a call of 1024 columns had 784 waves
// on the chip, each a serial chain of loads: 15 -> 9 us.
template <int MAXZ>
__global__ __launch_bounds__(256) void k_sep_z(SepGeom s, const cx<double> *__restrict__ H,
                                               cx<double> *__restrict__ part) {
  __shared__ cx<double> sum[MAXZ][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t col = (int64_t)blockIdx.x * 64 + lane;
  const int sl = blockIdx.y;
  const bool in = col < s.ncols;
  const cx<double> *Hc = H + (int64_t)sl * s.ncols + (in ? col : s.ncols - 1);
  // the pair's momenta, padded to MAXZ (padding: n_z residue 0, momentum -1)
  const int *rz = s.sl_rz + sl * MAXZ, *mm = s.sl_m + sl * MAXZ;
  cx<double> acc[MAXZ];
#pragma unroll
  for (int j = 0; j < MAXZ; j++) acc[j] = cmake<double>(0, 0);
#pragma unroll 2
  for (int z = wave; z < s.Lz; z += 4) {
    const cx<double> h = gload(Hc + (int64_t)z * s.NS * s.ncols);
#pragma unroll
    for (int j = 0; j < MAXZ; j++) {  // (cos - i sin) h
      const cx<double> ph = s.ph3[rz[j] * s.Lz + z];
      acc[j].re += ph.re * h.re;
      acc[j].re += ph.im * h.im;
      acc[j].im += ph.re * h.im;
      acc[j].im -= ph.im * h.re;
    }
  }
  for (int w = 3; w > 0; w--) {
    if (wave == w)
#pragma unroll
      for (int j = 0; j < MAXZ; j++) sum[j][lane] = w == 3 ? acc[j] : sum[j][lane] + acc[j];
    __syncthreads();
  }
  if (wave == 0 && in)
#pragma unroll
    for (int j = 0; j < MAXZ; j++)
      if (mm[j] >= 0) gstore(part + (int64_t)mm[j] * s.ncols + col, acc[j] + sum[j][lane]);
}

// ------------------------------------------------------------------ host
// sites of a lane's load in the matrix form: 16 bytes where a line is whole
// groups of the lanes' sites
static int sep_epu(int Lx, bool f64) { return !f64 && Lx % 8 == 0 ? 2 : 1; }
// functions of y the matrix form's kernels are built for: components up to 2, 3 and 4
static int sep_ng(int nf, int ng) { return nf > 8 ? 9 : ng <= 5 ? 5 : ng <= 7 ? 7 : 9; }

void sep_build(const int L[3], int M, const std::vector<int> &ms, int64_t ncols, bool f64, SepHost &h) {
  h = SepHost{};
  const int nmom = (int)ms.size() / 3;
  const int Lx = L[0], Ly = L[1], Lz = L[2];
  if (nmom <= 0 || (Lx * Ly) % 16 || ncols <= 0) return;
  const int SCH = f64 ? SepT<double>::SCH : SepT<float>::SCH;
  const int PASS = f64 ? SepT<double>::PASS : SepT<float>::PASS;
  const int ELEMS = f64 ? SepT<double>::ELEMS : SepT<float>::ELEMS;
  // residues of the components (ms holds n_k (M / L_k) mod M)
  std::vector<int> rx(nmom), ry(nmom), rz(nmom);
  for (int m = 0; m < nmom; m++) {
    rx[m] = ms[3 * m] / (M / Lx);
    ry[m] = ms[3 * m + 1] / (M / Ly);
    rz[m] = ms[3 * m + 2] / (M / Lz);
  }
  std::map<int, int> amap, rxmap, rymap, bmap;
  for (int m = 0; m < nmom; m++) {
    amap[std::min(rx[m], Lx - rx[m])] = 0;
    rxmap[rx[m]] = 0;
    rymap[ry[m]] = 0;
    bmap[std::min(ry[m], Ly - ry[m])] = 0;
  }
  int k = 0;
  for (auto &e : amap) e.second = k++;
  k = 0;
  for (auto &e : rxmap) e.second = k++;
  k = 0;
  for (auto &e : rymap) e.second = k++;
  k = 0;
  for (auto &e : bmap) e.second = k++;
  SepGeom &g = h.g;
  g.Lx = Lx;
  g.Ly = Ly;
  g.Lz = Lz;
  g.ncols = ncols;
  g.nmom = nmom;
  g.NA = (int)amap.size();
  g.NXR = (int)rxmap.size();
  g.NYR = (int)rymap.size();
  g.NB = (int)bmap.size();
  if (g.NA > 8 || g.NXR > 16 || g.NB > 8) return;
  // chunk: CHL lines (a power of two dividing Ly and 16), whole tiles, the
  // most lines whose staged sites and line sums fit the LDS
  auto fits = [&](int cl) {
    if (Ly % cl || cl * Lx > SCH || (cl * Lx) % 16 || Lx % (16 / cl)) return false;
    g.NPART = 16 / cl;
    g.W = Lx / g.NPART;
    g.PS = g.W + (((1 - g.W) % PASS) + PASS) % PASS;  // PS = 1 mod PASS
    g.LS = g.NPART * g.PS;
    g.RS = cl * g.LS;
    if (g.NPART < PASS)
      while (g.RS % PASS != g.NPART % PASS) g.RS++;
    return 16 * g.RS <= ELEMS && cl * g.NXR * 16 * (int)sizeof(cx<double>) <= SEP_LDS;
  };
  int CHL = 0;
  for (int cl = 16; cl >= 1 && !CHL; cl >>= 1)
    if (fits(cl)) CHL = cl;
  if (!CHL) return;
  // (n_x, n_y) pairs and their momenta
  std::map<std::pair<int, int>, std::vector<int>> pairs;
  for (int m = 0; m < nmom; m++) pairs[{rxmap[rx[m]], rymap[ry[m]]}].push_back(m);
  g.NS = (int)pairs.size();
  int maxcnt = 0;
  for (auto &e : pairs) maxcnt = std::max(maxcnt, (int)e.second.size());
  if (maxcnt > 16) return;
  g.small = g.NA <= 5 && g.NB <= 5 && maxcnt <= 9;
  // the matrix form: functions cos a, sin a (unless the sine vanishes at every site)
  std::map<int, std::pair<int, int>> fx, fy;
  auto functions = [](const std::map<int, int> &cls, int L, std::map<int, std::pair<int, int>> &f) {
    int n = 0;
    for (auto &e : cls) {
      const bool odd = e.first != 0 && 2 * e.first != L;
      f[e.first] = {n, odd ? n + 1 : -1};
      n += odd ? 2 : 1;
    }
    return n;
  };
  g.NF = functions(amap, Lx, fx);
  g.NG = functions(bmap, Ly, fy);
  g.mm = g.small && Lx % 4 == 0 && g.NF <= 12 && g.NG <= 9;
  // tables padded to the kernel's class and momentum counts
  const int NAP = g.small ? 5 : 8, NBP = g.small ? 5 : 8, NZP = g.small ? 9 : 16;
  std::vector<int> ryres(g.NYR);
  for (auto &e : rymap) ryres[e.second] = e.first;
  std::vector<int> slot, xs, slq, slm(g.NS * NZP, -1), slrz(g.NS * NZP, 0);
  {
    int sidx = 0;
    for (auto &e : pairs) {
      for (size_t j = 0; j < e.second.size(); j++) {
        slm[sidx * NZP + j] = e.second[j];
        slrz[sidx * NZP + j] = rz[e.second[j]];
      }
      sidx++;
    }
  }
  // phases from exact integer residues
  auto phase = [](int64_t num, int den) {
    const double t = 2.0 * M_PI * (double)(num % den) / (double)den;
    return std::make_pair(std::cos(t), std::sin(t));
  };
  std::vector<double> ph1, ph1p, ph2, pha, ph2f, ph3;
  if (!g.mm) {  // the staged form's tables
    slot.assign(g.NXR * NBP * 2, -1);
    int sidx = 0;
    for (auto &e : pairs) {
      // the pair's n_y residue as class b, sign + (r = b) or - (r = Ly - b != b)
      const int r = ryres[e.first.second], b = std::min(r, Ly - r);
      slot[(e.first.first * NBP + bmap[b]) * 2 + (r == b ? 0 : 1)] = sidx++;
    }
    // residue slots of +a and -a
    xs.assign(2 * NAP, -1);
    for (auto &e : amap) {
      const int a = e.first;
      auto ip = rxmap.find(a);
      if (ip != rxmap.end()) xs[2 * e.second] = ip->second;
      auto im = rxmap.find((Lx - a) % Lx);
      if (a != 0 && 2 * a != Lx && im != rxmap.end()) xs[2 * e.second + 1] = im->second;
    }
    ph1.assign(2 * g.W * NAP, 0.0);
    ph1p.assign(2 * g.NPART * NAP, 0.0);
    ph2.assign(2 * Ly * NBP, 0.0);
    for (auto &e : amap)
      for (int i = 0; i < g.W; i++) {
        auto cs = phase((int64_t)e.first * i, Lx);
        ph1[2 * (i * NAP + e.second)] = cs.first;
        ph1[2 * (i * NAP + e.second) + 1] = cs.second;
      }
    for (auto &e : amap)
      for (int p = 0; p < g.NPART; p++) {
        auto cs = phase((int64_t)e.first * p * g.W, Lx);
        ph1p[2 * (p * NAP + e.second)] = cs.first;
        ph1p[2 * (p * NAP + e.second) + 1] = cs.second;
      }
    for (auto &e : bmap)
      for (int y = 0; y < Ly; y++) {
        auto cs = phase((int64_t)e.first * y, Ly);
        ph2[2 * (y * NBP + e.second)] = cs.first;
        ph2[2 * (y * NBP + e.second) + 1] = cs.second;
      }
  }
  for (int r = 0; r < Lz; r++)
    for (int z = 0; z < Lz; z++) {
      auto cs = phase((int64_t)r * z, Lz);
      ph3.push_back(cs.first);
      ph3.push_back(cs.second);
    }
  if (g.mm) {
    const int NGP = sep_ng(g.NF, g.NG);
    const int EP = sep_epu(Lx, f64);
    pha.assign((size_t)Lx * 16, 0.0);
    for (int st = 0; st < Lx / 4; st++)
      for (int k = 0; k < 4; k++) {
        const int x = st / EP * (4 * EP) + k * EP + st % EP;
        for (auto &e : fx) {
          auto cs = phase((int64_t)e.first * x, Lx);
          pha[st * 64 + 16 * k + e.second.first] = cs.first;
          if (e.second.second >= 0) pha[st * 64 + 16 * k + e.second.second] = cs.second;
        }
      }
    ph2f.assign((size_t)Ly * NGP, 0.0);
    for (int y = 0; y < Ly; y++)
      for (auto &e : fy) {
        auto cs = phase((int64_t)e.first * y, Ly);
        ph2f[y * NGP + e.second.first] = cs.first;
        if (e.second.second >= 0) ph2f[y * NGP + e.second.second] = cs.second;
      }
    std::vector<int> rxres(g.NXR);
    for (auto &e : rxmap) rxres[e.second] = e.first;
    for (auto &e : pairs) {
      const int rx_ = rxres[e.first.first], ry_ = ryres[e.first.second];
      const int a = std::min(rx_, Lx - rx_), b = std::min(ry_, Ly - ry_);
      slq.insert(slq.end(), {fx[a].first, fx[a].second, rx_ == a ? 1 : -1, fy[b].first, fy[b].second, ry_ == b ? 1 : -1});
    }
  }
  // one blob, 256-byte aligned pieces
  auto put = [&](const void *src, size_t bytes) {
    const size_t off = (h.blob.size() + 255) / 256 * 256;
    h.blob.resize(off + std::max<size_t>(bytes, 1));
    if (bytes) std::memcpy(h.blob.data() + off, src, bytes);
    return off;
  };
  h.off_pha = put(pha.data(), pha.size() * sizeof(double));
  h.off_ph2f = put(ph2f.data(), ph2f.size() * sizeof(double));
  h.off_slq = put(slq.data(), slq.size() * sizeof(int));
  h.off_ph1 = put(ph1.data(), ph1.size() * sizeof(double));
  h.off_ph1p = put(ph1p.data(), ph1p.size() * sizeof(double));
  h.off_ph2 = put(ph2.data(), ph2.size() * sizeof(double));
  h.off_ph3 = put(ph3.data(), ph3.size() * sizeof(double));
  h.off_xs = put(xs.data(), xs.size() * sizeof(int));
  h.off_slot = put(slot.data(), slot.size() * sizeof(int));
  h.off_slm = put(slm.data(), slm.size() * sizeof(int));
  h.off_slrz = put(slrz.data(), slrz.size() * sizeof(int));
  h.ok = true;
}

SepGeom sep_geom(const SepHost &h, const void *d_blob) {
  SepGeom g = h.g;
  g.gstride = 16 * g.ncols;  // the tile-major site correlator
  g.cstride = 16;
  const unsigned char *b = (const unsigned char *)d_blob;
  g.pha = (const double *)(b + h.off_pha);
  g.ph2f = (const double *)(b + h.off_ph2f);
  g.slq = (const int *)(b + h.off_slq);
  g.ph1 = (const cx<double> *)(b + h.off_ph1);
  g.ph1p = (const cx<double> *)(b + h.off_ph1p);
  g.ph2 = (const cx<double> *)(b + h.off_ph2);
  g.ph3 = (const cx<double> *)(b + h.off_ph3);
  g.xs = (const int *)(b + h.off_xs);
  g.slot = (const int *)(b + h.off_slot);
  g.sl_m = (const int *)(b + h.off_slm);
  g.sl_rz = (const int *)(b + h.off_slrz);
  return g;
}

template <typename T, int MAXA, int MAXB>
static int launch_xy(const SepGeom &g, const cx<T> *c, cx<double> *H, hipStream_t st) {
  dim3 block(256), grid((unsigned)((g.ncols + 15) / 16), (unsigned)g.Lz);
  switch (g.NPART) {
  case 1: k_sep_xy<T, 1, MAXA, MAXB><<<grid, block, 0, st>>>(g, c, H); break;
  case 2: k_sep_xy<T, 2, MAXA, MAXB><<<grid, block, 0, st>>>(g, c, H); break;
  case 4: k_sep_xy<T, 4, MAXA, MAXB><<<grid, block, 0, st>>>(g, c, H); break;
  case 8: k_sep_xy<T, 8, MAXA, MAXB><<<grid, block, 0, st>>>(g, c, H); break;
  case 16: k_sep_xy<T, 16, MAXA, MAXB><<<grid, block, 0, st>>>(g, c, H); break;
  default: return PLG_ERR_UNSUPPORTED;
  }
  return PLG_OK;
}

template <typename T, int EPU>
static void launch_xy_mm(const SepGeom &g, const cx<T> *c, cx<double> *H, hipStream_t st) {
  dim3 block(256), grid((unsigned)((g.ncols + 15) / 16), (unsigned)g.Lz);
  const int ng = sep_ng(g.NF, g.NG);
  auto lds = [&](int RF, int NG) { return (size_t)g.Lx * 16 * sizeof(double) + 4 * RF * NG * 16 * sizeof(cx<double>); };
  if (ng == 5) k_sep_xy_mm<T, EPU, 2, 5><<<grid, block, lds(2, 5), st>>>(g, c, H);
  else if (ng == 7) k_sep_xy_mm<T, EPU, 2, 7><<<grid, block, lds(2, 7), st>>>(g, c, H);
  else k_sep_xy_mm<T, EPU, 3, 9><<<grid, block, lds(3, 9), st>>>(g, c, H);
}

int launch_project_sep(const SepGeom &g, const void *c, int c_prec, double *part, hipStream_t st) {
  cx<double> *P = (cx<double> *)part;
  cx<double> *H = P + (int64_t)g.nmom * g.ncols;
  int rc = PLG_OK;
  if (g.mm) {
    if (c_prec == PLG_F64) launch_xy_mm<double, 1>(g, (const cx<double> *)c, H, st);
    else if (sep_epu(g.Lx, false) == 2) launch_xy_mm<float, 2>(g, (const cx<float> *)c, H, st);
    else launch_xy_mm<float, 1>(g, (const cx<float> *)c, H, st);
  } else if (c_prec == PLG_F64)
    rc = g.small ? launch_xy<double, 5, 5>(g, (const cx<double> *)c, H, st)
                 : launch_xy<double, 8, 8>(g, (const cx<double> *)c, H, st);
  else
    rc = g.small ? launch_xy<float, 5, 5>(g, (const cx<float> *)c, H, st)
                 : launch_xy<float, 8, 8>(g, (const cx<float> *)c, H, st);
  if (rc) return rc;
  dim3 block(256), grid((unsigned)((g.ncols + 63) / 64), (unsigned)g.NS);
  if (g.small) k_sep_z<9><<<grid, block, 0, st>>>(g, H, P);
  else k_sep_z<16><<<grid, block, 0, st>>>(g, H, P);
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

}  // namespace plg
