// plg_mesmes.hip -- heavy-light mesons and the four-propagator meson-meson
// (tetraquark-like) contraction on gfx950.
//
// Counterpart of lib/kernels/PLEGMA_heavy_light_tetraquarks.cu:5-61,163-212
// (a table-driven sum over spin/colour entries of S1 S2 conj(S3) conj(S4)),
// in the factorised form of two colour-traced meson blocks plus the crossed
// term.  On 12x12 spin-colour matrices, with X = g5 G (a signed permutation):
//   A_G = G S_L X S_H^dag g5 = G M_G G^-1,   M_G = S_L X S_H^dag X
//   meson(G)  = Tr M_G                          (16 GAMMAS, enum order)
//   mesmes(G) = (Tr M_G)^2 - Tr[M_G M_G]        (G = g5, g1, g2, g3)
// with the colour blocks (x the xor class of X, phi its row phases)
//   M'^{ab}_{mu nu} = sum_rho phi(rho) sum_c S_L^{ac}_{mu rho} conj(S_H^{bc}_{nu^x rho^x})
//   M = M' phi(nu^x),   meson(G) = sum_{a b} phi(a^x) phi(b) S_L[a][b] . conj(S_H[a^x][b^x])
// g5/g3 share X's class 0 and g1/g2 class 1; within a class the row phases
// differ by +-i^RA, so one pass over rho fills both operators (the sums x, y
// over the two kinds of rows; the operators are x + y and i^RA (x - y)).
//
// Work split: four lanes per site, 16 sites per wave, lane j = nu and
// mu = j ^ s.  The block and its transposed partner M_{nu mu} then sit at the
// same s in lanes j and j ^ s, an exchange within the quad, and the phases of
// Tr[M M] are compile-time signs, phi(j^x) phi(j^s^x) = phi(0) phi(s) (phi is a
// sign character of the spin index up to its entry 0).  Four waves share the
// staged sites of both propagators: wave (x, h) takes the class x, the s of
// half h, and the mesons of class 2 h + x, whose operands it reads anyway for
// h = 0.  The halves' sums meet in LDS.
//
// What bounds it: the workgroups' alternation of staging (2 304 bytes a site;
// alone 5.4 ms of the figure below) and vector instructions (4 600 wave FMAs a
// tile; alone 4.4 ms), four 4-wave workgroups a CU (38 KB of LDS, 128
// registers) overlapping each other.  Prefetching the next tile into
// registers (spills, or two waves per SIMD), eight waves of one s each, tiles
// of 32 sites and other tile orders over the XCDs measured slower or equal.
// 8.4 M sites (64^3 x 32 slices) in FP32: sixteen lanes per site, two waves
// per SIMD and one LDS read per three FMAs took 7.9 ms, this form 6.1 ms
// (3.4 TB/s; reading the propagators alone would take 4 ms).
#include "plg_tile.h"

namespace plg {

// entry (mu, nu, colour pair cc) of site t at cc 256 + nu 64 + mu 16 +
// (t ^ MM_SW mu): the lanes of an LDS pass (the four mu of four sites) read
// distinct banks
constexpr int MM_TILE = 144 * 16, MM_SW = 4, MM_THREADS = 256;

template <typename T> struct MmShared {
  cx<T> t1[MM_TILE], t2[MM_TILE];
  // per site: Tr M of g3, g5 (class 0), g1, g2 (class 1), then the two halves'
  // crossed sums of (g5, g3) and (g1, g2)
  cx<T> x[16][13];
};

// class X, half H (see above): crossed sums of OPA, OPB over s = 2 H, 2 H + 1
// (every lane of the site), and the four mesons of class 2 H + X (lane n the
// n-th)
template <typename T, int X, int H>
__device__ __forceinline__ void mm_wave(const cx<T> *SL, const cx<T> *SH, int site, int j, cx<T> (&cross)[2], cx<T> &mes) {
  constexpr int OPA = X == 0 ? 5 : 1, OPB = X == 0 ? 3 : 2, d = 2 * H + X;
  constexpr SPerm XA = sp_mul(G_5, gamma_op(OPA)), XB = sp_mul(G_5, gamma_op(OPB));
  static_assert(sp_class(XA) == X && sp_class(XB) == X && char_ok(XA.ph) && char_ok(XB.ph), "class and sign characters");
  constexpr int RA = (XB.ph[0] - XA.ph[0]) & 3;
  auto col = [&](const cx<T> *S, int mu) { return S + mu * 16 + (site ^ (MM_SW * mu)); };
  const cx<T> *l0 = col(SL, j ^ (2 * H)), *l1 = col(SL, j ^ (2 * H + 1)), *hh = col(SH, j ^ X);
  cx<T> U[2][2][9];  // [kind][s][ab]
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 9; i++) U[k][s][i] = cmake<T>(0, 0);
  cx<T> w[4];
#pragma unroll
  for (int n = 0; n < 4; n++) w[n] = cmake<T>(0, 0);
  static_for<0, 4>([&](auto rho_) {
    constexpr int rho = rho_.value, kind = (XB.ph[rho] - XA.ph[rho] - RA) & 3;
    static_assert(kind == 0 || kind == 2, "row phases of a class pair differ by +-i^RA");
    cx<T> b[9];
#pragma unroll
    for (int i = 0; i < 9; i++) b[i] = hh[(rho ^ X) * 64 + i * 256];
    cx<T> g = cmake<T>(0, 0);  // G_d[j ^ 2H][rho] of the mesons
    static_for<0, 3>([&](auto ca) {
      static_for<0, 2>([&](auto s_) {
        const cx<T> *l = s_.value == 0 ? l0 : l1;
        cx<T> a[3];
#pragma unroll
        for (int i = 0; i < 3; i++) a[i] = l[rho * 64 + (ca.value * 3 + i) * 256];
        if constexpr (s_.value == 0) {
#pragma unroll
          for (int i = 0; i < 3; i++)
            cfma_conj(g, a[i], H == 0 ? b[ca.value * 3 + i] : hh[(rho ^ d) * 64 + (ca.value * 3 + i) * 256]);
        }
        static_for<0, 3>([&](auto cc) {
          static_for<0, 3>([&](auto cb) {
            cfma_conj_iph<XA.ph[rho]>(U[kind / 2][s_.value][ca.value * 3 + cb.value], a[cc.value], b[cb.value * 3 + cc.value]);
          });
        });
      });
      // (without it the scheduler hoists the next operands' reads and spills)
      __builtin_amdgcn_sched_barrier(0);
    });
    static_for<0, 4>([&](auto n) { w[n.value] = w[n.value] + cmul_iph(g, MESON_X.ph[meson_op(d, n.value)][rho]); });
  });
  cx<T> sa = cmake<T>(0, 0), sb = cmake<T>(0, 0);
  static_for<0, 2>([&](auto s_) {
    constexpr int s = 2 * H + s_.value;
    constexpr int pha = (XA.ph[0] + XA.ph[s]) & 3, phb = (XB.ph[0] + XB.ph[s] + 2 * RA) & 3;
    cx<T> A[9], B[9];
#pragma unroll
    for (int i = 0; i < 9; i++) {
      A[i] = U[0][s_.value][i] + U[1][s_.value][i];
      B[i] = U[0][s_.value][i] - U[1][s_.value][i];
    }
    // sum_ab M'^{ab}_{mu nu} M'^{ba}_{nu mu}, the partner block from lane j ^ s
#pragma unroll
    for (int ca = 0; ca < 3; ca++)
#pragma unroll
      for (int cb = 0; cb < 3; cb++) {
        const cx<T> ta = A[cb * 3 + ca], tb = B[cb * 3 + ca];
        cfma_iph<pha>(sa, A[ca * 3 + cb], cmake<T>(quad_xor<s>(ta.re), quad_xor<s>(ta.im)));
        cfma_iph<phb>(sb, B[ca * 3 + cb], cmake<T>(quad_xor<s>(tb.re), quad_xor<s>(tb.im)));
      }
  });
  cross[0] = cmake<T>(quad_sum(sa.re), quad_sum(sa.im));
  cross[1] = cmake<T>(quad_sum(sb.re), quad_sum(sb.im));
  static_for<0, 4>([&](auto n) {
    constexpr int op = meson_op(d, n.value);
    static_assert(op >= 0 && char_ok(MESON_X.ph[op < 0 ? 0 : op]), "four channels per class, sign characters");
    // lane j holds row a = j ^ 2H, phase phi(a^d) = phi(j^X) = phi(X) sigma(j)
    w[n.value] = char_sign<T>(MESON_X.ph[op], j) * cmul_iph(w[n.value], MESON_X.ph[op][X]);
  });
  mes = quad_scatter_sum(w, j);
}

// rotation of a staged tile to the physical basis in place (thr of nthr threads)
template <typename T> __device__ __forceinline__ void mm_rotate(cx<T> *S, int sign, int thr, int nthr) {
  for (int it = thr; it < 16 * 36; it += nthr) {
    const int t = it & 15, cq = it >> 4, cp = cq % 9, q = cq / 9, m = q >> 1, n = q & 1;
    auto at = [&](int mu, int nu) -> cx<T> & { return S[cp * 256 + nu * 64 + mu * 16 + (t ^ (MM_SW * mu))]; };
    cx<T> a = at(m, n), b = at(m, n + 2), c = at(m + 2, n), d = at(m + 2, n + 2);
    rot_physical(a, b, c, d, sign);
    at(m, n) = a;
    at(m, n + 2) = b;
    at(m + 2, n) = c;
    at(m + 2, n + 2) = d;
  }
}

// Output channels per row (from ch0): 16 mesons Tr[G S_L g5 G S_H^dag g5]
// (GAMMAS order), then mesmes for G = g5, g1, g2, g3.
template <typename T>
__global__ __launch_bounds__(MM_THREADS) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2)))
void k_mesmes(const PropDev<T> *__restrict__ props, const RowDev *__restrict__ rows, cx<T> *__restrict__ out,
              int64_t V3, int T_lat, int nch_total, int ch0, int ntiles) {
  // staging: 128 threads per propagator, 16-byte units; thread group g takes
  // the spin pairs mu = g % 4, nu = g / 4 (+ 2 in FP64), nine colour pairs each
  constexpr int EPU = 16 / (int)sizeof(cx<T>), UPC = 16 / EPU, NH = UPC / 8;
  typedef typename SiteVec<T, EPU>::v vec;
  typedef T av __attribute__((ext_vector_type(2 * EPU)));
  __shared__ __align__(16) MmShared<T> sh;
  const RowDev row = rows[blockIdx.y];
  const PropDev<T> P1 = props[row.pa], P2 = props[row.pb];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), f = wave >> 1;
  const PropDev<T> PF = f == 0 ? P1 : P2;
  const int thr = threadIdx.x & 127, g = thr / UPC, e0 = (thr % UPC) * EPU, gm = g & 3, gn = g >> 2;
  const cx<T> *src = PF.data + (int64_t)((row.t - PF.t_first + T_lat) % T_lat) * V3 + (int64_t)((gm * 4 + gn) * 9) * PF.cs + e0;
  // the mesons are bilinear in the propagators (the boundary signs of the
  // meson-meson channels cancel)
  const T sg = prop_sign(P1, row.t) * prop_sign(P2, row.t);
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total + ch0;
  for (int tl = blockIdx.x; tl < ntiles; tl += gridDim.x) {
    const int64_t x0 = (int64_t)tl * 16;
    int tid = threadIdx.x;  // opaque: what derives from it is not kept across the loop
    asm volatile("" : "+v"(tid));
    const int j = tid & 3, site = (tid & 63) >> 2;
    cx<T> *dst = (f == 0 ? sh.t1 : sh.t2) + gn * 64 + gm * 16 + (e0 ^ (MM_SW * gm));
    __syncthreads();  // the previous tile's reads are done
    if (x0 + 16 <= V3) {
      vec v[9 * NH];
#pragma unroll
      for (int k = 0; k < 9 * NH; k++)
        v[k] = *(const __attribute__((address_space(1))) vec *)(src + x0 + ((k / 9) * 18 + k % 9) * PF.cs);
#pragma unroll
      for (int k = 0; k < 9 * NH; k++) *(av *)&dst[(k / 9) * 128 + (k % 9) * 256] = v[k];
    } else {
#pragma unroll 1
      for (int k = 0; k < 9 * NH; k++)
#pragma unroll
        for (int e = 0; e < EPU; e++)
          dst[(k / 9) * 128 + (k % 9) * 256 + e] =
              x0 + e0 + e < V3 ? gload(src + x0 + ((k / 9) * 18 + k % 9) * PF.cs + e) : cmake<T>(0, 0);
    }
    __syncthreads();
    if (P1.rot != 0 || P2.rot != 0) {
      if (PF.rot) mm_rotate(f == 0 ? sh.t1 : sh.t2, PF.rot, thr, 128);
      __syncthreads();
    }
    cx<T> cross[2], mes;
    if (wave == 0) mm_wave<T, 0, 0>(sh.t1, sh.t2, site, j, cross, mes);
    else if (wave == 1) mm_wave<T, 1, 0>(sh.t1, sh.t2, site, j, cross, mes);
    else if (wave == 2) mm_wave<T, 0, 1>(sh.t1, sh.t2, site, j, cross, mes);
    else mm_wave<T, 1, 1>(sh.t1, sh.t2, site, j, cross, mes);
    const int xc = wave & 1, h = wave >> 1, dcl = 2 * h + xc;
    cx<T> *xs = sh.x[site];
    if (h == 0 && j < 2) xs[2 * xc + j] = mes;
    if (j < 2) xs[4 + 4 * xc + 2 * h + j] = j == 0 ? cross[0] : cross[1];
    const bool in = x0 + site < V3;
    cx<T> *o = out + ((x0 >> 4) * ncols + col0) * 16 + site;
    {
      // the op of lane j: the class's j-th
      int op = 0;
#pragma unroll
      for (int k = 0; k < 16; k++) op = dcl * 4 + j == k ? meson_op(k >> 2, k & 3) : op;
      if (in) gstore(o + (int64_t)op * 16, sg * mes);
    }
    __syncthreads();
    if (wave == 0 && in) {  // lane j: mesmes of g5, g1, g2, g3
      const int xk = (j == 1 || j == 2) ? 1 : 0, tn = (j == 0 || j == 2) ? 1 : 0, cn = j >> 1;
      const cx<T> t = xs[2 * xk + tn], c = xs[4 + 4 * xk + cn] + xs[4 + 4 * xk + 2 + cn];
      gstore(o + (int64_t)(16 + j) * 16, t * t - c);
    }
  }
}

template <typename T>
int launch_mesmes(const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out, int64_t V3, int T_lat,
                  int nch_total, int ch0, int tiles_per_block, hipStream_t st) {
  const int ntiles = (int)((V3 + 15) / 16);
  const int gx = (ntiles + tiles_per_block - 1) / tiles_per_block;
  dim3 grid((unsigned)gx, (unsigned)nrows), block(MM_THREADS);
  k_mesmes<T><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0, ntiles);
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template int launch_mesmes<double>(const PropDev<double> *, const RowDev *, int, cx<double> *, int64_t, int, int,
                                   int, int, hipStream_t);
template int launch_mesmes<float>(const PropDev<float> *, const RowDev *, int, cx<float> *, int64_t, int, int,
                                  int, int, hipStream_t);

}  // namespace plg
