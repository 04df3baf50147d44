// plg_contract.hip -- per-site contractions of the 2pt path (gfx950).
//
// The kernels write the site correlator c[row][ch][x] (complex T,
// x contiguous) that the projection GEMM consumes as its K-contiguous operand.
//
//  k_meson_herm, k_meson_pair   one thread per site, HBM-bound.  Replace the
//                   meson bodies of lib/kernels/PLEGMA_mesons.cuh:25-52 and
//                   PLEGMA_mesonsNew.cuh:25-48.
//                   Single-propagator sets use the colour-traced spin Gram
//                   matrix G[p][q] = sum_ab S[p][ab] conj(S[q][ab]) restricted
//                   to the xor classes the channels touch (16 real + 24
//                   complex entries); two-propagator sets accumulate the
//                   channels directly.  Loads are coalesced SoA reads: lane i
//                   reads site x0+i of one spin-colour component.
//  k_meson_all      PLEGMA_mesonsAll.cuh:27-83: four lanes per site.
//
//  The baryon contractions and the fused meson + baryon kernel are in
//  plg_baryon.hip.
#include "plg_tile.h"

namespace plg {

// ------------------------------------------------------------------ tables
struct MTerm {
  int p, q, ph;  // coefficient i^ph on  S1[p] . conj(S2[q]) (colour traced)
};
struct ChanTable {
  int nch;
  MTerm t[16][16];
};

// Tr[G S1 g5 G S2^dag g5] = sum X[d][a] X[b][g] S1[a][b] conj(S2[d][g]), X = g5 G
constexpr void meson_terms(int op, MTerm *t) {
  SPerm X = sp_mul(G_5, gamma_op(op));
  int c = sp_class(X);
  int n = 0;
  for (int a = 0; a < 4; a++)
    for (int b = 0; b < 4; b++) {
      int d = a ^ c, g = b ^ c;
      t[n++] = MTerm{a * 4 + b, d * 4 + g, (X.ph[d] + X.ph[b]) & 3};
    }
}
constexpr ChanTable make_table(int set) {
  ChanTable T{};
  if (set == SET_M16) {
    T.nch = 16;
    for (int op = 0; op < 16; op++) meson_terms(op, T.t[op]);
  } else if (set == SET_M10 || set == SET_M10_PAIR) {
    T.nch = 10;
    for (int i = 0; i < 10; i++) meson_terms(MESON10_OPS[i], T.t[i]);
  }
  return T;
}

template <int SET> struct TableOf {
  static constexpr ChanTable v = make_table(SET);
};

__host__ __device__ constexpr int dmask(int d) { return (d << 2) | d; }
// index of p among the 8 representatives p < p^dmask(d)
constexpr int herm_rank(int d, int p) {
  int r = 0;
  for (int q = 0; q < p; q++)
    if (q < (q ^ dmask(d))) r++;
  return r;
}
constexpr int herm_rep(int d, int k) {
  int r = 0;
  for (int p = 0; p < 16; p++)
    if (p < (p ^ dmask(d))) {
      if (r == k) return p;
      r++;
    }
  return -1;
}

template <typename T>
__device__ __forceinline__ const cx<T> *site_base(const PropDev<T> &P, int t, int T_lat, int64_t V3,
                                                  int64_t x) {
  int plane = t - P.t_first;
  plane += plane < 0 ? T_lat : 0;
  return P.data + (int64_t)plane * V3 + x;
}

template <typename T> __device__ __forceinline__ cx<T> ldg(const cx<T> *p) { return gload(p); }

// ------------------------------------------------------------------ mesons
// Single propagator, Hermitian Gram form.  SET_M16 or SET_M10.
template <typename T, int SET>
__global__ __launch_bounds__(256) void k_meson_herm(const PropDev<T> *__restrict__ props,
                                                    const RowDev *__restrict__ rows,
                                                    cx<T> *__restrict__ out, int64_t V3,
                                                    int T_lat, int nch_total, int ch0) {
  const int r = blockIdx.y;
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= V3) return;
  const RowDev row = rows[r];
  const PropDev<T> P = props[row.pa];
  const cx<T> *base = site_base(P, row.t, T_lat, V3, x);
  const int64_t cs = P.cs;

  T n0[16];
  cx<T> gx[3][8];
#pragma unroll
  for (int p = 0; p < 16; p++) n0[p] = 0;
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int k = 0; k < 8; k++) gx[d][k] = cmake<T>(0, 0);

#pragma unroll 1
  for (int c = 0; c < 9; c++) {
    cx<T> s[16];
#pragma unroll
    for (int p = 0; p < 16; p++) s[p] = ldg(base + (int64_t)(p * 9 + c) * cs);
    // rotation to the physical basis (the boundary sign cancels in S x S^dag)
    if (P.rot) rot_spins(s, P.rot);
#pragma unroll
    for (int p = 0; p < 16; p++) n0[p] = fma(s[p].re, s[p].re, fma(s[p].im, s[p].im, n0[p]));
    static_for<1, 4>([&](auto d) {
      static_for<0, 8>([&](auto k) {
        constexpr int p = herm_rep(decltype(d)::value, decltype(k)::value);
        constexpr int q = p ^ dmask(decltype(d)::value);
        cfma_conj(gx[decltype(d)::value - 1][decltype(k)::value], s[p], s[q]);
      });
    });
  }
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)r * nch_total + ch0;
  static_for<0, TableOf<SET>::v.nch>([&](auto ch) {
    cx<T> acc = cmake<T>(0, 0);
    static_for<0, 16>([&](auto i) {
      constexpr MTerm tm = TableOf<SET>::v.t[decltype(ch)::value][decltype(i)::value];
      constexpr int d = (tm.p >> 2) ^ (tm.q >> 2);
      cx<T> v;
      if constexpr (d == 0) v = cmake<T>(n0[tm.p], 0);
      else if constexpr (tm.p < tm.q) v = gx[d - 1][herm_rank(d, tm.p)];
      else v = cconj(gx[d - 1][herm_rank(d, tm.q)]);
      acc = acc + cmul_iph(v, tm.ph);
    });
    gstore(out + ctile_idx(col0 + decltype(ch)::value, x, ncols), acc);
  });
}

// Two propagators, channels accumulated directly: SET_M10_PAIR.
template <typename T, int SET>
__global__ __launch_bounds__(256) void k_meson_pair(const PropDev<T> *__restrict__ props,
                                                    const RowDev *__restrict__ rows,
                                                    cx<T> *__restrict__ out, int64_t V3,
                                                    int T_lat, int nch_total, int ch0) {
  const int r = blockIdx.y;
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= V3) return;
  const RowDev row = rows[r];
  const PropDev<T> P1 = props[row.pa], P2 = props[row.pb];
  const cx<T> *b1 = site_base(P1, row.t, T_lat, V3, x);
  const cx<T> *b2 = site_base(P2, row.t, T_lat, V3, x);
  constexpr int NCH = TableOf<SET>::v.nch;
  cx<T> acc[NCH];
#pragma unroll
  for (int i = 0; i < NCH; i++) acc[i] = cmake<T>(0, 0);
#pragma unroll 1
  for (int c = 0; c < 9; c++) {
    cx<T> s1[16], s2[16];
#pragma unroll
    for (int p = 0; p < 16; p++) {
      s1[p] = ldg(b1 + (int64_t)(p * 9 + c) * P1.cs);
      s2[p] = ldg(b2 + (int64_t)(p * 9 + c) * P2.cs);
    }
    if (P1.rot) rot_spins(s1, P1.rot);
    if (P2.rot) rot_spins(s2, P2.rot);
    static_for<0, NCH>([&](auto ch) {
      static_for<0, 16>([&](auto i) {
        constexpr MTerm tm = TableOf<SET>::v.t[decltype(ch)::value][decltype(i)::value];
        cx<T> prod = cmake<T>(0, 0);
        cfma_conj(prod, s1[tm.p], s2[tm.q]);
        acc[decltype(ch)::value] = acc[decltype(ch)::value] + cmul_iph(prod, tm.ph);
      });
    });
  }
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)r * nch_total + ch0;
  // boundary signs: the channels are bilinear in S1 and S2
  const T sg = prop_sign(P1, row.t) * prop_sign(P2, row.t);
#pragma unroll
  for (int ch = 0; ch < NCH; ch++)
    gstore(out + ctile_idx(col0 + ch, x, ncols), cmake<T>(sg * acc[ch].re, sg * acc[ch].im));
}

// ------------------------------------------------------------------ mesonsAll
// The 34 channels of contractMesonsAll as Tr[M S1 N S2^dag] (M = N = X for the
// first two): signed permutations of xor classes c_M, c_N, so
//   ch = sum_b N[b] sum_a M[a ^ c_M] sum_colour S1[a][b] conj(S2[a ^ c_M][b ^ c_N]).
// Four lanes of a wave share a site, lane row j = lane / 16 holding the source
// spin b = j of S1: the sums over a and the colours depend on N through its
// class only (26 partial sums instead of 34 channels, a quarter of the terms
// each), and one launch holds them all.  The rows of a wave read the same
// entries of S2 for every class, in another order: one line from HBM, the
// other classes' from the L1.
// HBM-bound: one read of both propagators.  24 x 20 x 28 x 25 sites in FP64:
// two launches of 17 channels, each reading both, 2 x 350 us -> 370 us
// (FP32, rotated views included, faster than before alike: 490 -> 370 us a call,
// rotated 480; FP64 rotated 845 -> 700).
struct AllChan {
  int m, n;    // operators; X = g5 G of them if x
  bool x;
};
constexpr AllChan all_chan(int ch) {
  if (ch < 2) return AllChan{ch == 0 ? 5 : 0, ch == 0 ? 5 : 0, true};
  const int p = (ch - 2) / 16, i = (ch - 2) / 4 % 4, j = (ch - 2) % 4;
  return AllChan{1 + i + 5 * p, 1 + j + 5 * p, false};
}
constexpr SPerm all_mat(int op, bool x) { return x ? sp_mul(G_5, gamma_op(op)) : gamma_op(op); }
// the partial sums: (operator, x, class of N), in the order of the channels that need them first
constexpr int MALL_SUMS = 26;
struct AllSums {
  int m[MALL_SUMS], cn[MALL_SUMS];
  bool x[MALL_SUMS];
  int of[34];
  int n;
};
constexpr AllSums make_all_sums() {
  AllSums s{};
  for (int ch = 0; ch < 34; ch++) {
    const AllChan c = all_chan(ch);
    const int cn = sp_class(all_mat(c.n, c.x));
    int k = 0;
    while (k < s.n && !(s.m[k] == c.m && s.x[k] == c.x && s.cn[k] == cn)) k++;
    if (k == s.n) {
      s.m[k] = c.m;
      s.x[k] = c.x;
      s.cn[k] = cn;
      s.n++;
    }
    s.of[ch] = k;
  }
  return s;
}
constexpr AllSums ALL_SUMS = make_all_sums();
static_assert(ALL_SUMS.n == MALL_SUMS, "partial sums of mesonsAll");

// the value of row j ^ 2 (up: j is 2 or 3)
__device__ __forceinline__ float row_xor2(float v, bool up) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(up ? r[0] : r[1]);
}
__device__ __forceinline__ double row_xor2(double v, bool up) {
  const unsigned lo = (unsigned)__double_as_longlong(v), hi = (unsigned)(__double_as_longlong(v) >> 32);
  const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __longlong_as_double(((long long)(up ? h[0] : h[1]) << 32) | (up ? l[0] : l[1]));
}
// of four values per row, the sums over the rows: row n keeps value n
__device__ __forceinline__ float row_scatter_sum(float a, float b, float c, float d) {
  auto sum16 = [](float p, float q) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(p), __float_as_uint(q), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const auto r =
      __builtin_amdgcn_permlane32_swap(__float_as_uint(sum16(a, b)), __float_as_uint(sum16(c, d)), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double row_scatter_sum(double a, double b, double c, double d) {
  auto join = [](unsigned lo, unsigned hi) { return __longlong_as_double(((long long)hi << 32) | lo); };
  auto lo = [](double v) { return (unsigned)__double_as_longlong(v); };
  auto hi = [](double v) { return (unsigned)(__double_as_longlong(v) >> 32); };
  auto sum16 = [&](double p, double q) {
    const auto l = __builtin_amdgcn_permlane16_swap(lo(p), lo(q), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi(p), hi(q), false, false);
    return join(l[0], h[0]) + join(l[1], h[1]);
  };
  const double x = sum16(a, b), y = sum16(c, d);
  const auto l = __builtin_amdgcn_permlane32_swap(lo(x), lo(y), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi(x), hi(y), false, false);
  return join(l[0], h[0]) + join(l[1], h[1]);
}

// ROT: a view is rotated on load
template <typename T, bool ROT>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? (ROT ? 3 : 4) : 2) void k_meson_all(const PropDev<T> *__restrict__ props,
                                                                            const RowDev *__restrict__ rows,
                                                                            cx<T> *__restrict__ out, int64_t V3,
                                                                            int T_lat, int nch_total, int ch0) {
  const int lane = threadIdx.x & 63, j = lane >> 4;
  const int64_t xs = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + (lane & 15);
  const int64_t x = xs < V3 ? xs : V3 - 1;  // rows past the end repeat the last site
  const RowDev row = rows[blockIdx.y];
  const PropDev<T> P1 = props[row.pa], P2 = props[row.pb];
  const cx<T> *b1 = site_base(P1, row.t, T_lat, V3, x), *b2 = site_base(P2, row.t, T_lat, V3, x);
  // the entries [a][nu] of a colour pair, in the physical basis
  auto load = [&](const cx<T> *b, int64_t cs, int rot, int nu, cx<T> (&s)[4]) {
#pragma unroll
    for (int a = 0; a < 4; a++) s[a] = ldg(b + (int64_t)((a * 4 + nu) * 9) * cs);
    if (ROT && rot) {
      // with the entries o of source spin nu ^ 2, which the row j ^ 2 holds;
      // both pairs of rot_physical read alike from either side
      const T r = (T)rot, h = (T)0.5;
#pragma unroll
      for (int a = 0; a < 2; a++) {
        const cx<T> p = s[a], q = s[a + 2], o = cmake<T>(row_xor2(p.re, j & 2), row_xor2(p.im, j & 2)),
                    u = cmake<T>(row_xor2(q.re, j & 2), row_xor2(q.im, j & 2));
        s[a] = cmake<T>(h * ((p.re - u.re) - r * (o.im + q.im)), h * ((p.im - u.im) + r * (o.re + q.re)));
        s[a + 2] = cmake<T>(h * ((q.re - o.re) - r * (u.im + p.im)), h * ((q.im - o.im) + r * (u.re + p.re)));
      }
    }
  };
  cx<T> w[MALL_SUMS];
#pragma unroll
  for (int i = 0; i < MALL_SUMS; i++) w[i] = cmake<T>(0, 0);
#pragma unroll 1
  for (int c = 0; c < 9; c++) {
    cx<T> s1[4];
    load(b1 + c * P1.cs, P1.cs, P1.rot, j, s1);
    static_for<0, 4>([&](auto cn) {
      cx<T> s2[4];
      load(b2 + c * P2.cs, P2.cs, P2.rot, j ^ cn.value, s2);
      static_for<0, MALL_SUMS>([&](auto i) {
        if constexpr (ALL_SUMS.cn[i.value] == cn.value) {
          constexpr SPerm M = all_mat(ALL_SUMS.m[i.value], ALL_SUMS.x[i.value]);
          constexpr int cm = sp_class(M);
          static_assert(char_ok(M.ph), "sign characters");
          static_for<0, 4>([&](auto a) {
            constexpr int d = a.value ^ cm, ph = (M.ph[d] - M.ph[0]) & 3;
            if constexpr (ph == 0) cfma_conj(w[i.value], s1[a.value], s2[d]);
            else cfma_conj(w[i.value], cmake<T>(-s1[a.value].re, -s1[a.value].im), s2[d]);
          });
        }
      });
      if constexpr (ROT) __builtin_amdgcn_sched_barrier(0);  // one class's loads at a time: registers
    });
  }
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total + ch0;
  // boundary signs: the channels are bilinear in S1 and S2
  const T sg = prop_sign(P1, row.t) * prop_sign(P2, row.t);
  static_for<0, 9>([&](auto g) {
    cx<T> v[4];
    static_for<0, 4>([&](auto k) {
      constexpr int ch = 4 * g.value + k.value < 34 ? 4 * g.value + k.value : 33;
      constexpr AllChan c = all_chan(ch);
      constexpr SPerm M = all_mat(c.m, c.x), N = all_mat(c.n, c.x);
      const cx<T> u = cmul_iph(w[ALL_SUMS.of[ch]], M.ph[0] + N.ph[0]);
      const T f = sg * char_sign<T>(N.ph, j);
      v[k.value] = cmake<T>(f * u.re, f * u.im);
    });
    const cx<T> r = cmake<T>(row_scatter_sum(v[0].re, v[1].re, v[2].re, v[3].re),
                             row_scatter_sum(v[0].im, v[1].im, v[2].im, v[3].im));
    if (4 * g.value + j < 34 && xs < V3) gstore(out + ctile_idx(col0 + 4 * g.value + j, xs, ncols), r);
  });
}

// ------------------------------------------------------------------ launchers
template <typename T>
int launch_meson(int set, const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out,
                 int64_t V3, int T_lat, int nch_total, int ch0, bool rot, hipStream_t st) {
  dim3 block(256), grid((unsigned)((V3 + 255) / 256), (unsigned)nrows);
  switch (set) {
  case SET_M16:
    k_meson_herm<T, SET_M16><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0);
    break;
  case SET_M10:
    k_meson_herm<T, SET_M10><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0);
    break;
  case SET_M10_PAIR:
    k_meson_pair<T, SET_M10_PAIR><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0);
    break;
  case SET_MALL:
    grid.x = (unsigned)((V3 + 63) / 64);
    if (rot) k_meson_all<T, true><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0);
    else k_meson_all<T, false><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0);
    break;
  default:
    return PLG_ERR_INVALID;
  }
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template int launch_meson<double>(int, const PropDev<double> *, const RowDev *, int, cx<double> *,
                                  int64_t, int, int, int, bool, hipStream_t);
template int launch_meson<float>(int, const PropDev<float> *, const RowDev *, int, cx<float> *,
                                 int64_t, int, int, int, bool, hipStream_t);

}  // namespace plg
