// plg_baryon.hip -- baryon two-point contractions (and the fused meson +
// baryon two-point kernel) on gfx950.
//
// Replaces PLEGMA_baryons_NtoN.cu:6-46 (proton, Cg5 x Cg5) and
// PLEGMA_baryons_deltas.cu:61-110 (Delta iso-3/2, Cg_k x g4 (Cg_k)^dag g4)
// with factorised forms.  For a diquark matrix A (Abar = g4 A^dag g4) and
// propagators P (quarks outside the diquark's partner) and Qm:
//   St^{bb'}_{nu nu'}  = A_{nu lam} Qm^{bb'}_{lam lam'} Abar_{lam' nu'}
//   W^{ck}_{nu' mu'}   = eps_abc eps_kb'c' sum_nu St^{bb'}_{nu nu'} P^{ac'}_{nu mu'}
//   X_{mu mu'}         = sum_{nu' c k} P^{ck}_{mu nu'} W^{ck}_{nu' mu'}
//   D_{mu mu'}         = -sum_{ck} tr(W^{ck}) P^{ck}_{mu mu'}
//   proton  (Qm = other flavour)      = D - X
//   Delta_k (uuu, Cg_k symmetric)     = 2 D - 4 X
// (the direct term's colour sum eps eps' P St over nu = mu is minus the trace
// of W, by renaming the eps' indices).  Both results are one product of P
// with W whose diagonal takes up the trace:
//   D - X     =    - sum P^{ck}_{mu nu'} (W^{ck}_{nu' mu'} + delta_{nu' mu'}     tr W^{ck})
//   2 D - 4 X = -4 * sum P^{ck}_{mu nu'} (W^{ck}_{nu' mu'} + delta_{nu' mu'} 1/2 tr W^{ck})
//
// The four diquarks Cg5, Cg3 and Cg1, Cg2 are signed permutations of two xor
// classes c; the two of a class differ by phases, so their W come from the
// same colour products M(Qm_{nu^c nu'^c}, P_{nu mu'}) (sum x +- y over the two
// kinds of rows nu).  M is symmetric in its arguments: with Qm = P, rows nu
// and nu^c exchange (nu', mu') with (mu'^c, nu'^c), so half of the products
// (one row of each pair for c = 1, one order of (a, b) for c = 0) give W by a
// transposition.
//
// Work split: four lanes per site, 16 sites per wave, lane j = mu'; the other
// spin index runs relative to it, nu' = j ^ s, s = 0..3, so the transposition
// is the exchange of lanes j and j ^ s (or j ^ s ^ 1), a DPP operand of the
// adds, the diagonal is s = 0, and W stays in registers.  The Abar phase of
// nu' is a sign character of the spin index: sigma(j ^ s) = sigma(j) sigma(s),
// a lane sign of the result and compile-time signs of the products.  The
// operands come from the staged tile in LDS, 8 FMAs per 8-byte read.  One wave
// contracts {Cg5, Cg3}, another {Cg1, Cg2} and each half of the mesons of
// the same staged 16 sites.
//
// Rounding: the diagonal with the trace holds the largest terms of the last
// product, so they come last in chains of 12 products, one per colour row c.
// Rms error in FP32 on normal entries (proton, Delta, proton of two flavours):
// 9.7, 9.0, 12.0 e-8; the two terms summed apart, 9.9, 13.0, 12.7; one chain of
// 36 products, the diagonal first, 15.9, 16.3, 18.5 (at the same speed within 1 %).
//
// What bounds it: vector instructions (per site and propagator 278 of the 372
// wave instructions are the products' FMAs, 9 300 flop per lane-site), and in
// FP32 the power they take: two waves issue FMAs together (2.9 cycles per
// instruction measured here, 2.45 in a loop of FMAs alone), and the clock
// falls to 1.7 GHz.  Four waves per SIMD (18 KB of LDS per 2-wave workgroup,
// 128 registers) measured best; two or three waves, operands read two or
// three steps ahead, the next tile prefetched into registers, and 4 x 4 spin
// products on v_mfma_f32_4x4x1 (12.8 cycles each, not beside the vector
// unit's work) were within 5 % or slower.  Sixteen lanes per site with W
// exchanged through LDS and the trace formed apart (the earlier form) took
// 16.3 ms on 10.98 M sites x 80 channels in FP32, this one 7.1 ms (1 550 M
// sites/s; the HBM floor of its 20 GB is 4.2 ms); FP64, two flavours, 276 k
// sites x 128 channels: 2.36 -> 0.95 ms.
#include "plg_tile.h"

namespace plg {

// entry (mu, nu, colour pair cc) of site x at cc 256 + mu 64 + nu 16 + (x ^ SW nu):
// the 16 lanes of an LDS pass, which hold the four nu of four sites (consecutive
// ones for 8-byte reads, sites 0, 3, 5, 6 mod 8 for 16-byte reads), read distinct
// banks; the spin mu and colour offsets are immediates
constexpr int BQ_TILE = 144 * 16;
constexpr int BQ_SW = 4;
template <typename T> struct BqT {
  static constexpr int EPU = sizeof(T) == 4 ? 2 : 1;  // sites of a 16-byte unit
  static constexpr int WPE = sizeof(T) == 4 ? 4 : 2;  // waves per SIMD (LDS and registers)
};
// R[b][mu] (column mu' = j) of diquark W0 and, if W1 >= 0, of W1 of its class:
// sum over nu', c, k of P (W + kappa delta tr W), up to the scale and lane
// sign of bq_scale.  P, Q: the tiles at (lane, s = 0 column); SAME: Q = P
template <int W0, int W1> struct BqClass {
  static constexpr SPerm A0 = diquark(W0), A1 = diquark(W1 >= 0 ? W1 : W0);
  static constexpr SPerm Ab0 = diquark_bar(W0), Ab1 = diquark_bar(W1 >= 0 ? W1 : W0);
  static constexpr int cls = sp_class(A0);
  static constexpr int RA = (A1.ph[0] - A0.ph[0]) & 3;
  // the second diquark's row phases are A1.ph = A0.ph + RA + kind
  static constexpr int kind(int nu) { return (A1.ph[nu] - A0.ph[nu] - RA) & 3; }
  // the n-th row of the halved sum (c = 1): one of each pair, of kind 0
  static constexpr int row(int n) {
    for (int nu = 0; nu < 4; nu++)
      if ((W1 >= 0 ? kind(nu) == 0 : nu < (nu ^ cls)) && n-- == 0) return nu;
    return -1;
  }
  // phase of row nu ^ c relative to row nu: 0 symmetric, 2 antisymmetric
  static constexpr int partner = cls ? (A0.ph[row(0) ^ cls] - A0.ph[row(0)]) & 3 : 0;
  static constexpr bool ok() {
    if (sp_class(A1) != cls || sp_class(Ab0) != cls || sp_class(Ab1) != cls || cls > 1) return false;
    for (int nu = 0; nu < 4; nu++)
      if (kind(nu) & 1) return false;
    if (cls && (((A0.ph[row(1) ^ cls] - A0.ph[row(1)]) & 3) != partner || (partner & 1))) return false;
    return char_ok(Ab0.ph) && char_ok(Ab1.ph);
  }
  // phase of Abar row nu' (character of nu', with the class shift as an offset)
  static constexpr int ab(int b, int n) { return b == 0 ? Ab0.ph[n ^ cls] : Ab1.ph[n ^ cls]; }
  static constexpr int sig(int b, int s) { return (ab(b, s) - ab(b, 0)) & 3; }  // 0 or 2
  // phase of a whole result
  static constexpr int phase(int b) { return (ab(b, 0) + (b == 1 ? RA : 0)) & 3; }
};

template <typename T, int W0, int W1, bool SAME>
__device__ __forceinline__ void bq_class(const cx<T> *P, const cx<T> *Q, int site, int j, cx<T> (&R)[2][4]) {
  using B = BqClass<W0, W1>;
  static_assert(B::ok(), "row phases, symmetry and sign characters of the class");
  constexpr int NB = W1 >= 0 ? 2 : 1, cls = B::cls;
  constexpr bool HALF_NU = SAME && cls == 1, HALF_AB = SAME && cls == 0;
  constexpr int NN = HALF_NU ? 2 : 4;                       // rows nu summed
  constexpr bool TWO_ACC = NB == 2 && !HALF_NU;             // kinds summed apart
  // columns nu' = j ^ s of the tiles
  const cx<T> *pc[4], *qc[4];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int n = j ^ s;
    pc[s] = P + n * 16 + (site ^ (BQ_SW * n));
    qc[s] = SAME ? pc[s] : Q + n * 16 + (site ^ (BQ_SW * n));
  }
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int m = 0; m < 4; m++) R[b][m] = cmake<T>(0, 0);
  // The operands of a step are read from LDS while the previous step's
  // products run (two buffers): a step is a row nu and an s in the sums of W,
  // a row mu and an s in the products with P.  The scheduler, left alone,
  // places the reads next to their use.
  cx<T> p[2][2][3], q[2][2][3];
  auto load_p = [&](auto r_, int o0, int o1) {
    constexpr int r = r_.value, nu = HALF_NU ? B::row(r) : r;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      p[r & 1][0][k] = pc[0][nu * 64 + o0 + k * 256];
      if constexpr (!HALF_AB) p[r & 1][1][k] = pc[0][nu * 64 + o1 + k * 256];
    }
  };
  auto load_q = [&](auto i_, int o0, int o1) {
    constexpr int i = i_.value, r = i / 4, s = i % 4, nu = HALF_NU ? B::row(r) : r;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      if constexpr (!HALF_AB) q[i & 1][0][k] = qc[s ^ cls][(nu ^ cls) * 64 + o0 + k * 256];
      q[i & 1][1][k] = qc[s ^ cls][(nu ^ cls) * 64 + o1 + k * 256];
    }
  };
  auto load_x = [&](auto i_, int oc) {
    constexpr int i = i_.value, s = 3 - i % 4, m = i / 4;
#pragma unroll
    for (int k = 0; k < 3; k++) q[i & 1][0][k] = pc[s][m * 64 + oc + k * 256];
  };
  load_p(ic<0>{}, 768, 1536);
  load_q(ic<0>{}, 768, 1536);
#pragma unroll 1
  for (int c = 0; c < 3; c++) {
    const int o0 = (c < 2 ? c + 1 : 0) * 768, o1 = (c > 0 ? c - 1 : 2) * 768;
    cx<T> x[4][3], y[4][3];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int k = 0; k < 3; k++) x[s][k] = y[s][k] = cmake<T>(0, 0);
    static_for<0, 4 * NN>([&](auto i_) {
      constexpr int i = i_.value, r = i / 4, s = i % 4, nu = HALF_NU ? B::row(r) : r;
      if constexpr (s == 2 && r + 1 < NN) load_p(ic<r + 1>{}, o0, o1);
      if constexpr (i + 1 < 4 * NN) load_q(ic<i + 1>{}, o0, o1);
      else load_x(ic<0>{}, c * 768);
      __builtin_amdgcn_sched_barrier(0);
      // the eps_abc orders (a, b) = (r0, r1), (r1, r0), the eps_kb'c' orders of every k
      static_for<0, (HALF_AB ? 1 : 2)>([&](auto e1) {
        static_for<0, 2>([&](auto e2) {
          static_for<0, 3>([&](auto k_) {
            constexpr int k = k_.value, bp = (k + 1 + e2.value) % 3, cp = (k + 2 - e2.value) % 3;
            constexpr int ph = B::A0.ph[nu] + (e1.value == e2.value ? 0 : 2);
            if constexpr (TWO_ACC && B::kind(nu) == 2)
              cfma_iph<ph>(y[s][k], q[i & 1][1 - e1.value][bp], p[r & 1][e1.value][cp]);
            else
              cfma_iph<ph>(x[s][k], q[i & 1][1 - e1.value][bp], p[r & 1][e1.value][cp]);
          });
        });
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    // V[0] = x + y, V[1] = x - y (times i^RA, in the result's phase)
    cx<T> V[2][4][3];
    static_for<0, 4>([&](auto s_) {
      constexpr int s = s_.value;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        cx<T> a = x[s][k], d = y[s][k];
        if constexpr (HALF_AB) {
          a = cmake<T>(a.re + quad_xor<s>(a.re), a.im + quad_xor<s>(a.im));
          if constexpr (TWO_ACC) d = cmake<T>(d.re + quad_xor<s>(d.re), d.im + quad_xor<s>(d.im));
        }
        if constexpr (HALF_NU) {
          d = cmake<T>(quad_xor<s ^ 1>(a.re), quad_xor<s ^ 1>(a.im));
          V[0][s][k] = B::partner == 0 ? a + d : a - d;
          V[1][s][k] = B::partner == 0 ? a - d : a + d;
        } else if constexpr (TWO_ACC) {
          V[0][s][k] = a + d;
          V[1][s][k] = a - d;
        } else {
          V[0][s][k] = a;
        }
      }
    });
    // the trace over nu' = mu' joins the diagonal s = 0 with weight kappa; up
    // to the lane sign sigma(j), sum_j' sigma(j') v(j') = sum_s sigma(s) v(j ^ s)
    static_for<0, NB>([&](auto b_) {
      constexpr int b = b_.value;
      constexpr T kap = (b == 0 ? W0 : W1) == 0 ? (T)1 : (T)0.5;
      auto trace = [&](T t) {
        t = B::sig(b, 1) == 0 ? t + quad_xor<1>(t) : t - quad_xor<1>(t);
        return B::sig(b, 2) == 0 ? t + quad_xor<2>(t) : t - quad_xor<2>(t);
      };
#pragma unroll
      for (int k = 0; k < 3; k++) {
        cx<T> &v = V[b][0][k];
        v = cmake<T>(fma(kap, trace(v.re), v.re), fma(kap, trace(v.im), v.im));
      }
    });
    // R[b][mu] += P[mu][nu'] . V[b][nu'], the sign of s included.  A row's
    // products of one colour row are summed by themselves, the diagonal s = 0,
    // which holds the trace, last (the header has the errors).
    cx<T> r[2];
    static_for<0, 16>([&](auto i_) {
      constexpr int i = i_.value, s = 3 - i % 4, m = i / 4;
      if constexpr (i < 15) {
        load_x(ic<i + 1>{}, c * 768);
      } else {  // the next colour row's first operands
        load_p(ic<0>{}, (c < 1 ? c + 2 : c - 1) * 768, c * 768);
        load_q(ic<0>{}, (c < 1 ? c + 2 : c - 1) * 768, c * 768);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s == 3) r[0] = r[1] = cmake<T>(0, 0);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const cx<T> pv = q[i & 1][0][k];
        // (an antisymmetric diquark has no s = 1 part)
        if constexpr (!(HALF_NU && s == 1 && B::partner == 2)) cfma_iph<B::sig(0, s)>(r[0], pv, V[0][s][k]);
        if constexpr (NB == 2 && !(HALF_NU && s == 1 && B::partner == 0)) cfma_iph<B::sig(1, s)>(r[1], pv, V[1][s][k]);
      }
      if constexpr (s == 0)
#pragma unroll
        for (int b = 0; b < NB; b++) R[b][m] = R[b][m] + r[b];
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // lane sign and phase of the results
  static_for<0, NB>([&](auto b_) {
    constexpr int b = b_.value;
    const T sg = char_sign<T>(b == 0 ? B::Ab0.ph : B::Ab1.ph, j);
#pragma unroll
    for (int m = 0; m < 4; m++) R[b][m] = sg * cmul_iph(R[b][m], B::phase(b));
  });
}

// mesons of the xor classes [D0, D1): G_d[al][be] = sum_cc S[al][be] conj(S[al^d][be^d]),
// channel op of class d: sum_{al be} i^(ph[al^d] + ph[be]) G_d[al][be].
// Lane j holds column be = j.  Of the pair (al, j), (al^d, j^d), whose entries
// are conjugate, each lane sums its own column at the al without d's top bit;
// the other half comes from the partner lane.  Of the four channels of a
// class, lane n of the site receives the n-th (store(op, value)).
template <int D0, int D1, typename T, typename F>
__device__ __forceinline__ void bq_mesons(const cx<T> *S, int site, int j, F &&store) {
  const cx<T> *col = S + j * 16 + (site ^ (BQ_SW * j));
  T n0[4] = {0, 0, 0, 0};
  cx<T> g[3][2];
#pragma unroll
  for (int d = 0; d < 3; d++) g[d][0] = g[d][1] = cmake<T>(0, 0);
#pragma unroll 3
  for (int cc = 0; cc < 9; cc++) {
    cx<T> s[4];
#pragma unroll
    for (int al = 0; al < 4; al++) s[al] = col[al * 64 + cc * 256];
    static_for<D0, D1>([&](auto d_) {
      constexpr int d = d_.value;
      if constexpr (d == 0) {
#pragma unroll
        for (int al = 0; al < 4; al++) n0[al] = fma(s[al].re, s[al].re, fma(s[al].im, s[al].im, n0[al]));
      } else {
        static_for<0, 2>([&](auto h) {
          constexpr int al = d >= 2 ? h.value : 2 * h.value;
          const cx<T> o = cmake<T>(quad_xor<d>(s[al ^ d].re), quad_xor<d>(s[al ^ d].im));
          cfma_conj(g[d - 1][h.value], s[al], o);
        });
      }
    });
  }
  static_for<D0, D1>([&](auto d_) {
    constexpr int d = d_.value;
    cx<T> G[4];
    if constexpr (d == 0) {
#pragma unroll
      for (int al = 0; al < 4; al++) G[al] = cmake<T>(n0[al], 0);
    } else {
      static_for<0, 2>([&](auto h) {
        constexpr int al = d >= 2 ? h.value : 2 * h.value;
        G[al] = g[d - 1][h.value];
        G[al ^ d] = cmake<T>(quad_xor<d>(G[al].re), -quad_xor<d>(G[al].im));
      });
    }
    cx<T> v[4];
    static_for<0, 4>([&](auto n) {
      constexpr int op = meson_op(d, n.value);
      static_assert(op >= 0 && char_ok(MESON_X.ph[op < 0 ? 0 : op]), "four channels per class, sign characters");
      cx<T> w = cmake<T>(0, 0);
      static_for<0, 4>([&](auto al) { w = w + cmul_iph(G[al.value], MESON_X.ph[op][al.value ^ d] + MESON_X.ph[op][0]); });
      v[n.value] = char_sign<T>(MESON_X.ph[op], j) * w;
    });
    const int op = j == 0 ? meson_op(d, 0) : j == 1 ? meson_op(d, 1) : j == 2 ? meson_op(d, 2) : meson_op(d, 3);
    store(op, quad_scatter_sum(v, j));
  });
}

// rotation of a staged tile to the physical basis in place (nthr threads)
template <typename T> __device__ __forceinline__ void bq_rotate(cx<T> *S, int sign, int thr, int nthr) {
  for (int it = thr; it < 16 * 36; it += nthr) {
    const int s = it & 15, cq = it >> 4, cp = cq % 9, q = cq / 9, m = q >> 1, n = q & 1;
    auto at = [&](int mu, int nu) -> cx<T> & { return S[cp * 256 + mu * 64 + nu * 16 + (s ^ (BQ_SW * nu))]; };
    cx<T> a = at(m, n), b = at(m, n + 2), c = at(m + 2, n), d = at(m + 2, n + 2);
    rot_physical(a, b, c, d, sign);
    at(m, n) = a;
    at(m, n + 2) = b;
    at(m + 2, n) = c;
    at(m + 2, n + 2) = d;
  }
}

// waves of a workgroup and the work of each: the datasets times the halves
// (diquark classes {Cg5, Cg3} and {Cg1, Cg2}, or baryons and mesons)
template <bool TWO, bool MES, int GMASK> struct BqSplit {
  static constexpr bool H0 = GMASK & 1, H1 = GMASK & (1 << 7), H2 = GMASK & (1 << 8), H3 = GMASK & (1 << 9);
  static_assert(H1 == H2 && H2 == H3, "the Delta groups are computed together");
  static constexpr int halves = (H1 || MES) ? 2 : 1;
  static constexpr int ND = TWO ? 2 : 1;
  static constexpr int threads = 64 * halves * ND;
};

// Output channels per row (from ch0): [16 mesons of S1 if MES], then for each
// dataset d (2 if TWO) and each selected group g in the reference order
// (nucl_nucl, deltapp_deltamm_11, _22, _33): 16 components mu*4 + mu'.
template <typename T, bool TWO, bool MES, int GMASK>
__global__ __launch_bounds__((BqSplit<TWO, MES, GMASK>::threads)) __attribute__((amdgpu_waves_per_eu(BqT<T>::WPE)))
void k_baryon(const PropDev<T> *__restrict__ props, const RowDev *__restrict__ rows, cx<T> *__restrict__ out,
              int64_t V3, int T_lat, int nch_total, int ch0, int ntiles) {
  using B = BqSplit<TWO, MES, GMASK>;
  constexpr bool H0 = B::H0, HD = B::H1;
  constexpr int NG = (int)H0 + 3 * (int)HD;
  constexpr int R0 = 0, R1 = (int)H0, R2 = R1 + 1, R3 = R1 + 2;
  constexpr int MOFF = MES ? 1 : 0;
  constexpr int NT = 64 * B::halves;  // threads that stage a propagator
  // staging: UPC threads of a spin pair load the 16 sites of a component in
  // 16-byte units; thread group g takes the spin pairs g + PG h, the nine
  // colour pairs of each (nu = g % 4: one LDS offset per thread)
  constexpr int EPU = BqT<T>::EPU, UPC = 16 / EPU, PG = NT / UPC, NH = 16 / PG, NU = 9 * NH;
  static_assert(PG % 4 == 0 && NH * PG == 16, "whole passes over the spin pairs");
  typedef typename SiteVec<T, EPU>::v vec;
  __shared__ __align__(16) cx<T> tile[B::ND][BQ_TILE];
  const RowDev row = rows[blockIdx.y];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave % B::halves, ds = wave / B::halves;
  const PropDev<T> P1 = props[row.pa], P2 = props[TWO ? row.pb : row.pa];
  // the propagator this wave stages: its dataset's
  const PropDev<T> PD = ds == 0 ? P1 : P2;
  const int thr = threadIdx.x - ds * NT, g0 = thr / UPC, e0 = (thr % UPC) * EPU;
  const cx<T> *src = PD.data + (int64_t)((row.t - PD.t_first + T_lat) % T_lat) * V3 + (int64_t)(g0 * 9) * PD.cs + e0;
  // the boundary signs multiply the results: a baryon of dataset d holds its
  // propagator squared times the diquark's other one (proton) or cubed
  const T sgp = prop_sign(PD, row.t), sgo = TWO ? prop_sign(ds == 0 ? P2 : P1, row.t) : sgp;
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total + ch0;

  for (int tl = blockIdx.x; tl < ntiles; tl += gridDim.x) {
    const int64_t x0 = (int64_t)tl * 16;
    // opaque: addresses and masks derived from it are formed per tile instead
    // of being kept in registers across the loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int j = tid & 3, site = (tid & 63) >> 2;
    cx<T> *dst = tile[ds] + g0 * 16 + (e0 ^ (BQ_SW * (g0 & 3)));
    __syncthreads();  // the previous tile's reads are done
    if (x0 + 16 <= V3) {
      vec v[NU];
#pragma unroll
      for (int k = 0; k < NU; k++)
        v[k] = *(const __attribute__((address_space(1))) vec *)(src + x0 + ((k / 9) * (9 * PG) + k % 9) * PD.cs);
#pragma unroll
      for (int k = 0; k < NU; k++) {
        typedef T av __attribute__((ext_vector_type(2 * EPU)));
        *(av *)&dst[(k / 9) * (16 * PG) + (k % 9) * 256] = v[k];
      }
    } else {
#pragma unroll 1
      for (int k = 0; k < NU; k++)
#pragma unroll
        for (int e = 0; e < EPU; e++)
          dst[(k / 9) * (16 * PG) + (k % 9) * 256 + e] =
              x0 + e0 + e < V3 ? gload(src + x0 + ((k / 9) * (9 * PG) + k % 9) * PD.cs + e) : cmake<T>(0, 0);
    }
    __syncthreads();
    if (P1.rot != 0 || (TWO && P2.rot != 0)) {
      if (PD.rot) bq_rotate(tile[ds], PD.rot, thr, NT);
      __syncthreads();
    }
    const bool in = x0 + site < V3;
    cx<T> *o = out + ((x0 >> 4) * ncols + col0) * 16 + site;
    // the 4 rows mu of column mu' = j: a wave's stores of a row cover 4 columns of 16 sites
    auto put = [&](int g, T scale, const cx<T> (&r)[4]) {
      if (in)
#pragma unroll
        for (int m = 0; m < 4; m++) gstore(o + (int64_t)((MOFF + g) * 16 + 4 * m + j) * 16, scale * r[m]);
    };
    auto put_meson = [&](int op, cx<T> v) {
      if (in) gstore(o + (int64_t)op * 16, v);
    };
    const cx<T> *P = tile[TWO ? ds : 0], *Qo = tile[TWO ? 1 - ds : 0];
    const int base = ds * NG;
    cx<T> R[2][4];
    if (half == 0) {
      if constexpr (H0 && HD && !TWO) {
        bq_class<T, 0, 3, true>(P, P, site, j, R);
        put(base + R0, -sgo, R[0]);
        put(base + R3, -4 * sgp, R[1]);
      } else {
        if constexpr (H0) {
          bq_class<T, 0, -1, !TWO>(P, Qo, site, j, R);
          put(base + R0, -sgo, R[0]);
        }
        if constexpr (HD) {
          bq_class<T, 3, -1, true>(P, P, site, j, R);
          put(base + R3, -4 * sgp, R[0]);
        }
      }
      if constexpr (MES && (HD || !H0)) bq_mesons<0, 2>(P, site, j, put_meson);
    } else {
      if constexpr (HD) {
        bq_class<T, 1, 2, true>(P, P, site, j, R);
        put(base + R1, -4 * sgp, R[0]);
        put(base + R2, -4 * sgp, R[1]);
      }
      if constexpr (MES && (HD || !H0)) bq_mesons<2, 4>(P, site, j, put_meson);
      if constexpr (MES && H0 && !HD) bq_mesons<0, 4>(P, site, j, put_meson);
    }
  }
}

template <typename T, bool TWO, bool MES, int GM>
static int launch_baryon_t(const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out, int64_t V3,
                           int T_lat, int nch_total, int ch0, int tiles_per_block, hipStream_t st) {
  const int ntiles = (int)((V3 + 15) / 16);
  const int gx = (ntiles + tiles_per_block - 1) / tiles_per_block;
  dim3 grid((unsigned)gx, (unsigned)nrows), block(BqSplit<TWO, MES, GM>::threads);
  k_baryon<T, TWO, MES, GM><<<grid, block, 0, st>>>(props, rows, out, V3, T_lat, nch_total, ch0, ntiles);
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template <typename T>
int launch_baryon(bool two, bool mes, int gmask, const PropDev<T> *props, const RowDev *rows, int nrows,
                  cx<T> *out, int64_t V3, int T_lat, int nch_total, int ch0, int tiles_per_block,
                  hipStream_t st) {
#define PLG_B(TW, ME, GMV)                                                                       \
  if (two == TW && mes == ME && gmask == GMV)                                                    \
    return launch_baryon_t<T, TW, ME, GMV>(props, rows, nrows, out, V3, T_lat, nch_total, ch0,  \
                                           tiles_per_block, st);
  constexpr int NUC = 1, DEL = (1 << 7) | (1 << 8) | (1 << 9), ALL = NUC | DEL;
  PLG_B(true, false, NUC)
  PLG_B(true, false, DEL)
  PLG_B(true, false, ALL)
  PLG_B(false, false, NUC)
  PLG_B(false, false, DEL)
  PLG_B(false, false, ALL)
  PLG_B(false, true, 0)
  PLG_B(false, true, NUC)
  PLG_B(false, true, DEL)
  PLG_B(false, true, ALL)
#undef PLG_B
  return PLG_ERR_INVALID;
}

template int launch_baryon<double>(bool, bool, int, const PropDev<double> *, const RowDev *, int, cx<double> *,
                                   int64_t, int, int, int, int, hipStream_t);
template int launch_baryon<float>(bool, bool, int, const PropDev<float> *, const RowDev *, int, cx<float> *,
                                  int64_t, int, int, int, int, hipStream_t);

}  // namespace plg
