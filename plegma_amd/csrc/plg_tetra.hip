// plg_tetra.hip -- four-propagator table contractions (gfx950): the term
// sums of lib/kernels/PLEGMA_heavy_light_tetraquarks.cu:6-62,
//   O_k = sum_t v_t sum_{a0..a3} P1[i0][i1][a[c0]][a[c1]] P2[i2][i3][a[c2]][a[c3]]
//                 conj(P3[i5+2][i4+2][a[c5]][a[c4]]) conj(P4[i7+2][i6+2][a[c7]][a[c6]])
// (spin indices + 2 mod 4: the gamma5 of the backward propagators), for
// tables in the reference's format (8 spin indices, 8 colour slots, a float2
// per term).
//
// The reference sums the 81 colour assignments of every term.  Every term of
// its heavy-light tables has one of two colour structures, which close into
// colour traces of the 3x3 blocks B1 = P1[i0][i1], ..., B4 = P4[i7+2][i6+2]:
//   direct  (c0 = c5, c1 = c4, c2 = c7, c3 = c6):  <B1, B3> <B2, B4>,   <X, Y> = sum X conj(Y)
//   crossed (c0 = c5, c1 = c6, c2 = c7, c3 = c4):  Tr[(B3^dag B1)(B4^dag B2)]
// Terms that pair P1 with P4 and P2 with P3 instead (the bcud tables) close
// into the same two structures on the views P1, P2, P4, P3: a second set.
// The host classifies every term; a table with another structure is refused.
//
// Terms of one structure with the same four spin pairs are one product with a
// coefficient per operator: the 12.7 k terms of the heavy-light tables are
// 3648 products, the 63 k of the bcud table 10496.  With M = B3^dag B1 of the
// spin pairs p = (s1, s3), both structures are scalar products with B4:
//   crossed: <X, B4>, X = B2 M;    direct: <X, B4>, X = Tr(M) B2,
// so the products are walked as p, then s2 (X in registers), then s4.
#include "plg_internal.h"

#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <numeric>

namespace plg {

// A workgroup of 8 waves stages the four propagators of 16 consecutive sites
// in LDS, entries outermost (a row of 16 sites is 128 or 256 bytes).  The lane
// of site s and quarter q = lane / 16 takes its quarter's spin pairs of every
// step, so that the walk is uniform over the wave and a product's 64 values
// (16 sites, 4 sets of spin pairs) are, as they lie in the registers, the B
// operand of a 16x16x4 matrix product with the coefficients of 16 operators.
// A wave reads its walk 64 words at a time and hands them out by lane reads;
// the coefficients are loaded two products ahead.  The waves' sums meet in LDS
// at the end.
// Bound by the vector unit: M 108 FMAs, X 108 (crossed) or 36, a product 36
// and its matrix instructions.
// Of 2.7 M cycles on 16^3 x 24 sites with the udbb table, FP32, the FMAs take
// 1.5 M, the matrix instructions 0.35 M, LDS is busy 1.4 M.  Term by term from
// tables of B3^dag B1 and B4^dag B2 in LDS, a site at a time, the same took
// 3.65 ms, bound by the 160 bytes of LDS a term reads; this 1.15 ms.
// Entries that are not finite, and products that overflow, reach the operators
// that have a term with them at that site and no others, as term by term (SAFE
// below).
template <typename T> struct TtAcc;
template <> struct TtAcc<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  static __device__ __forceinline__ int slot(int k, int s) { return (k & 3) * 64 + (k >> 2) * 16 + s; }  // r * 64 + lane
};
template <> struct TtAcc<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
  static __device__ __forceinline__ int slot(int k, int s) { return (k >> 2) * 64 + (k & 3) * 16 + s; }
};

// NB: blocks of 16 operators
template <typename T, int NB>
__global__ __launch_bounds__(64 * TT_WAVES, sizeof(T) == 4 ? 4 : 2) void k_tetra(
    TetraSched S, const PropDev<T> *__restrict__ props, const RowDev *__restrict__ rows, cx<T> *__restrict__ out,
    int64_t V3, int T_lat, int nch_total, int ch0) {
  typedef typename TtAcc<T>::v4 v4;
  constexpr int NT = 64 * TT_WAVES;
  __shared__ cx<T> sp[4 * 144 * 16];  // [propagator][m01][a b][site]
  __shared__ T red[TT_WAVES][256];    // the waves' sums of 16 operators, real or imaginary
  const int tid = threadIdx.x, lane = tid & 63, s = tid & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const RowDev row = rows[blockIdx.y];
  const int64_t x0 = (int64_t)blockIdx.x * 16;
  T sg = 1;
  int rot_any = 0;
  {
    const bool xin = x0 + s < V3;
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const PropDev<T> Q = props[f];
      sg *= prop_sign(Q, row.t);
      rot_any |= Q.rot;
      int plane = row.t - Q.t_first;
      plane += plane < 0 ? T_lat : 0;
      const cx<T> *b = Q.data + (int64_t)plane * V3 + x0 + s;
#pragma unroll
      for (int i = 0; i < (144 * 16 + NT - 1) / NT; i++) {
        const int c = i * (NT / 16) + (tid >> 4);
        if (c < 144) sp[(f * 144 + c) * 16 + s] = xin ? gload(b + (int64_t)c * Q.cs) : cmake<T>(0, 0);
      }
    }
  }
  __syncthreads();
  if (rot_any) {  // rotation to the physical basis, per (site, propagator, colour pair)
    for (int k = tid; k < 4 * 9 * 16; k += NT) {
      const int f = k / 144, cc = (k >> 4) % 9, rot = props[f].rot;
      if (rot) {
        cx<T> *b = sp + (f * 144 + cc) * 16 + (k & 15);
        cx<T> w[16];
#pragma unroll
        for (int m = 0; m < 16; m++) w[m] = b[m * 9 * 16];
        rot_spins(w, rot);
#pragma unroll
        for (int m = 0; m < 16; m++) b[m * 9 * 16] = w[m];
      }
    }
    __syncthreads();
  }
  // the sums, and those of the last few products: sums of sums round less
  // than one long sum
  v4 tr[NB], ti[NB];
  // SAFE: values that are not finite stay out of the matrix products, where a
  // zero coefficient would spread them over the operators of a block, and go
  // one by one to those that have a coefficient, in spec
  T *spec = &red[0][0];  // [operator block][real, imaginary][as a wave's sums lie in red]
  static_assert(2 * NB <= TT_WAVES, "spec fits red");
  auto walk = [&](auto SAFE) {
    constexpr bool safe = SAFE.value;
    v4 ar[NB], ai[NB];
    int nsum = 0;
#pragma unroll
    for (int b = 0; b < NB; b++) tr[b] = ti[b] = ar[b] = ai[b] = (v4)(T)0;
    auto flush = [&]() {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        tr[b] += ar[b];
        ti[b] += ai[b];
        ar[b] = ai[b] = (v4)(T)0;
      }
      nsum = 0;
    };
    // the wave's words, 64 at a time and the next 64 on the way
    const uint32_t *wp = S.words + S.word0[wave] + lane;
    uint32_t wcur = wp[0], wnext = wp[64];
    int wpos = 0;
    auto word = [&]() -> uint32_t {
      if (wpos == 64) {
        wcur = wnext;
        wp += 64;
        wnext = wp[64];
        wpos = 0;
      }
      return (uint32_t)__builtin_amdgcn_readlane((int)wcur, wpos++);
    };
    const T *cp = (const T *)S.coef + (int64_t)S.coef0[wave] * 64 + lane;
    T c0 = cp[0], c1 = cp[64];
    cp += 128;
    for (int st = 0; st < S.nsteps[wave]; st++) {
      const uint32_t pw = word(), fw = word();
      const int p = (pw >> (8 * kq)) & 255;
      const cx<T> *P3 = sp + ((fw >> 16) & 1 ? 3 : 2) * 2304 + s, *P4 = sp + ((fw >> 16) & 1 ? 2 : 3) * 2304 + s;
      cx<T> m[9];  // (B3^dag B1)[z][y] at z * 3 + y
      {
        const cx<T> *A = sp + s + (p >> 4) * 144, *B = P3 + (p & 15) * 144;
        cx<T> a[9], b[9];
#pragma unroll
        for (int j = 0; j < 9; j++) {
          a[j] = A[j * 16];
          b[j] = B[j * 16];
        }
#pragma unroll
        for (int z = 0; z < 3; z++)
#pragma unroll
          for (int y = 0; y < 3; y++) {
            m[z * 3 + y] = cmake<T>(0, 0);
#pragma unroll
            for (int w = 0; w < 3; w++) cfma_conj(m[z * 3 + y], a[w * 3 + y], b[w * 3 + z]);
          }
      }
      const int ncr = fw & 255, ng = ncr + ((fw >> 8) & 255);
      for (int g = 0; g < ng; g++) {
        const uint32_t gw = word();
        cx<T> X[9];
        {
          const cx<T> *B2 = sp + 2304 + s + ((gw >> (4 * kq)) & 15) * 144;
          cx<T> b[9];
#pragma unroll
          for (int j = 0; j < 9; j++) b[j] = B2[j * 16];
          if (g < ncr) {
#pragma unroll
            for (int w = 0; w < 3; w++)
#pragma unroll
              for (int y = 0; y < 3; y++) {
                X[w * 3 + y] = cmake<T>(0, 0);
#pragma unroll
                for (int z = 0; z < 3; z++) cfma(X[w * 3 + y], b[w * 3 + z], m[z * 3 + y]);
              }
          } else {
            const cx<T> d = m[0] + m[4] + m[8];  // <B1, B3>
#pragma unroll
            for (int j = 0; j < 9; j++) X[j] = d * b[j];
          }
        }
        const int nt = (int)(gw >> 16);
        for (int e = 0; e < nt; e++) {
          const uint32_t uw = word();
          const cx<T> *B4 = P4 + ((uw >> (4 * kq)) & 15) * 144;
          cx<T> t = cmake<T>(0, 0);
#pragma unroll
          for (int j = 0; j < 9; j++) cfma_conj(t, X[j], B4[j * 16]);
          cx<T> u = cmake<T>(0, 0);  // what of t is not finite
          bool odd = false;
          if constexpr (safe) {
            const bool fr = __builtin_isfinite(t.re), fi = __builtin_isfinite(t.im);
            u = cmake<T>(fr ? (T)0 : t.re, fi ? (T)0 : t.im);
            t = cmake<T>(fr ? t.re : (T)0, fi ? t.im : (T)0);
            odd = __any(!fr || !fi);
          }
          // operators of block b that have a coefficient v: real sum += v re, imaginary sum += v im
          auto apart = [&](int b, T v, T re, T im) {
            const bool r = !__builtin_isfinite(re), i = !__builtin_isfinite(im);
            for (unsigned ops = (unsigned)(__ballot(v != 0) >> (16 * kq)) & 0xffff; __any(ops); ops &= ops - 1) {
              const int k = ops ? __ffs(ops) - 1 : 0;
              const T w = __shfl(v, 16 * kq + k);
              T *d = spec + 512 * b + TtAcc<T>::slot(k, s);
              if (ops && r) atomicAdd(d, w * re);
              if (ops && i) atomicAdd(d + 256, w * im);
            }
          };
          // O[k] += V[k] t in the operator blocks the products have coefficients in
#pragma unroll
          for (int b = 0; b < NB; b++)
            if (uw >> (16 + b) & 1) {
              const T v = c0;
              c0 = c1;
              c1 = *cp;
              cp += 64;
              ar[b] = TtAcc<T>::mma(v, t.re, ar[b]);
              ai[b] = TtAcc<T>::mma(v, t.im, ai[b]);
              if (safe && odd) apart(b, v, u.re, u.im);
            }
          if (uw >> 20) {
#pragma unroll
            for (int b = 0; b < NB; b++)
              if (uw >> (20 + b) & 1) {
                const T v = c0;
                c0 = c1;
                c1 = *cp;
                cp += 64;
                ar[b] = TtAcc<T>::mma(v, -t.im, ar[b]);
                ai[b] = TtAcc<T>::mma(v, t.re, ai[b]);
                if (safe && odd) apart(b, v, -u.im, u.re);
              }
          }
        }
        nsum += nt;
        if (nsum >= 6) flush();
      }
    }
    flush();
  };
  // the waves' sums: thread tid < 256 holds operator row(lane, wave) of every block at its site
  T o[NB][2];
  int *flag = (int *)spec;  // [256 / 64]: a sum of the wave is not finite, in the wave's own place of red
  auto reduce = [&]() {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave][r * 64 + lane] = h ? ti[b][r] : tr[b][r];
        __syncthreads();
        if (tid < 256) {
          T v[TT_WAVES];
#pragma unroll
          for (int w = 0; w < TT_WAVES; w++) v[w] = red[w][tid];
#pragma unroll
          for (int n = TT_WAVES / 2; n > 0; n /= 2)  // pairwise
#pragma unroll
            for (int w = 0; w < n; w++) v[w] += v[w + n];
          o[b][h] = v[0];
          if (h == 1 && b + 1 == NB) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < NB; i++) bad = bad || !__builtin_isfinite(o[i][0]) || !__builtin_isfinite(o[i][1]);
            const int mine = __any(bad);
            if (lane == 0) flag[(int)(sizeof(T) / 4) * tid] = mine;
          }
        }
        __syncthreads();
      }
  };
  walk(std::false_type{});
  reduce();
  {
    // a sum that is not finite: its tile again, with the care of SAFE
    int any = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) any |= flag[(int)(sizeof(T) / 4) * 64 * w];
    if (__builtin_amdgcn_readfirstlane(any)) {
      __syncthreads();
      for (int i = tid; i < 512 * NB; i += NT) spec[i] = 0;
      __syncthreads();
      walk(std::true_type{});
      __syncthreads();
      T apart[NB][2];
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int h = 0; h < 2; h++) apart[b][h] = spec[512 * b + 256 * h + (tid & 255)];
      __syncthreads();
      reduce();
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int h = 0; h < 2; h++) o[b][h] += apart[b][h];
    }
  }
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total + ch0;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int k = 16 * b + TtAcc<T>::row(lane, wave);
    if (tid < 256 && k < S.nops && x0 + s < V3)
      gstore(out + ctile_idx(col0 + k, x0 + s, ncols), cmake<T>(sg * o[b][0], sg * o[b][1]));
  }
}

template <typename T>
int launch_tetra(const TetraSched &S, const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out,
                 int64_t V3, int T_lat, int nch_total, int ch0, hipStream_t st) {
  dim3 block(64 * TT_WAVES), grid((unsigned)((V3 + 15) / 16), (unsigned)nrows);
  switch ((S.nops + 15) / 16) {
  case 1: k_tetra<T, 1><<<grid, block, 0, st>>>(S, props, rows, out, V3, T_lat, nch_total, ch0); break;
  case 2: k_tetra<T, 2><<<grid, block, 0, st>>>(S, props, rows, out, V3, T_lat, nch_total, ch0); break;
  default: return PLG_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template int launch_tetra<double>(const TetraSched &, const PropDev<double> *, const RowDev *, int, cx<double> *,
                                  int64_t, int, int, int, hipStream_t);
template int launch_tetra<float>(const TetraSched &, const PropDev<float> *, const RowDev *, int, cx<float> *,
                                 int64_t, int, int, int, hipStream_t);

// the walk of operators k0 .. k0 + nops - 1: its steps by wave
struct TetraWalk {
  // per (set, p): its groups of one structure and s2, most products first
  struct Group {
    int s2;
    std::vector<std::pair<int, int>> e;  // s4, product
  };
  struct Item {
    int p;
    std::array<std::vector<Group>, 2> g;  // crossed, direct
    std::vector<int> sig;
    int n = 0;
  };
  struct Step {
    int set;
    std::array<const Item *, 4> it;
    int cost;
  };
  int k0, nops;
  std::vector<uint8_t> mask;  // of a product: operator blocks with a real (bits 0-3) and an imaginary (4-7) coefficient
  std::array<std::vector<Item>, 2> items;
  std::vector<Step> steps;
  std::array<std::vector<const Step *>, TT_WAVES> mine;
  TetraWalk(const TetraProds &P, int k0, int nops);
  TetraWalk(const TetraWalk &) = delete;  // steps point at items
  // the groups of a structure of a step, four quarters each (NULL: none), and the products of a group
  static size_t groups(const Step &st, int ty) {
    size_t n = 0;
    for (const Item *I : st.it) n = I ? std::max(n, I->g[ty].size()) : n;
    return n;
  }
  static std::array<const Group *, 4> group(const Step &st, int ty, size_t g) {
    std::array<const Group *, 4> G;
    for (int j = 0; j < 4; j++) G[j] = st.it[j] && g < st.it[j]->g[ty].size() ? &st.it[j]->g[ty][g] : nullptr;
    return G;
  }
  static size_t products(const std::array<const Group *, 4> &G) {
    size_t n = 0;
    for (const Group *q : G) n = q ? std::max(n, q->e.size()) : n;
    return n;
  }
  uint32_t blocks(const std::array<const Group *, 4> &G, size_t e) const {
    uint32_t m = 0;
    for (const Group *q : G) m |= q && e < q->e.size() ? mask[q->e[e].second] : 0;
    return m;
  }
};

TetraWalk::TetraWalk(const TetraProds &P, int k0, int nops) : k0(k0), nops(nops), mask(P.prods.size(), 0) {
  std::vector<uint8_t> used(P.prods.size(), 0);
  for (size_t i = 0; i < P.prods.size(); i++)
    for (const auto &kv : P.prods[i].v) {
      const int k = kv.first - k0;
      if (k < 0 || k >= nops) continue;
      used[i] = 1;
      for (int h = 0; h < 2; h++)
        if (kv.second[h] != 0) mask[i] |= 1u << (4 * h + k / 16);
    }
  for (int set = 0; set < 2; set++) {
    for (int p = 0; p < 256; p++) {
      Item I;
      I.p = p;
      for (int ty = 0; ty < 2; ty++) {
        const int *ix = &P.index[set << 17 | ty << 16 | p << 8];
        for (int s2 = 0; s2 < 16; s2++) {
          Group G;
          G.s2 = s2;
          for (int s4 = 0; s4 < 16; s4++) {
            const int id = ix[s2 * 16 + s4];
            if (id >= 0 && used[id]) G.e.push_back({s4, id});
          }
          I.n += (int)G.e.size();
          if (!G.e.empty()) I.g[ty].push_back(std::move(G));
        }
        std::stable_sort(I.g[ty].begin(), I.g[ty].end(),
                         [](const Group &a, const Group &b) { return a.e.size() > b.e.size(); });
        for (const Group &G : I.g[ty]) I.sig.push_back((int)G.e.size());
        I.sig.push_back(0);
      }
      if (I.n) items[set].push_back(std::move(I));
    }
    // steps of four spin pairs p with like groups
    std::stable_sort(items[set].begin(), items[set].end(),
                     [](const Item &a, const Item &b) { return a.n != b.n ? a.n > b.n : a.sig > b.sig; });
    for (size_t i = 0; i < items[set].size(); i += 4) {
      Step st;
      st.set = set;
      st.cost = 4;
      for (size_t j = 0; j < 4; j++) {
        st.it[j] = i + j < items[set].size() ? &items[set][i + j] : nullptr;
        if (st.it[j])
          st.cost = std::max(st.cost, 4 + 2 * st.it[j]->n + 4 * (int)st.it[j]->g[0].size() + 2 * (int)st.it[j]->g[1].size());
      }
      steps.push_back(st);
    }
  }
  std::stable_sort(steps.begin(), steps.end(), [](const Step &a, const Step &b) { return a.cost > b.cost; });
  std::array<int, TT_WAVES> load{};
  for (const Step &st : steps) {
    const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[w] += st.cost;
    mine[w].push_back(&st);
  }
}

void tetra_pack(const TetraProds &P, const TetraWalks &walks, std::vector<TetraPacked> &outs) {
  outs.clear();
  for (const auto &walk : walks) {
    const TetraWalk &W = *walk;
    outs.emplace_back();
    TetraPacked &out = outs.back();
    for (int w = 0; w < TT_WAVES; w++) {
      out.s.word0[w] = (int)out.words.size();
      out.s.coef0[w] = (int)(out.coef.size() / 64);
      out.s.nsteps[w] = (int)W.mine[w].size();
      for (const TetraWalk::Step *st : W.mine[w]) {
        uint32_t pw = 0;
        for (int j = 0; j < 4; j++)
          if (st->it[j]) pw |= (uint32_t)st->it[j]->p << (8 * j);
        const size_t ng[2] = {TetraWalk::groups(*st, 0), TetraWalk::groups(*st, 1)};
        out.words.push_back(pw);
        out.words.push_back((uint32_t)ng[0] | (uint32_t)ng[1] << 8 | (uint32_t)st->set << 16);
        for (int ty = 0; ty < 2; ty++)
          for (size_t g = 0; g < ng[ty]; g++) {
            const auto G = TetraWalk::group(*st, ty, g);
            const size_t nt = TetraWalk::products(G);
            uint32_t gw = (uint32_t)nt << 16;
            for (int j = 0; j < 4; j++)
              if (G[j]) gw |= (uint32_t)G[j]->s2 << (4 * j);
            out.words.push_back(gw);
            for (size_t e = 0; e < nt; e++) {
              const uint32_t m = W.blocks(G, e);
              uint32_t uw = m << 16;
              for (int j = 0; j < 4; j++)
                if (G[j] && e < G[j]->e.size()) uw |= (uint32_t)G[j]->e[e].first << (4 * j);
              // a coefficient vector of 64, [quarter][operator of the block], per block of the word
              double *V[8];
              size_t at = out.coef.size();
              out.coef.resize(at + 64 * (size_t)__builtin_popcount(m), 0.0);
              for (int b = 0; b < 8; b++) {
                V[b] = m >> b & 1 ? &out.coef[at] : nullptr;
                at += m >> b & 1 ? 64 : 0;
              }
              for (int j = 0; j < 4; j++) {
                if (!G[j] || e >= G[j]->e.size()) continue;
                for (const auto &kv : P.prods[G[j]->e[e].second].v) {
                  const int k = kv.first - W.k0;
                  if (k < 0 || k >= W.nops) continue;
                  for (int h = 0; h < 2; h++)
                    if (double *v = V[4 * h + k / 16]) v[16 * j + k % 16] = kv.second[h];
                }
              }
              out.words.push_back(uw);
            }
          }
      }
      out.words.resize((out.words.size() + 63) / 64 * 64 + 128, 0u);  // the reads ahead
    }
    out.coef.resize(out.coef.size() + 3 * 64, 0.0);
    out.s.nops = W.nops;
  }
}

// The walk against the terms one by one (plg_tetra_terms.hip), fitted to
// calls with 60 tables -- 1 to 64 operators of 40 to 4 000 terms, real and
// complex coefficients, few and many shared products -- on 4 096 to 221 184
// sites.  Microseconds of as many workgroups as the chip holds:
//   walk   12 and 0.87 per thousand FMAs of a lane, a matrix instruction counted as 26
//   terms  195, and per operator of the wave with most of them 73, 11.6 per 64
//          direct and 18.4 (FP64 23.6) per 64 crossed terms
// (measured walk / terms in ms: the udbb table 1.2 / 3.7 on 98 304 sites; 16
// operators of 768 random complex terms in FP32 7.8 / 6.6 on 221 184 sites, 0.72
// / 0.98 on 13 824; in FP64 15.0 / 13.0 and 1.22 / 1.03; 64 operators of 40
// terms 1.5 / 6.4 on 110 592).  The walk has to be the faster by 1.25, about
// the error of the fit: so none of those calls is slower than term by term,
// and the choice is within 1.25 of the better form.
TetraCost tetra_cost(const TetraProds &P, int per, bool f64, TetraWalks &walks) {
  TetraCost c;
  c.slots = f64 ? 256 : 512;
  for (int k0 = 0; k0 < P.nops; k0 += per) {
    walks.push_back(std::make_shared<const TetraWalk>(P, k0, std::min(per, P.nops - k0)));
    const TetraWalk &W = *walks.back();
    int64_t fma = 0;
    for (const TetraWalk::Step &st : W.steps) {
      fma += 108;
      for (int ty = 0; ty < 2; ty++)
        for (size_t g = 0; g < TetraWalk::groups(st, ty); g++) {
          const auto G = TetraWalk::group(st, ty, g);
          const size_t nt = TetraWalk::products(G);
          fma += ty ? 36 : 108;
          for (size_t e = 0; e < nt; e++) fma += 36 + 26 * __builtin_popcount(W.blocks(G, e));
        }
    }
    c.walk += 12 + 0.87e-3 * (double)fma;
  }
  for (int set = 0; set < 2; set++) {
    double wave[4] = {0, 0, 0, 0};
    bool any = set == 0;
    for (int k = 0; k < P.nops; k++) {
      const auto &n = P.terms[set][k];
      any = any || n[0] + n[1] > 0;
      wave[k % 4] += 73 + 11.6 * ((n[1] + 63) / 64) + (f64 ? 23.6 : 18.4) * ((n[0] + 63) / 64);
    }
    if (any) c.terms += 195 + *std::max_element(wave, wave + 4);
  }
  return c;
}

bool tetra_by_terms(const TetraCost &c, int64_t V3, int64_t nrows) {
  auto rounds = [&](int64_t sites) { return (double)(((V3 + sites - 1) / sites * nrows + c.slots - 1) / c.slots); };
  return rounds(64) * c.terms < 1.25 * rounds(16) * c.walk;
}

// host: the terms of a table (reference format) by product
int tetra_products(const int16_t *idxs, const int16_t *cols, const float *vals, const int16_t *counts, int nops,
                   TetraProds &out) {
  if (nops <= 0 || nops > TETRA_MAXOPS) return PLG_ERR_UNSUPPORTED;
  std::map<std::pair<uint32_t, uint32_t>, int> cidx;  // distinct coefficients, zero among them
  cidx.emplace(std::make_pair(0u, 0u), 0);
  out = TetraProds{};
  out.nops = nops;
  out.index.assign(1 << 18, -1);
  for (auto &v : out.terms) v.assign(nops, {0, 0});
  size_t t = 0;
  for (int k = 0; k < nops; k++) {
    if (counts[k] < 0) return PLG_ERR_INVALID;
    for (int i = 0; i < counts[k]; i++, t++) {
      const int16_t *m = idxs + 8 * t, *c = cols + 8 * t;
      for (int j = 0; j < 8; j++)
        if (m[j] < 0 || m[j] > 3 || c[j] < 0 || c[j] > 3) return PLG_ERR_INVALID;
      bool perm = true;  // c0..c3 a permutation of the four colour sums
      for (int a = 0; a < 4; a++)
        for (int b = a + 1; b < 4; b++) perm &= c[a] != c[b];
      if (!perm) return PLG_ERR_UNSUPPORTED;
      const int s1 = m[0] * 4 + m[1], s2 = m[2] * 4 + m[3];
      const int s3 = ((m[5] + 2) & 3) * 4 + ((m[4] + 2) & 3), s4 = ((m[7] + 2) & 3) * 4 + ((m[6] + 2) & 3);
      uint32_t re, im;
      std::memcpy(&re, vals + 2 * t, 4);
      std::memcpy(&im, vals + 2 * t + 1, 4);
      if (cidx.emplace(std::make_pair(re, im), 0).second && (int)cidx.size() > TETRA_MAXCOEF)
        return PLG_ERR_UNSUPPORTED;
      // set 0 on (P1, P2, P3, P4); set 1 on (P1, P2, P4, P3): P4's spin pair
      // takes the third place and P3's the fourth
      const int u0 = (s1 * 16 + s3) << 8 | (s2 * 16 + s4), u1 = (s1 * 16 + s4) << 8 | (s2 * 16 + s3);
      int key;
      if (c[0] == c[5] && c[1] == c[4] && c[2] == c[7] && c[3] == c[6]) key = 1 << 16 | u0;
      else if (c[0] == c[5] && c[1] == c[6] && c[2] == c[7] && c[3] == c[4]) key = u0;
      else if (c[0] == c[7] && c[1] == c[6] && c[2] == c[5] && c[3] == c[4]) key = 3 << 16 | u1;
      else if (c[0] == c[7] && c[1] == c[4] && c[2] == c[5] && c[3] == c[6]) key = 2 << 16 | u1;
      else return PLG_ERR_UNSUPPORTED;
      out.terms[key >> 17][k][key >> 16 & 1]++;
      if (out.index[key] < 0) {
        out.index[key] = (int)out.prods.size();
        out.prods.emplace_back();
      }
      auto &v = out.prods[out.index[key]].v;
      if (v.empty() || v.back().first != k) v.push_back({k, {0.0, 0.0}});
      v.back().second[0] += (double)vals[2 * t];
      v.back().second[1] += (double)vals[2 * t + 1];
    }
  }
  return PLG_OK;
}

}  // namespace plg
