// plg_udsc.hip -- the udsc baryon two-point functions (gfx950), the table-
// driven three-propagator contraction of lib/kernels/PLEGMA_baryons_udsc.cu:
//   O_k(x) = sum_t v_kt sum_{eps, eps'} sgn sgn' S1[m0][m1][a][a'] S2[m2][m3][b][b'] S3[m4][m5][c][c']
// with the term tables of plg_udsc_tables.h (generated from the interpolating
// fields by plegma_amd/gen_udsc.py).
//
// The reference gives every site one thread that walks all terms with its
// three propagators in registers (PLEGMA_baryons_udsc.cu:86-121).  Here the
// terms are factorised through the colour "diquark" of two of the propagators:
//   D_q[c][c'] = sum eps_abc eps_a'b'c' S1[m0m1][a][a'] S2[m2m3][b][b']   (q = m0m1, m2m3)
//   T_m        = sum_cc' D_q[c][c'] S3[m4m5][c][c']                     (distinct terms m)
//   O_k        = sum_m v_km T_m
// The built-in products of a call share one launch (k_udsc_all, below).  A
// caller's table (k_udsc): one wave works on one site at a time with the
// site's 432 propagator entries in LDS; quads are processed in chunks of 64,
// one per lane: the lane forms D_q in registers and the (at most four)
// distinct terms of its quad, which go to LDS slots; then each operator sums
// its entries over those slots (4 lanes per operator).  D costs 36 complex products per quad, a term 9, an entry 1.
// A workgroup stages whole 128-byte lines of the propagators (16 FP32 or 8
// FP64 consecutive sites), so every line is read from HBM once.
#include "plg_internal.h"
#include "plg_udsc_tables.h"

#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace plg {

// ------------------------------------------------------------------ schedule
// host: the chunked schedule of nops operators, operator k being the terms
// [first[k], first[k] + count[k]) of `terms`
int udsc_schedule_terms(const UdscTerm *terms, const int *first, const int *count, int nops, UdscSchedHost &h) {
  if (nops <= 0 || nops > UD_MAXOPS) return PLG_ERR_UNSUPPORTED;
  auto key6 = [](const UdscTerm &t) {
    int k = 0;
    for (int i = 0; i < 6; i++) k = k * 4 + t.m[i];
    return k;
  };
  auto quad_of = [](int k6) {  // m01 | m23 << 4
    const int m0 = (k6 >> 10) & 3, m1 = (k6 >> 8) & 3, m2 = (k6 >> 6) & 3, m3 = (k6 >> 4) & 3;
    return (m0 * 4 + m1) | ((m2 * 4 + m3) << 4);
  };
  for (int k = 0; k < nops; k++)
    for (int i = 0; i < count[k]; i++)
      for (int j = 0; j < 6; j++)
        if (terms[first[k] + i].m[j] < 0 || terms[first[k] + i].m[j] > 3) return PLG_ERR_INVALID;
  // distinct terms grouped by quad
  std::map<int, std::vector<int>> by_quad;  // quad -> distinct key6 terms
  for (int k = 0; k < nops; k++)
    for (int i = 0; i < count[k]; i++) {
      const int k6 = key6(terms[first[k] + i]);
      auto &v = by_quad[quad_of(k6)];
      if (std::find(v.begin(), v.end(), k6) == v.end()) v.push_back(k6);
    }
  std::vector<int> quads;
  for (auto &kv : by_quad) {
    if ((int)kv.second.size() > UD_TPQ) return PLG_ERR_UNSUPPORTED;
    quads.push_back(kv.first);
  }
  // quads with the most distinct terms first: a wave runs the term loop of a
  // chunk as often as its fullest quad needs, so the later chunks run fewer
  std::sort(quads.begin(), quads.end(), [&](int a, int b) {
    const size_t na = by_quad[a].size(), nb = by_quad[b].size();
    if (na != nb) return na > nb;
    return (a & 15) != (b & 15) ? (a & 15) < (b & 15) : (a >> 4) < (b >> 4);
  });
  const int nch = std::max(1, ((int)quads.size() + 63) / 64);
  if (nch > UD_MAXC) return PLG_ERR_UNSUPPORTED;
  std::map<int, std::pair<int, int>> slot;  // key6 -> (chunk, chunk-local slot)
  h = UdscSchedHost{};
  h.s.nops = nops;
  h.s.nchunks = nch;
  h.quads.assign((size_t)nch * 64, (short)-1);
  h.tp.assign((size_t)nch * 64 * UD_TPQ, (signed char)-1);
  for (size_t i = 0; i < quads.size(); i++) {
    const int c = (int)i / 64, l = (int)i % 64;
    h.quads[i] = (short)quads[i];
    const auto &v = by_quad[quads[i]];
    h.s.ntp[c] = std::max(h.s.ntp[c], (int)v.size());
    for (size_t e = 0; e < v.size(); e++) {
      h.tp[i * UD_TPQ + e] = (signed char)((v[e] >> 2 & 3) * 4 + (v[e] & 3));
      slot[v[e]] = {c, (int)e * 64 + l};  // term-major: a wave's 64 writes hit distinct banks
    }
  }
  // each operator's entries per chunk: slot | coefficient index << 8
  std::map<std::pair<float, float>, int> cix;
  h.coef = {0.f, 0.f};
  cix[{0.f, 0.f}] = 0;
  h.s.real_coef = 1;
  std::vector<std::vector<std::vector<uint16_t>>> lists(nch, std::vector<std::vector<uint16_t>>(nops));
  for (int k = 0; k < nops; k++)
    for (int i = 0; i < count[k]; i++) {
      const UdscTerm &t = terms[first[k] + i];
      const auto &sl = slot[key6(t)];
      auto it = cix.find({t.re, t.im});
      if (it == cix.end()) {
        if ((int)h.coef.size() / 2 >= UD_MAXCOEF) return PLG_ERR_UNSUPPORTED;
        it = cix.insert({{t.re, t.im}, (int)h.coef.size() / 2}).first;
        h.coef.push_back(t.re);
        h.coef.push_back(t.im);
        if (t.im != 0.f) h.s.real_coef = 0;
      }
      lists[sl.first][k].push_back((uint16_t)(sl.second | (it->second << 8)));
    }
  // lanes per operator: one each, then one at a time to the operator whose
  // extra lane lowers the blocks summed over the chunks the most (a chunk
  // takes as many blocks as its longest lane list)
  auto blocks = [&](const std::vector<int> &L) {
    int tot = 0;
    for (int c = 0; c < nch; c++) {
      int m = 0;
      for (int k = 0; k < nops; k++) {
        const int per = ((int)lists[c][k].size() + L[k] - 1) / L[k];
        m = std::max(m, (per + 3) / 4);
      }
      tot += m;
    }
    return tot;
  };
  std::vector<int> L(nops, 1), tot_ent(nops, 0);
  for (int c = 0; c < nch; c++)
    for (int k = 0; k < nops; k++) tot_ent[k] += (int)lists[c][k].size();
  for (int extra = 0; extra < 64 - nops; extra++) {
    int best_k = 0, best_b = 1 << 30;
    double best_load = -1;
    for (int k = 0; k < nops; k++) {
      L[k]++;
      const int bl = blocks(L);
      const double load = (double)tot_ent[k] / L[k];
      L[k]--;
      if (bl < best_b || (bl == best_b && load > best_load)) {
        best_b = bl;
        best_load = load;
        best_k = k;
      }
    }
    L[best_k]++;
  }
  for (int k = 0, lo = 0; k < nops; k++) {
    h.s.op_lo[k] = lo;
    h.s.op_n[k] = L[k];
    lo += L[k];
  }
  // blocks: [block][lane][4]; operator k's list split into L[k] contiguous
  // shares of near-equal length, one per lane
  int nblk_tot = 0;
  for (int c = 0; c < nch; c++) {
    std::vector<std::vector<uint16_t>> lane(64);
    int nb = 0;
    for (int k = 0; k < nops; k++) {
      const auto &v = lists[c][k];
      const int n = (int)v.size();
      for (int r = 0; r < L[k]; r++) {
        auto &ln = lane[h.s.op_lo[k] + r];
        for (int i = r * n / L[k]; i < (r + 1) * n / L[k]; i++) ln.push_back(v[i]);
        nb = std::max(nb, ((int)ln.size() + 3) / 4);
      }
    }
    h.s.blk0[c] = nblk_tot;
    h.s.nblk[c] = nb;
    nblk_tot += nb;
    if (nblk_tot > UD_MAXBLK) return PLG_ERR_UNSUPPORTED;
    for (int b = 0; b < nb; b++)
      for (int l = 0; l < 64; l++)
        for (int j = 0; j < 4; j++) {
          const size_t e = (size_t)b * 4 + j;
          h.ents.push_back(e < lane[l].size() ? lane[l][e] : (uint16_t)0);
        }
  }
  h.s.nent = (int)h.ents.size();
  h.s.ncoef = (int)h.coef.size() / 2;
  if (h.s.nent > UD_MAXENT || h.s.ncoef > UD_MAXCOEF) return PLG_ERR_UNSUPPORTED;
  return PLG_OK;
}

// ------------------------------------------------------------------ built-in products
// The flavour products of one call, grouped by the pair of propagators whose
// colour diquarks they share.  The colour structure is symmetric under an
// exchange of the three propagators with their spin pairs, so a product may
// take any two of its flavours as the pair:
//  - two equal flavours are the pair (uuc, uud, uus and uuu share the diquarks
//    of uu), and D of the spin pairs (a, b) equals D of (b, a): 136 quads
//    instead of 256, and terms that differ by the exchange are one term (uuu:
//    by all exchanges of the three);
//  - of three different flavours u, d if both are there, else s, c (udc and
//    uds share ud; usc and dsc share sc).
// All 20 products: 1056 quads and 8.7 k terms instead of 4928 and 12.1 k.
int udsc_groups(const std::vector<int> &prods, const int fidx[4], UdscAllHost &h) {
  static const char letters[5] = "udsc";
  struct Key {
    int a, b;
    bool operator<(const Key &o) const { return a != o.a ? a < o.a : b < o.b; }
  };
  struct Item {
    int prod, third, perm[3], ch0;
  };
  std::map<Key, std::vector<Item>> by_pair;
  int ch = 0;
  for (int prod : prods) {
    const char *f = UDSC_PRODS[prod].flavours;
    Item it;
    it.prod = prod;
    it.ch0 = ch;
    ch += UDSC_PRODS[prod].nops;
    int x = 0, y = 1;  // the positions of the pair
    if (f[0] == f[1]) x = 0, y = 1;
    else if (f[1] == f[2]) x = 1, y = 2;
    else if (f[0] == f[2]) x = 0, y = 2;
    else {
      const std::string fs(f, 3);
      const bool ud = fs.find('u') != std::string::npos && fs.find('d') != std::string::npos;
      x = (int)fs.find(ud ? 'u' : 's');
      y = (int)fs.find(ud ? 'd' : 'c');
    }
    const int z = 3 - x - y;
    it.perm[0] = x;
    it.perm[1] = y;
    it.perm[2] = z;
    auto fl = [&](int i) { return fidx[std::strchr(letters, f[i]) - letters]; };
    it.third = fl(z);
    by_pair[Key{fl(x), fl(y)}].push_back(it);
  }
  h = UdscAllHost{};
  for (auto &kv : by_pair) {
    if ((int)kv.second.size() > UD_NJ || h.s.ngroups >= UD_MAXGROUPS) return PLG_ERR_UNSUPPORTED;
    UdscGroup &G = h.s.g[h.s.ngroups++];
    G.pa = kv.first.a;
    G.pb = kv.first.b;
    G.nprod = (int)kv.second.size();
    // quad -> per product: spin pair of the third propagator -> coefficient of every operator
    typedef std::map<int, std::array<double, UD_MAXOPS>> Terms;
    std::map<int, std::array<Terms, UD_NJ>> quads;
    for (int j = 0; j < G.nprod; j++) {
      const Item &it = kv.second[j];
      const UdscProd &P = UDSC_PRODS[it.prod];
      if (P.nops > UD_MAXOPS) return PLG_ERR_UNSUPPORTED;
      G.third[j] = it.third;
      G.nops[j] = P.nops;
      G.ch0[j] = it.ch0;
      for (int k = 0; k < P.nops; k++) {
        const UdscOp &op = UDSC_OPS[P.first_op + k];
        for (int i = 0; i < op.count; i++) {
          const UdscTerm &t = UDSC_TERMS[op.first + i];
          if (t.im != 0.f) return PLG_ERR_UNSUPPORTED;
          int sp[3];
          for (int v = 0; v < 3; v++) sp[v] = t.m[2 * it.perm[v]] * 4 + t.m[2 * it.perm[v] + 1];
          if (G.pa == G.pb) {
            if (it.third == G.pa) std::sort(sp, sp + 3);
            else if (sp[0] > sp[1]) std::swap(sp[0], sp[1]);
          }
          auto &T = quads[sp[0] | sp[1] << 4][j];
          auto e = T.emplace(sp[2], std::array<double, UD_MAXOPS>{}).first;
          e->second[k] += (double)t.re;
        }
      }
    }
    for (auto &q : quads)  // terms whose coefficients cancelled
      for (auto &T : q.second)
        for (auto e = T.begin(); e != T.end();)
          e = std::all_of(e->second.begin(), e->second.end(), [](double v) { return v == 0; }) ? T.erase(e)
                                                                                              : std::next(e);
    // the spin pairs of the third propagator a quad has terms with, per product
    typedef std::pair<const int, std::array<Terms, UD_NJ>> Quad;
    struct Item {  // the quads of a quarter of a step: one, or two that share reads of the third propagator
      const Quad *q[2];
      std::array<uint32_t, UD_NJ> set;
      int n;
    };
    auto sets = [](const Quad &q) {
      std::array<uint32_t, UD_NJ> m{};
      for (int j = 0; j < UD_NJ; j++)
        for (auto &e : q.second[j]) m[j] |= 1u << e.first;
      return m;
    };
    auto count = [](const std::array<uint32_t, UD_NJ> &m) {
      int n = 0;
      for (uint32_t v : m) n += __builtin_popcount(v);
      return n;
    };
    std::vector<Item> single, pairs;
    for (const Quad &q : quads) {
      const auto m = sets(q);
      single.push_back({{&q, nullptr}, m, count(m)});
    }
    auto more = [](const Item &x, const Item &y) { return x.n != y.n ? x.n > y.n : x.set > y.set; };
    std::stable_sort(single.begin(), single.end(), more);
    // as many steps of two as leave the waves even: whole rounds of the
    // waves, then two quads per quarter where the rest exceeds one round
    const int half = ((int)single.size() + 3) / 4, rest = half % (2 * UD_WAVES);
    const size_t npairs = 4 * (size_t)((half - rest) / 2 + (rest > UD_WAVES ? rest / 2 : 0));
    while (pairs.size() < npairs && single.size() > 1) {
      // the quad with most terms and the one that shares most of its spin pairs
      size_t best = 1;
      int bw = 1 << 30;
      for (size_t i = 1; i < single.size(); i++) {
        std::array<uint32_t, UD_NJ> u;
        for (int j = 0; j < UD_NJ; j++) u[j] = single[0].set[j] | single[i].set[j];
        const int waste = 2 * count(u) - single[0].n - single[i].n;
        if (waste < bw) {
          bw = waste;
          best = i;
        }
      }
      Item P = single[0];
      P.q[1] = single[best].q[0];
      for (int j = 0; j < UD_NJ; j++) P.set[j] |= single[best].set[j];
      P.n = count(P.set);
      pairs.push_back(P);
      single.erase(single.begin() + best);
      single.erase(single.begin());
    }
    std::stable_sort(pairs.begin(), pairs.end(), more);
    // steps of four items, to the wave with the least work so far
    struct Step {
      const Item *it[4];
      int cnt[UD_NJ];
      int cost;
      bool two;
    };
    std::vector<Step> steps;
    for (int two = 1; two >= 0; two--) {
      const std::vector<Item> &v = two ? pairs : single;
      for (size_t i = 0; i < v.size(); i += 4) {
        Step S{};
        S.two = two;
        S.cost = two ? 9 : 5;  // a diquark costs four terms, and its loads
        for (size_t k = 0; k < 4; k++) S.it[k] = i + k < v.size() ? &v[i + k] : nullptr;
        for (int j = 0; j < UD_NJ; j++) {
          for (int k = 0; k < 4; k++)
            if (S.it[k]) S.cnt[j] = std::max(S.cnt[j], __builtin_popcount(S.it[k]->set[j]));
          S.cost += S.cnt[j] * (two ? 2 : 1);
        }
        steps.push_back(S);
      }
    }
    std::vector<std::vector<const Step *>> mine(UD_WAVES);
    int load[UD_WAVES] = {0};
    for (const Step &S : steps) {
      const int w = (int)(std::min_element(load, load + UD_WAVES) - load);
      load[w] += S.cost;
      mine[w].push_back(&S);  // steps of two first, as they come
    }
    for (int w = 0; w < UD_WAVES; w++) {
      G.step0[w] = (int)h.steps.size() / 3;
      G.nsteps[w] = (int)mine[w].size();
      G.npair[w] = (int)std::count_if(mine[w].begin(), mine[w].end(), [](const Step *S) { return S->two; });
      G.unit0[w] = (int)h.units.size() / 2;
      G.coef0[w] = (int)h.coef.size() / 256;
      for (const Step *S : mine[w]) {
        uint32_t qw[2] = {0, 0}, cw = 0;
        for (int i = 0; i < 4; i++)
          for (int b = 0; b < 2; b++)
            if (S->it[i] && S->it[i]->q[b]) qw[b] |= (uint32_t)S->it[i]->q[b]->first << (8 * i);
        for (int j = 0; j < UD_NJ; j++) cw |= (uint32_t)S->cnt[j] << (8 * j);
        h.steps.insert(h.steps.end(), {qw[0], qw[1], cw});
        for (int j = 0; j < UD_NJ; j++)
          for (int e0 = 0; e0 < S->cnt[j]; e0 += 4) {  // a unit: four terms of each quarter's quads
            uint64_t pw = 0;
            const size_t c0 = h.coef.size();
            h.coef.resize(c0 + (S->two ? 512 : 256), 0.0);
            for (int i = 0; i < 4; i++) {
              if (!S->it[i]) continue;
              int u = 0;  // the quarter's spin pairs in order
              for (int sp = 0; sp < 16; sp++) {
                if (!(S->it[i]->set[j] >> sp & 1)) continue;
                if (u >= e0 && u < e0 + 4) {
                  pw |= (uint64_t)sp << (16 * i + 4 * (u - e0));
                  for (int b = 0; b < 2; b++) {
                    if (!S->it[i]->q[b]) continue;
                    auto e = S->it[i]->q[b]->second[j].find(sp);
                    if (e == S->it[i]->q[b]->second[j].end()) continue;
                    for (int k = 0; k < UD_MAXOPS; k++)
                      h.coef[c0 + b * 256 + (i * 16 + k) * 4 + (u - e0)] = e->second[k];
                  }
                }
                u++;
              }
            }
            h.units.push_back((uint32_t)pw);
            h.units.push_back((uint32_t)(pw >> 32));
          }
      }
    }
  }
  // the kernel loads a wave's next unit ahead of its use
  h.units.resize(h.units.size() + 2, 0u);
  h.coef.resize(h.coef.size() + 4 * 256, 0.0);
  return PLG_OK;
}

int udsc_products() { return UDSC_NPROD; }
const char *udsc_flavours(int prod) { return UDSC_PRODS[prod].flavours; }
int udsc_nops(int prod) { return UDSC_PRODS[prod].nops; }
const char *udsc_op_name(int prod, int k) { return UDSC_OPS[UDSC_PRODS[prod].first_op + k].name; }

// ------------------------------------------------------------------ kernel
// A workgroup of W waves stages the three propagators of G consecutive sites
// (one 128-byte line of every component) into LDS with coalesced loads; each
// wave then contracts G/W of those sites, one at a time.  The staged sites
// take 55.4 KB of LDS in either precision; FP32 runs 8 waves on them (two
// workgroups of 78 KB fill a CU's 160 KB with 4 waves per SIMD), FP64 4
// waves (its 159 VGPRs allow 3 waves per SIMD, and 8 waves would double
// the term slots to 94 KB, one workgroup per CU).
// LDS written and read by lanes of one wave only: a wavefront-scope fence
// orders the accesses (a wave's LDS operations are performed in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// D[c][c'] = sum eps_abc eps_a'b'c' a[a][a'] b[b][b']
template <typename T>
__device__ __forceinline__ void udsc_diquark(const cx<T> (&a)[9], const cx<T> (&b)[9], cx<T> (&d)[9]) {
#pragma unroll
  for (int cc = 0; cc < 3; cc++) {
    const int a1 = (cc + 1) % 3, a2 = (cc + 2) % 3;
#pragma unroll
    for (int dd = 0; dd < 3; dd++) {
      const int e1 = (dd + 1) % 3, e2 = (dd + 2) % 3;
      // + a[a1][e1] b[a2][e2] - a[a1][e2] b[a2][e1] - a[a2][e1] b[a1][e2] + a[a2][e2] b[a1][e1]
      const cx<T> p0 = a[a1 * 3 + e1], q0 = b[a2 * 3 + e2], p1 = a[a1 * 3 + e2], q1 = b[a2 * 3 + e1];
      const cx<T> p2 = a[a2 * 3 + e1], q2 = b[a1 * 3 + e2], p3 = a[a2 * 3 + e2], q3 = b[a1 * 3 + e1];
      T re = p0.re * q0.re;
      re = fma(-p0.im, q0.im, re);
      re = fma(-p1.re, q1.re, re);
      re = fma(p1.im, q1.im, re);
      re = fma(-p2.re, q2.re, re);
      re = fma(p2.im, q2.im, re);
      re = fma(p3.re, q3.re, re);
      re = fma(-p3.im, q3.im, re);
      T im = p0.re * q0.im;
      im = fma(p0.im, q0.re, im);
      im = fma(-p1.re, q1.im, im);
      im = fma(-p1.im, q1.re, im);
      im = fma(-p2.re, q2.im, im);
      im = fma(-p2.im, q2.re, im);
      im = fma(p3.re, q3.im, im);
      im = fma(p3.im, q3.re, im);
      d[cc * 3 + dd] = cmake<T>(re, im);
    }
  }
}

template <typename T> struct UdscGeom {
  static constexpr int G = 128 / (int)sizeof(cx<T>);  // sites per line
  static constexpr int SPAD = 433;                    // LDS stride of a site (432 + 1)
  static constexpr int W = sizeof(T) == 4 ? 8 : 4;    // waves per workgroup
  static constexpr int NT = 64 * W;
};

// RC: every coefficient is real (as in the built-in tables), an entry costs two
// FMAs instead of a complex product
template <typename T, bool RC>
__global__ __launch_bounds__(64 * UdscGeom<T>::W) void k_udsc(UdscSched S, const PropDev<T> *__restrict__ props,
                                              const RowDev *__restrict__ rows, cx<T> *__restrict__ out, int64_t V3,
                                              int T_lat, int nch_total, int ch0, int groups_per_block) {
  constexpr int G = UdscGeom<T>::G, SPAD = UdscGeom<T>::SPAD, W = UdscGeom<T>::W, NT = UdscGeom<T>::NT;
  constexpr int CPP = NT / G;                   // components one pass of the workgroup stages
  constexpr int NPASS = (144 + CPP - 1) / CPP;  // passes over a propagator's 144 components
  __shared__ cx<T> sp[G * SPAD];              // [site][f][m01][c c']
  __shared__ cx<T> sterm[W][64 * UD_TPQ];     // each wave's chunk terms, then its lanes' sums
  __shared__ __align__(16) uint16_t sent[UD_MAXENT];
  __shared__ T scoef[2 * UD_MAXCOEF];         // RC: the real parts only
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const RowDev row = rows[blockIdx.y];
  const PropDev<T> P0 = props[row.pa], P1 = props[row.pb], P2 = props[row.pc];
  auto plane_base = [&](const PropDev<T> &Q) {
    int plane = row.t - Q.t_first;
    plane += plane < 0 ? T_lat : 0;
    return Q.data + (int64_t)plane * V3;
  };
  const cx<T> *b0 = plane_base(P0), *b1 = plane_base(P1), *b2 = plane_base(P2);
  const T sg = prop_sign(P0, row.t) * prop_sign(P1, row.t) * prop_sign(P2, row.t);
  const int rot_any = P0.rot | P1.rot | P2.rot;
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total + ch0;
  // the lane's quads and terms in registers; the entries and coefficients in LDS
  int qv[UD_MAXC], tpv[UD_MAXC];
#pragma unroll
  for (int c = 0; c < UD_MAXC; c++) {
    const bool live = c < S.nchunks;
    qv[c] = live ? S.quads[c * 64 + lane] : -1;
    tpv[c] = live ? *(const int *)(S.tp + (c * 64 + lane) * UD_TPQ) : -1;
  }
  for (int i = tid; i < S.nent; i += NT) sent[i] = S.ents[i];
  if (RC)
    for (int i = tid; i < S.ncoef; i += NT) scoef[i] = (T)S.coef[2 * i];
  else
    for (int i = tid; i < 2 * S.ncoef; i += NT) scoef[i] = (T)S.coef[i];
  cx<T> *st = sterm[wave];
  // staging: thread (site s_l, component c_l) loads components c_l + i CPP of
  // the three propagators at site x0 + s_l; the G threads of a component read
  // one 128-byte line
  const int s_l = tid % G, c_l = tid / G;
  const int64_t o0 = (int64_t)c_l * P0.cs + s_l, o1 = (int64_t)c_l * P1.cs + s_l, o2 = (int64_t)c_l * P2.cs + s_l;
  const int64_t d0 = (int64_t)CPP * P0.cs, d1 = (int64_t)CPP * P1.cs, d2 = (int64_t)CPP * P2.cs;
  cx<T> *dst = sp + s_l * SPAD + c_l;

  for (int gi = 0; gi < groups_per_block; gi++) {
    const int64_t x0 = ((int64_t)blockIdx.x * groups_per_block + gi) * G;
    if (x0 >= V3) break;  // uniform over the workgroup
    // all loads of the group in flight at once, issued before the wait for
    // the previous group's sites
    const bool xin = x0 + s_l < V3;
    cx<T> v[3][NPASS];
#pragma unroll
    for (int i = 0; i < NPASS; i++) {
      const bool ok = xin && c_l + i * CPP < 144;
      v[0][i] = ok ? gload(b0 + x0 + o0 + i * d0) : cmake<T>(0, 0);
      v[1][i] = ok ? gload(b1 + x0 + o1 + i * d1) : cmake<T>(0, 0);
      v[2][i] = ok ? gload(b2 + x0 + o2 + i * d2) : cmake<T>(0, 0);
    }
    __syncthreads();  // the previous group's sites are done
#pragma unroll
    for (int i = 0; i < NPASS; i++)
      if (c_l + i * CPP < 144) {
        dst[i * CPP] = v[0][i];
        dst[144 + i * CPP] = v[1][i];
        dst[288 + i * CPP] = v[2][i];
      }
    __syncthreads();
    if (rot_any) {  // rotation to the physical basis, per (site, propagator, colour pair)
      for (int k = tid; k < G * 27; k += NT) {
        const int s = k / 27, f = (k % 27) / 9, cc = k % 9;
        const int rot = f == 0 ? P0.rot : (f == 1 ? P1.rot : P2.rot);
        if (rot) {
          cx<T> *b = sp + s * SPAD + f * 144 + cc;
          cx<T> w[16];
#pragma unroll
          for (int m = 0; m < 16; m++) w[m] = b[m * 9];
          rot_spins(w, rot);
#pragma unroll
          for (int m = 0; m < 16; m++) b[m * 9] = w[m];
        }
      }
      __syncthreads();
    }
    for (int s = wave; s < G; s += W) {
      const cx<T> *spx = sp + s * SPAD;
      cx<T> acc = cmake<T>(0, 0);
#pragma unroll
      for (int c = 0; c < UD_MAXC; c++) {
        if (c >= S.nchunks) break;
        const int q = qv[c];
        if (q >= 0) {
          // D of this lane's quad, in registers
          const cx<T> *A = spx + (q & 15) * 9, *B = spx + 144 + (q >> 4) * 9;
          cx<T> a[9], b[9], d[9];
#pragma unroll
          for (int j = 0; j < 9; j++) {
            a[j] = A[j];
            b[j] = B[j];
          }
          udsc_diquark(a, b, d);
          // its distinct terms T = sum_cc' D[c][c'] S3[m4m5][c][c']
#pragma unroll
          for (int e = 0; e < UD_TPQ; e++) {
            if (e >= S.ntp[c]) break;  // uniform: the chunk's fullest quad is done
            const int p = (signed char)(tpv[c] >> (8 * e));
            if (p >= 0) {
              const cx<T> *C3 = spx + 288 + p * 9;
              cx<T> t = cmake<T>(0, 0);
#pragma unroll
              for (int j = 0; j < 9; j++) cfma(t, d[j], C3[j]);
              st[e * 64 + lane] = t;
            }
          }
        }
        wave_sync();
        // the lane's share of its operator's entries: nblk[c] blocks of four
        const uint16_t *ec = sent + S.blk0[c] * 256 + lane * 4;
        for (int bk = 0; bk < S.nblk[c]; bk++) {
          const uint2 w = *(const uint2 *)(ec + bk * 256);
          const int u[4] = {(int)(w.x & 0xffff), (int)(w.x >> 16), (int)(w.y & 0xffff), (int)(w.y >> 16)};
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const cx<T> t = st[u[j] & 255];
            const int ci = u[j] >> 8;
            if (RC) {
              const T cr = scoef[ci];
              acc.re = fma(cr, t.re, acc.re);
              acc.im = fma(cr, t.im, acc.im);
            } else {
              cfma(acc, cmake<T>(scoef[2 * ci], scoef[2 * ci + 1]), t);
            }
          }
        }
        wave_sync();
      }
      // each operator sums the shares of its lanes
      st[lane] = acc;
      wave_sync();
      const int64_t x = x0 + s;
      if (lane < S.nops && x < V3) {
        const int lo = S.op_lo[lane], n = S.op_n[lane];
        cx<T> sum = cmake<T>(0, 0);
        for (int r = 0; r < n; r++) sum = sum + st[lo + r];
        gstore(out + ctile_idx(col0 + lane, x, ncols), cmake<T>(sg * sum.re, sg * sum.im));
      }
      wave_sync();
    }
  }
}

template <typename T>
int launch_udsc(const UdscSched &S, const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out, int64_t V3,
                int T_lat, int nch_total, int ch0, int spw, hipStream_t st) {
  // spw: sites per workgroup, rounded to whole groups
  constexpr int G = UdscGeom<T>::G;
  const int gpb = std::max(1, spw / G);
  const int64_t ngroups = (V3 + G - 1) / G;
  dim3 block(UdscGeom<T>::NT), grid((unsigned)((ngroups + gpb - 1) / gpb), (unsigned)nrows);
  if (S.real_coef)
    k_udsc<T, true><<<grid, block, 0, st>>>(S, props, rows, out, V3, T_lat, nch_total, ch0, gpb);
  else
    k_udsc<T, false><<<grid, block, 0, st>>>(S, props, rows, out, V3, T_lat, nch_total, ch0, gpb);
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template int launch_udsc<double>(const UdscSched &, const PropDev<double> *, const RowDev *, int, cx<double> *,
                                 int64_t, int, int, int, int, hipStream_t);
template int launch_udsc<float>(const UdscSched &, const PropDev<float> *, const RowDev *, int, cx<float> *,
                                int64_t, int, int, int, int, hipStream_t);

// ------------------------------------------------------------------ all products of a call
// The contraction of a call's flavour products in one launch.  A workgroup of
// 8 waves stages the four flavours of 16 consecutive sites in LDS, entries
// outermost (a row of 16 sites is 128 or 256 bytes), and the lane of site s
// and quarter q = lane / 16 forms the diquark of its quarter's quad of the
// step, then its terms, so that the schedule is uniform over the wave and a
// term's 64 values (16 sites, 4 quads) are, as they lie in the registers, the
// B operand of a 16x16x4 matrix product with the coefficients of the 16
// operators: O[k][site] += sum_q V[k][term of quad q] T[q][site], for the
// real and the imaginary part.  The waves share a group's steps and their
// sums meet in LDS at the group's end.
// Where the quads pair up, a quarter takes two at a time whose terms have like
// spin pairs of the third propagator: one read of it serves both.
// Bound by the vector unit and LDS (a term is 36 FMAs, two matrix instructions
// and 9 reads; one quad at a time the FMAs took 4.5 M of 9.2 M cycles, the
// matrix instructions 1.9 M, LDS was busy 5.5 M; two at a time LDS is busy
// 3.5 M of 8.6 M, 1.4 % of it bank conflicts).  20 products on 24^3 x 16
// sites, FP32, whole calls: 20 launches of k_udsc 14.6 ms, here one quad at a
// time 4.16 ms, two 3.89 ms.  k_udsc reads the terms, coefficients and entry
// indexes of its operator sums and every diquark's blocks from LDS 20 times
// per site, and is bound there.
// Entries that are not finite, and products that overflow, reach the operators
// that have a term with them at that site and no others (SAFE below).
template <typename T> struct UdAcc;
template <> struct UdAcc<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  static __device__ __forceinline__ int slot(int k, int s) { return (k & 3) * 64 + (k >> 2) * 16 + s; }  // r * 64 + lane
};
template <> struct UdAcc<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
  static __device__ __forceinline__ int slot(int k, int s) { return (k >> 2) * 64 + (k & 3) * 16 + s; }
};

template <typename T>
__global__ __launch_bounds__(64 * UD_WAVES, sizeof(T) == 4 ? 4 : 2) void k_udsc_all(
    UdscAll S, const PropDev<T> *__restrict__ props, const RowDev *__restrict__ rows, cx<T> *__restrict__ out,
    int64_t V3, int T_lat, int nch_total, int groups_per_block) {
  typedef typename UdAcc<T>::v4 v4;
  constexpr int NT = 64 * UD_WAVES;
  __shared__ cx<T> sp[4 * 144 * 16];        // [flavour][m01][c c'][site]
  __shared__ T red[UD_WAVES][256];          // the waves' sums of one product, real or imaginary
  const int tid = threadIdx.x, lane = tid & 63, s = tid & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const RowDev row = rows[blockIdx.y];
  const int64_t x0 = (int64_t)blockIdx.x * 16;
  {
    const bool xin = x0 + s < V3;
#pragma unroll
    for (int f = 0; f < 4; f++) {
      if (f >= S.nprops) break;
      const PropDev<T> Q = props[f];
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
  int rot_any = 0;
  for (int f = 0; f < S.nprops; f++) rot_any |= props[f].rot;
  if (rot_any) {  // rotation to the physical basis, per (site, propagator, colour pair)
    for (int k = tid; k < S.nprops * 9 * 16; k += NT) {
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
  const int64_t ncols = (int64_t)gridDim.y * nch_total, col0 = (int64_t)blockIdx.y * nch_total;
  const v4 *coef = (const v4 *)S.coef + lane;
  const int g1 = min((int)(blockIdx.z + 1) * groups_per_block, S.ngroups);
  for (int gi = blockIdx.z * groups_per_block; gi < g1; gi++) {
    const UdscGroup &G = S.g[gi];
    v4 ar[UD_NJ], ai[UD_NJ];
    const cx<T> *A = sp + G.pa * 2304 + s, *B = sp + G.pb * 2304 + s;
    // SAFE: values that are not finite stay out of the matrix products, where
    // a zero coefficient would spread them over the operators of a product,
    // and go one by one to those that have a coefficient, in spec
    T *spec = &red[0][0];  // [product][real, imaginary][as a wave's sums lie in red]
    static_assert(2 * UD_NJ <= UD_WAVES, "spec fits red");
    auto walk = [&](auto SAFE) {
      constexpr bool safe = SAFE.value;
#pragma unroll
      for (int j = 0; j < UD_NJ; j++) ar[j] = ai[j] = (v4)(T)0;
      const int st0 = G.step0[wave], nst = G.nsteps[wave];
      int un = G.unit0[wave], ci = G.coef0[wave];
      v4 cf[2] = {coef[ci * 64], coef[(ci + 1) * 64]};
      // a step: two quads of each quarter (N = 2, the terms' reads of the third
      // propagator serve both), or one
      auto step = [&](auto N, int st) {
        const uint32_t cw = S.steps[3 * st + 2];
        cx<T> d[N.value][9];
#pragma unroll
        for (int b = 0; b < N.value; b++) {
          const int q = (S.steps[3 * st + b] >> (8 * kq)) & 255;
          const cx<T> *Aq = A + (q & 15) * 144, *Bq = B + (q >> 4) * 144;
          cx<T> x[9], y[9];
#pragma unroll
          for (int j = 0; j < 9; j++) {
            x[j] = Aq[j * 16];
            y[j] = Bq[j * 16];
          }
          udsc_diquark(x, y, d[b]);
        }
#pragma unroll
        for (int j = 0; j < UD_NJ; j++) {
          const int nt = (cw >> (8 * j)) & 255;
          if (nt == 0) continue;
          const cx<T> *C = sp + G.third[j] * 2304 + s;
          for (int e0 = 0; e0 < nt; e0 += 4, un++, ci += N.value) {
            const uint64_t pw = (uint64_t)S.units[2 * un] | (uint64_t)S.units[2 * un + 1] << 32;
            const int pl = (int)(pw >> (16 * kq)) & 0xffff;
            v4 cn[N.value];  // the next unit's (SAFE: no loads ahead, for the registers)
#pragma unroll
            for (int b = 0; b < N.value; b++) {
              if constexpr (safe) cf[b] = coef[(ci + b) * 64];
              else cn[b] = coef[(ci + N.value + b) * 64];
            }
            v4 ur = (v4)(T)0, ui = (v4)(T)0;    // the unit's sums: sums of sums round less than one long sum
#pragma unroll
            for (int e = 0; e < 4; e++) {
              if (e0 + e >= nt) break;
              const cx<T> *Cp = C + ((pl >> (4 * e)) & 15) * 144;
              cx<T> t[N.value];
#pragma unroll
              for (int b = 0; b < N.value; b++) t[b] = cmake<T>(0, 0);
#pragma unroll
              for (int c = 0; c < 9; c++) {
                const cx<T> v = Cp[c * 16];
#pragma unroll
                for (int b = 0; b < N.value; b++) cfma(t[b], d[b][c], v);
              }
#pragma unroll
              for (int b = 0; b < N.value; b++) {
                if constexpr (safe) {
                  const bool fr = __builtin_isfinite(t[b].re), fi = __builtin_isfinite(t[b].im);
                  if (__any(!fr || !fi)) {
                    // (each quarter's operators with a coefficient in turn)
                    for (unsigned ops = (unsigned)(__ballot(cf[b][e] != 0) >> (16 * kq)) & 0xffff; __any(ops); ops &= ops - 1) {
                      const int k = ops ? __ffs(ops) - 1 : 0;
                      const T w = __shfl(cf[b][e], 16 * kq + k);
                      T *o = spec + 512 * j + UdAcc<T>::slot(k, s);
                      if (ops && !fr) atomicAdd(o, w * t[b].re);
                      if (ops && !fi) atomicAdd(o + 256, w * t[b].im);
                    }
                    t[b] = cmake<T>(fr ? t[b].re : (T)0, fi ? t[b].im : (T)0);
                  }
                }
                ur = UdAcc<T>::mma(cf[b][e], t[b].re, ur);
                ui = UdAcc<T>::mma(cf[b][e], t[b].im, ui);
              }
            }
            ar[j] += ur;
            ai[j] += ui;
            if constexpr (!safe)
#pragma unroll
              for (int b = 0; b < N.value; b++) cf[b] = cn[b];
          }
        }
      };
      const int mid = st0 + G.npair[wave];
      for (int st = st0; st < mid; st++) step(std::integral_constant<int, 2>{}, st);
      for (int st = mid; st < st0 + nst; st++) step(std::integral_constant<int, 1>{}, st);
    };
    walk(std::false_type{});
    int tq = threadIdx.x;  // opaque: what derives from it is not kept across the walk
    asm volatile("" : "+v"(tq));
    const int ln = tq & 63;
    // the waves' sums: thread tq < 256 holds operator row(ln, wave) of every product at its site
    T o[UD_NJ][2];
#pragma unroll
    for (int j = 0; j < UD_NJ; j++) o[j][0] = o[j][1] = 0;
    int *flag = (int *)spec;  // [256 / 64]: a sum of the wave is not finite, in the wave's own place of red
    auto reduce = [&]() {
#pragma unroll
      for (int j = 0; j < UD_NJ; j++) {
        if (j >= G.nprod) break;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
          for (int r = 0; r < 4; r++) red[wave][r * 64 + ln] = h ? ai[j][r] : ar[j][r];
          __syncthreads();
          if (tq < 256) {
            T v[UD_WAVES];
#pragma unroll
            for (int w = 0; w < UD_WAVES; w++) v[w] = red[w][tq];
#pragma unroll
            for (int n = UD_WAVES / 2; n > 0; n /= 2)  // pairwise
#pragma unroll
              for (int w = 0; w < n; w++) v[w] += v[w + n];
            o[j][h] = v[0];
            if (h == 1 && j + 1 == G.nprod) {
              bool bad = false;
#pragma unroll
              for (int i = 0; i <= j; i++) bad = bad || !__builtin_isfinite(o[i][0]) || !__builtin_isfinite(o[i][1]);
              const int mine = __any(bad);
              if (ln == 0) flag[(int)(sizeof(T) / 4) * tq] = mine;
            }
          }
          __syncthreads();
        }
      }
    };
    reduce();
    // a sum that is not finite: the group again, with the care of SAFE
    int any = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) any |= flag[(int)(sizeof(T) / 4) * 64 * w];
    __syncthreads();  // red is the next group's (or SAFE's) after this
    if (__builtin_amdgcn_readfirstlane(any)) {
      for (int i = tq; i < 512 * UD_NJ; i += NT) spec[i] = 0;
      __syncthreads();
      walk(std::true_type{});
      __syncthreads();
      T apart[UD_NJ][2];
#pragma unroll
      for (int j = 0; j < UD_NJ; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) apart[j][h] = spec[512 * j + 256 * h + (tq & 255)];
      __syncthreads();
      reduce();
#pragma unroll
      for (int j = 0; j < UD_NJ; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) o[j][h] += apart[j][h];
    }
    const T sgp = prop_sign(props[G.pa], row.t) * prop_sign(props[G.pb], row.t);
    const int k = UdAcc<T>::row(ln, wave);
    const int64_t x = (int64_t)blockIdx.x * 16 + (tq & 15);
#pragma unroll
    for (int j = 0; j < UD_NJ; j++) {
      if (j >= G.nprod) break;
      if (tq < 256 && k < G.nops[j] && x < V3) {
        const T sg = sgp * prop_sign(props[G.third[j]], row.t);
        gstore(out + ctile_idx(col0 + G.ch0[j] + k, x, ncols), cmake<T>(sg * o[j][0], sg * o[j][1]));
      }
    }
  }
}

template <typename T>
int launch_udsc_all(const UdscAll &S, const PropDev<T> *props, const RowDev *rows, int nrows, cx<T> *out, int64_t V3,
                    int T_lat, int nch_total, hipStream_t st) {
  const int64_t tiles = (V3 + 15) / 16;
  // few tiles: the groups go to workgroups of their own until the chip is full
  const int split = (int)std::max<int64_t>(1, std::min<int64_t>(S.ngroups, 512 / std::max<int64_t>(1, tiles * nrows)));
  const int gpb = (S.ngroups + split - 1) / split;
  dim3 grid((unsigned)tiles, (unsigned)nrows, (unsigned)((S.ngroups + gpb - 1) / gpb));
  k_udsc_all<T><<<grid, 64 * UD_WAVES, 0, st>>>(S, props, rows, out, V3, T_lat, nch_total, gpb);
  return hipGetLastError() == hipSuccess ? PLG_OK : PLG_ERR_HIP;
}

template int launch_udsc_all<double>(const UdscAll &, const PropDev<double> *, const RowDev *, int, cx<double> *,
                                     int64_t, int, int, hipStream_t);
template int launch_udsc_all<float>(const UdscAll &, const PropDev<float> *, const RowDev *, int, cx<float> *,
                                    int64_t, int, int, hipStream_t);

}  // namespace plg
