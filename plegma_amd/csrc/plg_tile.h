// plg_tile.h -- the site tile shared by the per-site contraction kernels
// (baryons, fused two-point, meson-meson): 16 lattice sites staged in LDS,
// four lanes of a wavefront per site (a DPP quad), and the spin algebra those
// lanes share.
#pragma once
#include "plg_internal.h"

namespace plg {

// per meson channel op (GAMMAS order): xor class and phases of X = g5 G
struct MesonX {
  int cls[16];
  int ph[16][4];
};
constexpr MesonX make_mesonx() {
  MesonX m{};
  for (int op = 0; op < 16; op++) {
    SPerm X = sp_mul(G_5, gamma_op(op));
    m.cls[op] = sp_class(X);
    for (int i = 0; i < 4; i++) m.ph[op][i] = X.ph[i];
  }
  return m;
}
constexpr MesonX MESON_X = make_mesonx();
// the n-th channel of xor class d (four each)
constexpr int meson_op(int d, int n) {
  for (int op = 0; op < 16; op++)
    if (MESON_X.cls[op] == d && n-- == 0) return op;
  return -1;
}

// ---- DPP row exchanges
template <int CTRL> __device__ __forceinline__ double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// ---- staging of a tile: 16-byte units of EPU sites
template <typename T, int N> struct SiteVec;
template <> struct SiteVec<float, 2> {  // two sites; site pairs are 8-byte aligned
  typedef float v __attribute__((ext_vector_type(4), aligned(8)));
};
template <> struct SiteVec<double, 1> {
  typedef double v __attribute__((ext_vector_type(2)));
};

// value of lane ^ S within the four lanes of a site
template <int S> __device__ __forceinline__ float quad_xor(float v) {
  if constexpr (S == 0) return v;
  else return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), S == 1 ? 0xB1 : S == 2 ? 0x4E : 0x1B, 0xF, 0xF, true));
}
template <int S> __device__ __forceinline__ double quad_xor(double v) {
  if constexpr (S == 0) return v;
  else {
    constexpr int ctrl = S == 1 ? 0xB1 : S == 2 ? 0x4E : 0x1B;
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, ctrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}
template <typename T> __device__ __forceinline__ T quad_sum(T v) {
  v += quad_xor<1>(v);
  v += quad_xor<2>(v);
  return v;
}

// sign of a phase table relative to its entry 0, as a character of the index
constexpr bool char_ok(const int (&ph)[4]) {
  for (int n = 0; n < 4; n++)
    if (((ph[n] - ph[0]) & 1) != 0) return false;
  return ((ph[1] - ph[0] + ph[2] - ph[0]) & 3) == ((ph[3] - ph[0]) & 3);
}
// lane j's sign of a character
template <typename T> __device__ __forceinline__ T char_sign(const int (&ph)[4], int j) {
  T s = 1;
#pragma unroll
  for (int n = 1; n < 4; n++) s = (j == n && ((ph[n] - ph[0]) & 3) == 2) ? (T)-1 : s;
  return s;
}
// of four values per lane, the sums over the four lanes: lane n keeps value n
template <typename T> __device__ __forceinline__ T quad_scatter_sum(T a, T b, T c, T d, int j) {
  const bool odd = j & 1, hi = j & 2;
  const T a1 = odd ? b : a, b1 = odd ? a : b, c1 = odd ? d : c, d1 = odd ? c : d;
  const T lo2 = a1 + quad_xor<1>(b1), hi2 = c1 + quad_xor<1>(d1);
  const T keep = hi ? hi2 : lo2, send = hi ? lo2 : hi2;
  return keep + quad_xor<2>(send);
}
template <typename T> __device__ __forceinline__ cx<T> quad_scatter_sum(const cx<T> (&v)[4], int j) {
  return cmake<T>(quad_scatter_sum(v[0].re, v[1].re, v[2].re, v[3].re, j),
                  quad_scatter_sum(v[0].im, v[1].im, v[2].im, v[3].im, j));
}

}  // namespace plg
