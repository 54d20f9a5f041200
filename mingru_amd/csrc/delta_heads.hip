// DeltaMinGRU's heads from one joined projection (gfx950): the mixer's normalisation,
// write strengths and layout change in one pass each way.
//
// The mixer (reference src/mingru/min_gru.py:3040-3100) splits its projections into
// heads, L2-normalises every key, takes beta = 2 sigmoid(.) and permutes all of it to
// the kernel layouts.  Run eagerly that is a norm, a division, a sigmoid, stacks and
// contiguous copies per tensor forward and their adjoints backward, some twenty
// launches over the same bytes; here the forward reads the projection once and writes
// the four kernel inputs, and the backward reads their gradients and writes the
// projection's whole gradient.
//
// P rows (N = H (dk + nh (dk + dv) + nh) elements): q (H, dk) | k (nh, H, dk) |
// v (nh, H, dv) | beta (nh, H).  A group of G = 16, 32 or 64 lanes (the smallest that
// holds max(dk, dv)) owns one (token, head): lane l holds element l of its q, k and v
// rows, so the key's norm and the backward's projection are group sums without LDS.
// HBM-bound copies: neighbouring groups take neighbouring heads of a token, so a wave
// reads consecutive bytes of P.  At B=8, T=1000, 4 heads of 64, fp32: 14 us each way for
// 49 and 74 MB; the layer's step, projections included, 1275 -> 700 to 810 us (host-bound).
#include "mg_common.h"

#include <type_traits>

namespace {

typedef uint16_t u16;
constexpr int HD_NT = 256;
constexpr float HD_EPS = 1e-12f;  // torch.nn.functional.normalize's default

__device__ __forceinline__ float ld1(const float* p) { return *p; }
__device__ __forceinline__ float ld1(const u16* p) { return __uint_as_float((unsigned)*p << 16); }
__device__ __forceinline__ void st1(float* p, float x) { *p = x; }
__device__ __forceinline__ void st1(u16* p, float x) {
  *p = __builtin_bit_cast(u16, (__bf16)x);
}

struct HdGeom {
  int64_t rows;  // B T H
  int64_t T, N;
  int H, nh, dk, dv;
};

// The group's (token row of P, kernel-layout row) and the lane's element.
struct HdRow {
  int64_t p;   // first element of the token's row of P
  int64_t o;   // (b H + h) T + t
  int h, l;
  bool ok;     // false past the last row: the lanes still take part in the group sums
};
template <int G>
__device__ __forceinline__ HdRow hd_row(const HdGeom& g) {
  HdRow r;
  int64_t i = ((int64_t)blockIdx.x * HD_NT + threadIdx.x) / G;
  r.ok = i < g.rows;
  if (!r.ok) i = g.rows - 1;
  r.l = threadIdx.x % G;
  const int64_t bt = i / g.H;
  r.h = (int)(i - bt * g.H);
  const int64_t b = bt / g.T;
  r.p = bt * g.N;
  r.o = (b * g.H + r.h) * g.T + (bt - b * g.T);
  return r;
}

// nrm (B, H, T, nh): max(|k|, eps), negated where the clamp was taken.
template <typename E, int G>
__global__ __launch_bounds__(HD_NT) void heads_fwd(const E* __restrict__ P, E* __restrict__ Q,
                                                   E* __restrict__ K, E* __restrict__ V,
                                                   E* __restrict__ beta, float* __restrict__ nrm,
                                                   HdGeom g) {
  const HdRow r = hd_row<G>(g);
  const bool lk = r.l < g.dk, lv = r.l < g.dv;
  const E* p = P + r.p;
  const E* pk = p + (int64_t)g.H * g.dk;
  const E* pv = pk + (int64_t)g.nh * g.H * g.dk;
  const E* pb = pv + (int64_t)g.nh * g.H * g.dv;
  const int kl = lk ? r.l : 0, vl = lv ? r.l : 0;
  const float q = ld1(p + r.h * g.dk + kl);
  if (r.ok && lk) st1(Q + r.o * g.dk + r.l, q);
  for (int j = 0; j < g.nh; ++j) {
    const int64_t jh = (int64_t)j * g.H + r.h, oj = r.o * g.nh + j;
    float k = ld1(pk + jh * g.dk + kl);
    const float v = ld1(pv + jh * g.dv + vl), b = ld1(pb + jh);
    k = lk ? k : 0.f;
    const float n = sqrtf(mg_group_sum<G>(k * k)), m = fmaxf(n, HD_EPS);
    if (!r.ok) continue;
    if (lk) st1(K + oj * g.dk + r.l, k / m);
    if (lv) st1(V + oj * g.dv + r.l, v);
    if (r.l == 0) {
      // The library's exp and a true division, not the hardware approximations of the gate
      // kernels: beta's error reaches its projection's gradients (relative error of the
      // bias gradient at B=8, T=1000, 4 heads of 64, three seeds: 0.8, 0.5, 1.0e-6 against
      // 1.6, 0.9, 1.0e-6 with them).
      st1(beta + oj, 2.f / (1.f + expf(-b)));
      if (nrm) nrm[oj] = n < HD_EPS ? -m : m;
    }
  }
}

// dk = (dK - K (K . dK)) / |k| (K the unit key; no projection where the norm was clamped),
// dbeta through 2 sigmoid: beta (1 - beta / 2).
template <typename E, int G>
__global__ __launch_bounds__(HD_NT) void heads_bwd(const E* __restrict__ K,
                                                   const E* __restrict__ beta,
                                                   const float* __restrict__ nrm,
                                                   const E* __restrict__ dQ,
                                                   const E* __restrict__ dK,
                                                   const E* __restrict__ dV,
                                                   const E* __restrict__ dbeta,
                                                   E* __restrict__ dP, HdGeom g) {
  const HdRow r = hd_row<G>(g);
  const bool lk = r.l < g.dk, lv = r.l < g.dv;
  E* p = dP + r.p;
  E* pk = p + (int64_t)g.H * g.dk;
  E* pv = pk + (int64_t)g.nh * g.H * g.dk;
  E* pb = pv + (int64_t)g.nh * g.H * g.dv;
  const int kl = lk ? r.l : 0, vl = lv ? r.l : 0;
  const float q = ld1(dQ + r.o * g.dk + kl);
  if (r.ok && lk) st1(p + r.h * g.dk + r.l, q);
  for (int j = 0; j < g.nh; ++j) {
    const int64_t jh = (int64_t)j * g.H + r.h, oj = r.o * g.nh + j;
    const float x = ld1(dK + oj * g.dk + kl), v = ld1(dV + oj * g.dv + vl);
    const float k = ld1(K + oj * g.dk + kl);
    const float n = nrm[oj], b = ld1(beta + oj), db = ld1(dbeta + oj);
    const float dot = mg_group_sum<G>(lk ? x * k : 0.f);
    if (!r.ok) continue;
    if (lk) st1(pk + jh * g.dk + r.l, (n > 0.f ? x - k * dot : x) / fabsf(n));
    if (lv) st1(pv + jh * g.dv + r.l, v);
    if (r.l == 0) st1(pb + jh, db * b * (1.f - 0.5f * b));
  }
}

// Lanes of a (token, head)'s group: the smallest that holds its rows.
int hd_group(const HdGeom& g) {
  const int d = g.dk > g.dv ? g.dk : g.dv;
  return d <= 16 ? 16 : d <= 32 ? 32 : 64;
}

bool hd_geom(HdGeom& g, int64_t B, int64_t T, int H, int nh, int dk, int dv, int dtype) {
  if (B <= 0 || T <= 0 || H <= 0 || nh <= 0 || dk <= 0 || dk > 64 || dv <= 0 || dv > 64 ||
      (dtype & ~1))
    return false;
  g = HdGeom{B * T * H, T, (int64_t)H * (dk + (int64_t)nh * (dk + dv) + nh), H, nh, dk, dv};
  return g.rows * hd_group(g) <= (1ll << 32) - HD_NT;  // a launch takes fewer than 2^32 threads
}

// f(element tag, group size) for the dtype (0 fp32, 1 bf16) and the head dims.
template <typename F>
int hd_pick(int dtype, const HdGeom& g, F&& f) {
  const int group = hd_group(g);
  auto by_group = [&](auto e) {
    if (group == 16) f(e, std::integral_constant<int, 16>{});
    else if (group == 32) f(e, std::integral_constant<int, 32>{});
    else f(e, std::integral_constant<int, 64>{});
  };
  if (dtype) by_group(u16{});
  else by_group(float{});
  return hipGetLastError() == hipSuccess ? MG_OK : MG_ERR_LAUNCH;
}

template <int G>
dim3 hd_grid(const HdGeom& g) {
  return dim3((unsigned)((g.rows * G + HD_NT - 1) / HD_NT));
}

}  // namespace

extern "C" {

int mg_delta_heads_fwd(const void* P, void* Q, void* K, void* V, void* beta, float* nrm, int64_t B,
                       int64_t T, int H, int nh, int dk, int dv, int dtype, hipStream_t stream) {
  HdGeom g;
  if (!P || !Q || !K || !V || !beta || !hd_geom(g, B, T, H, nh, dk, dv, dtype)) return MG_ERR_ARG;
  return hd_pick(dtype, g, [&](auto e, auto grp) {
    using E = decltype(e);
    constexpr int G = decltype(grp)::value;
    hipLaunchKernelGGL((heads_fwd<E, G>), hd_grid<G>(g), dim3(HD_NT), 0, stream, (const E*)P,
                       (E*)Q, (E*)K, (E*)V, (E*)beta, nrm, g);
  });
}

int mg_delta_heads_bwd(const void* K, const void* beta, const float* nrm, const void* dQ,
                       const void* dK, const void* dV, const void* dbeta, void* dP, int64_t B,
                       int64_t T, int H, int nh, int dk, int dv, int dtype, hipStream_t stream) {
  HdGeom g;
  if (!K || !beta || !nrm || !dQ || !dK || !dV || !dbeta || !dP ||
      !hd_geom(g, B, T, H, nh, dk, dv, dtype))
    return MG_ERR_ARG;
  return hd_pick(dtype, g, [&](auto e, auto grp) {
    using E = decltype(e);
    constexpr int G = decltype(grp)::value;
    hipLaunchKernelGGL((heads_bwd<E, G>), hd_grid<G>(g), dim3(HD_NT), 0, stream, (const E*)K,
                       (const E*)beta, nrm, (const E*)dQ, (const E*)dK, (const E*)dV,
                       (const E*)dbeta, (E*)dP, g);
  });
}

}  // extern "C"
