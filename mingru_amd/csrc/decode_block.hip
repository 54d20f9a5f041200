// Streaming decode of a residual block (gfx950): one token for a few sequences, where
// every layer is a read of its weights and the launches cost more than the bytes.
//
// MinGRUBlock.step (reference src/mingru/min_gru.py:3960-4008) run layer by layer is a
// dozen launches: norms, two to eight projections, the recurrent step, GELU, sums.  Here
// a block is three (diagonal mixers) or five (delta):
//   step_gate:    LayerNorm, the gate projections, the recurrent step, the residual sum;
//   step_project: LayerNorm (optional), any number of projections side by side, GELU or a
//                 residual sum (optional): the MLP's two products, delta's heads and output;
//   delta_step_heads: delta's key normalisation, write strengths and state update.
//
// Split: one wave per output column and projection.  Its lanes read the column's weight
// row in 4-element pieces, each piece times the same piece of every sequence's input, and
// the per-sequence sums meet in wave-wide DPP sums; lane b finishes sequence b.  Weights
// are read once; a few hundred to a few thousand waves are in flight.  Inputs that pass a
// LayerNorm are normalised by every workgroup for itself into LDS (two-pass, fp32), which
// costs less than the launch it saves; others are read through L1.  Sums and everything
// between the launches stay fp32 whatever the weights' type.  More than 16 sequences run
// as groups of 16 (grid rows), each reading the weights again, from the L2.  At B=8,
// d=256, four layers, fp32: 820 -> 259 us a token, most of what is left host time (90 us
// of kernels, of 264 before).
#include "mg_common.h"
#include "mg_gates.h"

#include <type_traits>

namespace {

typedef uint16_t u16;
constexpr int SB_WAVES = 4;
constexpr int SB_NT = SB_WAVES * MG_WAVE;
constexpr int SB_MAX_B = 16;      // sequences of a group
constexpr int SB_MAX_GROUPS = 16;
constexpr int SB_MAX_SEG = 16;
constexpr size_t SB_MAX_LDS = 64 << 10;

__device__ __forceinline__ float ld1(const float* p) { return *p; }
__device__ __forceinline__ float ld1(const u16* p) { return __uint_as_float((unsigned)*p << 16); }
__device__ __forceinline__ void st1(float* p, float x) { *p = x; }
__device__ __forceinline__ void st1(u16* p, float x) { *p = __builtin_bit_cast(u16, (__bf16)x); }
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4(const u16* p) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                     __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u));
}

enum : int { SB_PLAIN = 0, SB_GELU = 1, SB_RESIDUAL = 2 };  // step_project epilogues

struct SbArgs {
  const void* x;        // (B, K): fp32 if x_f32, else the weights' type
  const void *ln_w, *ln_b;  // (K): LayerNorm of x, or null
  float eps;
  int B, K, x_f32;      // all sequences; a workgroup's group: sb_first, sb_count
  int nseg;             // projections; segment s has n[s] rows of K, out columns off[s]..
  const void* w[SB_MAX_SEG];
  const void* bias[SB_MAX_SEG];  // null: none
  int off[SB_MAX_SEG + 1];
  void* out;            // (B, off[nseg]): fp32 if out_f32
  int out_f32, epi;
  const void* res;      // (B, columns) in the weights' type (SB_RESIDUAL; gates: x itself)
  // gates
  const float* gamma;   // (B, D) decay factors or null
  const void* h_prev;   // (B, D)
  void* h;              // (B, D)
};

// This workgroup's group of sequences: its first, and how many.
__device__ __forceinline__ int sb_first() { return (int)blockIdx.y * SB_MAX_B; }
__device__ __forceinline__ int sb_count(const SbArgs& a) {
  const int n = a.B - sb_first();
  return n < SB_MAX_B ? n : SB_MAX_B;
}

template <typename E>
__device__ __forceinline__ float4 sb_x4(const SbArgs& a, int b, int k) {
  const int64_t i = (int64_t)b * a.K + k;
  return a.x_f32 ? ld4((const float*)a.x + i) : ld4((const E*)a.x + i);
}

// The normalised input rows in LDS, (B, K) fp32: wave w takes rows w, w + SB_WAVES, ...
template <typename E>
__device__ __forceinline__ void sb_layer_norm(const SbArgs& a, float* xs) {
  const int lane = threadIdx.x & (MG_WAVE - 1);
  const int b0 = sb_first(), nb = sb_count(a);
  for (int b = threadIdx.x / MG_WAVE; b < nb; b += SB_WAVES) {
    float s = 0.f;
    for (int k = lane * 4; k < a.K; k += 4 * MG_WAVE) {
      const float4 v = sb_x4<E>(a, b0 + b, k);
      *reinterpret_cast<float4*>(xs + b * a.K + k) = v;
      s += (v.x + v.y) + (v.z + v.w);
    }
    const float mean = mg_group_sum<64>(s) / (float)a.K;
    float q = 0.f;
    for (int k = lane * 4; k < a.K; k += 4 * MG_WAVE) {
      const float4 v = *reinterpret_cast<float4*>(xs + b * a.K + k);  // this lane's own
      const float x = v.x - mean, y = v.y - mean, z = v.z - mean, w = v.w - mean;
      q += (x * x + y * y) + (z * z + w * w);
    }
    const float rstd = rsqrtf(mg_group_sum<64>(q) / (float)a.K + a.eps);
    for (int k = lane * 4; k < a.K; k += 4 * MG_WAVE) {
      float4 v = *reinterpret_cast<float4*>(xs + b * a.K + k);
      const float4 g = ld4((const E*)a.ln_w + k), c = ld4((const E*)a.ln_b + k);
      v.x = fmaf((v.x - mean) * rstd, g.x, c.x);
      v.y = fmaf((v.y - mean) * rstd, g.y, c.y);
      v.z = fmaf((v.z - mean) * rstd, g.z, c.z);
      v.w = fmaf((v.w - mean) * rstd, g.w, c.w);
      *reinterpret_cast<float4*>(xs + b * a.K + k) = v;
    }
  }
  __syncthreads();
}

// Lane b's sum over k of x[b][k] * row[k] for the NS weight rows (whole wave active).
template <typename E, int BT, int NS, bool LN>
__device__ __forceinline__ void sb_dots(const SbArgs& a, const float* xs,
                                        const E* const (&row)[NS], float (&mine)[NS]) {
  const int lane = threadIdx.x & (MG_WAVE - 1), b0 = sb_first(), nb = sb_count(a);
  float acc[NS][BT];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int b = 0; b < BT; ++b) acc[s][b] = 0.f;
  for (int k = lane * 4; k < a.K; k += 4 * MG_WAVE) {
    float4 w[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) w[s] = ld4(row[s] + k);
#pragma unroll
    for (int b = 0; b < BT; ++b) {
      const int bb = b < nb ? b : nb - 1;
      const float4 x =
          LN ? *reinterpret_cast<const float4*>(xs + bb * a.K + k) : sb_x4<E>(a, b0 + bb, k);
#pragma unroll
      for (int s = 0; s < NS; ++s)
        acc[s][b] = fmaf(x.x, w[s].x, fmaf(x.y, w[s].y, fmaf(x.z, w[s].z, fmaf(x.w, w[s].w,
                                                                               acc[s][b]))));
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    mine[s] = 0.f;
#pragma unroll
    for (int b = 0; b < BT; ++b) {
      const float t = mg_group_sum<64>(acc[s][b]);
      mine[s] = lane == b ? t : mine[s];
    }
  }
}

template <typename E, int BT, bool LN>
__global__ __launch_bounds__(SB_NT) void step_project(SbArgs a) {
  extern __shared__ float xs[];
  if constexpr (LN) sb_layer_norm<E>(a, xs);
  const int cols = a.off[a.nseg];
  const int col = blockIdx.x * SB_WAVES + (int)mg_uniform(threadIdx.x / MG_WAVE);
  if (col >= cols) return;
  int s = 0;
  while (col >= a.off[s + 1]) ++s;
  const int n = col - a.off[s], lane = threadIdx.x & (MG_WAVE - 1);
  const E* const row[1] = {(const E*)a.w[s] + (int64_t)n * a.K};
  float y[1];
  sb_dots<E, BT, 1, LN>(a, xs, row, y);
  if (lane >= sb_count(a)) return;
  float v = y[0] + (a.bias[s] ? ld1((const E*)a.bias[s] + n) : 0.f);
  if (a.epi == SB_GELU) v = 0.5f * v * (1.f + erff(v * 0.70710678118654752440f));
  const int64_t o = (int64_t)(sb_first() + lane) * cols + col;
  if (a.epi == SB_RESIDUAL) v += ld1((const E*)a.res + o);
  if (a.out_f32) st1((float*)a.out + o, v);
  else st1((E*)a.out + o, v);
}

// Column d of the gate projections (segments 0 .. NS - 1), the recurrent step, and the
// residual sum x + h into `out`.
template <typename E, int BT, int G>
__global__ __launch_bounds__(SB_NT) void step_gate(SbArgs a) {
  extern __shared__ float xs[];
  constexpr int NS = G == GATE_MINGRU ? 2 : 3;
  sb_layer_norm<E>(a, xs);
  const int D = a.off[1];
  const int d = blockIdx.x * SB_WAVES + (int)mg_uniform(threadIdx.x / MG_WAVE);
  if (d >= D) return;
  const int lane = threadIdx.x & (MG_WAVE - 1);
  const E* row[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) row[s] = (const E*)a.w[s] + (int64_t)d * a.K;
  const E* const(&crow)[NS] = row;
  float p[NS];
  sb_dots<E, BT, NS, true>(a, xs, crow, p);
  if (lane >= sb_count(a)) return;
#pragma unroll
  for (int s = 0; s < NS; ++s) p[s] += a.bias[s] ? ld1((const E*)a.bias[s] + d) : 0.f;
  float ca, cb;
  gate_coeffs<G>(p[0], p[1], NS == 3 ? p[NS - 1] : 0.f, ca, cb);
  const int64_t o = (int64_t)(sb_first() + lane) * D + d;
  if (a.gamma) ca *= a.gamma[o];
  const float h = fmaf(ca, ld1((const E*)a.h_prev + o), cb);
  st1((E*)a.h + o, h);
  st1((E*)a.out + o, ld1((const E*)a.res + o) + h);
}

// One wave per (sequence, head), lane j owning column j of H (d_k values in registers),
// as delta_step_kernel (decode_step.hip); q, k, v and beta come raw from a joined
// projection's fp32 row (segments q | k | v | beta, each (H, ..) per micro-step), and the
// key is normalised and beta formed here.  Every load is clamped, none conditional.
constexpr int SB_DK = 64;
__device__ __forceinline__ float lane_bcast(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

template <typename E>
__global__ __launch_bounds__(MG_WAVE) void delta_step_heads(const E* __restrict__ Hin,
                                                            const float* __restrict__ P,
                                                            const float* __restrict__ lg,
                                                            E* __restrict__ Hout,
                                                            float* __restrict__ y, int H, int nh,
                                                            int dk, int dv) {
  const int64_t head = blockIdx.x;
  const int64_t b = head / H;
  const int h = (int)(head - b * H), j = threadIdx.x;
  const int N = H * (dk + nh * (dk + dv) + nh);
  const float* p = P + b * N;
  const int jk = j < dk ? j : dk - 1, jv = j < dv ? j : dv - 1;
  const E* Hh = Hin + head * dk * dv;
  float hc[SB_DK];
#pragma unroll
  for (int i = 0; i < SB_DK; ++i) hc[i] = ld1(Hh + (i < dk ? i : dk - 1) * dv + jv);
  const float gm = lg ? expf(lg[head]) : 1.f;
#pragma unroll
  for (int i = 0; i < SB_DK; ++i) hc[i] = i < dk ? hc[i] * gm : 0.f;
  float q = p[h * dk + jk];
  q = j < dk ? q : 0.f;
  const float* pk = p + H * dk;
  const float* pv = pk + nh * H * dk;
  const float* pb = pv + nh * H * dv;
  for (int m = 0; m < nh; ++m) {
    const int mh = m * H + h;
    float k = pk[mh * dk + jk];
    k = j < dk ? k : 0.f;
    k /= fmaxf(sqrtf(mg_group_sum<64>(k * k)), 1e-12f);
    const float beta = 2.f / (1.f + expf(-pb[mh]));  // as delta_heads.hip
    float kh = 0.f;
#pragma unroll
    for (int i = 0; i < SB_DK; ++i) kh = fmaf(lane_bcast(k, i), hc[i], kh);
    const float bu = beta * (pv[mh * dv + jv] - kh);
#pragma unroll
    for (int i = 0; i < SB_DK; ++i) hc[i] = fmaf(lane_bcast(k, i), bu, hc[i]);
  }
  float yy = 0.f;
#pragma unroll
  for (int i = 0; i < SB_DK; ++i) yy = fmaf(lane_bcast(q, i), hc[i], yy);
  if (j < dv) {
    y[head * dv + j] = yy;
    E* Ho = Hout + head * dk * dv;
#pragma unroll
    for (int i = 0; i < SB_DK; ++i)
      if (i < dk) st1(Ho + i * dv + j, hc[i]);
  }
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

// Bytes of a group's normalised rows, and the grid's groups.
size_t sb_lds(int B, int K) { return (size_t)(B < SB_MAX_B ? B : SB_MAX_B) * K * sizeof(float); }
unsigned sb_groups(int B) { return (unsigned)((B + SB_MAX_B - 1) / SB_MAX_B); }

// The shared checks: sizes, 4-element pieces of every row, LDS for the normalised input.
bool sb_ok(const SbArgs& a, int dtype) {
  const uintptr_t e4 = dtype ? 8 : 16;
  if (!a.x || !a.out || a.B < 1 || a.B > SB_MAX_B * SB_MAX_GROUPS || a.K < 4 || a.K % 4 || a.K > (1 << 20) ||
      (dtype & ~1) || a.nseg < 1 || a.nseg > SB_MAX_SEG)
    return false;
  if (!aligned(a.x, a.x_f32 ? 16 : e4) || !aligned(a.ln_w, e4) || !aligned(a.ln_b, e4))
    return false;
  if (!a.ln_w != !a.ln_b) return false;
  if (a.ln_w && sb_lds(a.B, a.K) > SB_MAX_LDS) return false;
  for (int s = 0; s < a.nseg; ++s)
    if (!a.w[s] || !aligned(a.w[s], e4) || a.off[s + 1] <= a.off[s]) return false;
  return true;
}

// f(element tag, batch tile) for the dtype and the smallest tile that holds B.
template <typename F>
int sb_pick(int dtype, int B, F&& f) {
  auto by_tile = [&](auto e) {
    if (B == 1) f(e, std::integral_constant<int, 1>{});
    else if (B <= 4) f(e, std::integral_constant<int, 4>{});
    else if (B <= 8) f(e, std::integral_constant<int, 8>{});
    else f(e, std::integral_constant<int, 16>{});
  };
  if (dtype) by_tile(u16{});
  else by_tile(float{});
  return hipGetLastError() == hipSuccess ? MG_OK : MG_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int mg_step_project(int dtype, const void* x, int x_f32, int B, int K, const void* ln_w,
                    const void* ln_b, float eps, int nseg, const void* const* w,
                    const void* const* bias, const int* n, int epi, const void* res, void* out,
                    int out_f32, hipStream_t stream) {
  if (nseg < 1 || nseg > SB_MAX_SEG || !w || !bias || !n || epi < SB_PLAIN || epi > SB_RESIDUAL ||
      (epi == SB_RESIDUAL && !res))
    return MG_ERR_ARG;
  SbArgs a{};
  a.x = x, a.x_f32 = x_f32, a.B = B, a.K = K;
  a.ln_w = ln_w, a.ln_b = ln_b, a.eps = eps;
  a.nseg = nseg, a.epi = epi, a.res = res, a.out = out, a.out_f32 = out_f32;
  for (int s = 0; s < nseg; ++s) {
    if (n[s] < 1 || n[s] > (1 << 24)) return MG_ERR_ARG;
    a.w[s] = w[s], a.bias[s] = bias[s], a.off[s + 1] = a.off[s] + n[s];
  }
  if (!sb_ok(a, dtype)) return MG_ERR_ARG;
  const dim3 grid((a.off[nseg] + SB_WAVES - 1) / SB_WAVES, sb_groups(B));
  return sb_pick(dtype, B, [&](auto e, auto bt) {
    using E = decltype(e);
    constexpr int BT = decltype(bt)::value;
    if (a.ln_w)
      hipLaunchKernelGGL((step_project<E, BT, true>), grid, dim3(SB_NT),
                         sb_lds(B, K), stream, a);
    else
      hipLaunchKernelGGL((step_project<E, BT, false>), grid, dim3(SB_NT), 0, stream, a);
  });
}

int mg_step_gate(int dtype, int kind, const void* x, int B, int K, const void* ln_w,
                 const void* ln_b, float eps, const void* w0, const void* b0, const void* w1,
                 const void* b1, const void* w2, const void* b2, const float* gamma,
                 const void* h_prev, void* h, void* out, int D, hipStream_t stream) {
  if (kind < GATE_SIGNED || kind > GATE_MINGRU || !ln_w || !h_prev || !h || D < 1 || D > (1 << 24) ||
      D != K)
    return MG_ERR_ARG;
  SbArgs a{};
  a.x = x, a.B = B, a.K = K, a.ln_w = ln_w, a.ln_b = ln_b, a.eps = eps;
  a.nseg = kind == GATE_MINGRU ? 2 : 3;
  const void *w[3] = {w0, w1, w2}, *bias[3] = {b0, b1, b2};
  for (int s = 0; s < a.nseg; ++s) a.w[s] = w[s], a.bias[s] = bias[s], a.off[s + 1] = a.off[s] + D;
  a.res = x, a.out = out, a.gamma = gamma, a.h_prev = h_prev, a.h = h;
  if (!sb_ok(a, dtype)) return MG_ERR_ARG;
  const dim3 grid((D + SB_WAVES - 1) / SB_WAVES, sb_groups(B));
  const size_t lds = sb_lds(B, K);
  return sb_pick(dtype, B, [&](auto e, auto bt) {
    using E = decltype(e);
    constexpr int BT = decltype(bt)::value;
    if (kind == GATE_SIGNED)
      hipLaunchKernelGGL((step_gate<E, BT, GATE_SIGNED>), grid, dim3(SB_NT), lds, stream, a);
    else if (kind == GATE_SIGNED_COUPLED)
      hipLaunchKernelGGL((step_gate<E, BT, GATE_SIGNED_COUPLED>), grid, dim3(SB_NT), lds, stream,
                         a);
    else
      hipLaunchKernelGGL((step_gate<E, BT, GATE_MINGRU>), grid, dim3(SB_NT), lds, stream, a);
  });
}

int mg_delta_step_heads(int dtype, const void* H_in, const float* P, const float* log_gamma,
                        void* H_out, float* y, int64_t B, int H, int nh, int dk, int dv,
                        hipStream_t stream) {
  if (!H_in || !P || !H_out || !y || B < 1 || H < 1 || nh < 1 || dk < 1 || dk > SB_DK || dv < 1 ||
      dv > 64 || (dtype & ~1) || B * H > 0x7fffffff)
    return MG_ERR_ARG;
  const dim3 grid((unsigned)(B * H));
  if (dtype)
    hipLaunchKernelGGL(delta_step_heads<u16>, grid, dim3(MG_WAVE), 0, stream, (const u16*)H_in, P,
                       log_gamma, (u16*)H_out, y, H, nh, dk, dv);
  else
    hipLaunchKernelGGL(delta_step_heads<float>, grid, dim3(MG_WAVE), 0, stream, (const float*)H_in,
                       P, log_gamma, (float*)H_out, y, H, nh, dk, dv);
  return hipGetLastError() == hipSuccess ? MG_OK : MG_ERR_LAUNCH;
}

}  // extern "C"
