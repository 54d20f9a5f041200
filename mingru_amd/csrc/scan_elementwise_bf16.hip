// bf16 entry points of the elementwise scans (mg_elementwise.h), and the gate scans over
// strided pre-activations.
//
// The tensors are read and written as bf16 and every step computes in fp32.  Casting
// to fp32 outside instead moves each input 5 times its size (read 2, write 4, read 4)
// and each output as often.  What the backward restarts from stays fp32: the forward
// records its fp32 states at every sub-chunk start (1 byte per element for the gate
// and linear scans).  linear_scan forward + backward at B=6, T=3001, D=776: 278 -> 126 us
// a step; a decay SignedMinGRU layer at B=8, T=2048, D=1024, projections included:
// 996 -> 811 us (535 with its projections joined, which the strided entry points allow).
#include "mg_elementwise.h"

extern "C" {

size_t mg_linear_scan_bf16_state_bytes(int64_t B, int64_t T, int64_t D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (size_t)B * (size_t)((T + LIN_STATE - 1) / LIN_STATE) * 2 * (size_t)D * sizeof(float);
}

int mg_linear_scan_bf16_fwd(const void* a, const void* b, void* A, void* Bc, float* state,
                            int64_t B, int64_t T, int64_t D, void* ws, size_t ws_bytes,
                            hipStream_t stream) {
  if (!a || !b || !A || !Bc || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return linear_fwd_launch((const mg_bf16*)a, (const mg_bf16*)b, (mg_bf16*)A, (mg_bf16*)Bc, state,
                           B, T, D, ws, ws_bytes, stream);
}

int mg_linear_scan_bf16_bwd(const void* a, const void* b, const float* state, const void* gA,
                            const void* gB, void* da, void* db, int64_t B, int64_t T, int64_t D,
                            void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!a || !b || !state || !gA || !gB || !da || !db || !ws || !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  const bool v4 = D % 4 == 0 && all_aligned({a, b, gA, gB, da, db}, 8) && all_aligned({state}, 16);
  const int vec = ew_vec(B, T, D, v4, EW_WAVES_BWD * EW_TSUB_BWD);
  return by_vec(vec, [&](auto v) {
    constexpr int V = decltype(v)::value;
    constexpr int TS = EW_TSUB_BWD, W = EW_WAVES_BWD;
    EwPlan p = ew_plan(B, T, D, V, TS, W, 2);
    if (ws_bytes < p.total) return MG_ERR_WORKSPACE;
    return ew_run(ew_two_launch(p, B, T, D, 4, sizeof(mg_bf16)), linear_bwd_bf16_kernel<V, TS, W>,
                  linear_bwd_bf16_kernel<V, TS, W, EW_REDUCE>,
                  linear_bwd_bf16_kernel<V, TS, W, EW_FINAL>,
                  linear_bwd_bf16_kernel<V, TS, W, EW_AGG>, p, ws, stream, (const mg_bf16*)a,
                  (const mg_bf16*)b, state, (const mg_bf16*)gA, (const mg_bf16*)gB, (mg_bf16*)da,
                  (mg_bf16*)db);
  });
}

int mg_log_scan_bf16_fwd(const void* lc, const void* lv, void* h, float* hstate, int64_t B,
                         int64_t T, int64_t D, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!lc || !lv || !h || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return log_fwd_launch((const mg_bf16*)lc, (const mg_bf16*)lv, (mg_bf16*)h, hstate, B, T, D, ws,
                        ws_bytes, stream);
}

int mg_log_scan_bf16_bwd(const void* lc, const void* lv, const float* hstate, const void* gh,
                         void* dlc, void* dlv, int64_t B, int64_t T, int64_t D, void* ws,
                         size_t ws_bytes, hipStream_t stream) {
  if (!lc || !lv || !hstate || !gh || !dlc || !dlv || !ws || !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  return log_bwd_launch((const mg_bf16*)lc, (const mg_bf16*)lv, (const mg_bf16*)nullptr, hstate,
                        (const mg_bf16*)gh, (mg_bf16*)dlc, (mg_bf16*)dlv, B, T, D, ws, ws_bytes,
                        stream);
}

size_t mg_gate_scan_bf16_state_bytes(int64_t B, int64_t T, int64_t D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (size_t)B * (size_t)((T + GATE_STATE - 1) / GATE_STATE) * (size_t)D * sizeof(float);
}

int mg_gate_scan_bf16_fwd(int kind, const void* p0, const void* p1, const void* p2, int64_t ld,
                          const void* h0, int h0_half, float h0_const, const float* dt,
                          const float* lam, void* h, float* hstate, int64_t B, int64_t T, int64_t D, void* ws,
                          size_t ws_bytes, hipStream_t stream) {
  if (kind < GATE_SIGNED || kind > GATE_MINGRU || !p0 || !p1 || (kind != GATE_MINGRU && !p2) ||
      !h || !ws || !geometry_ok(B, T, D) || ld < D || !dt != !lam || (h0_half & ~1))
    return MG_ERR_ARG;
  return gate_fwd_any<mg_bf16>(kind, {p0, p1, p2, h0, ld, h0_half, h0_const}, h, hstate,
                               GateDecay{dt, lam, nullptr, nullptr}, B, T, D, ws, ws_bytes,
                               stream);
}

int mg_gate_scan_bf16_bwd(int kind, const void* p0, const void* p1, const void* p2, int64_t ld,
                          const float* dt, const float* lam, const float* hstate, const void* gh,
                          void* d0, void* d1, void* d2, float* dh0, float* dlam, float* ddt,
                          int64_t B, int64_t T, int64_t D, void* ws, size_t ws_bytes,
                          hipStream_t stream) {
  if (kind < GATE_SIGNED || kind > GATE_MINGRU || !p0 || !p1 || (kind != GATE_MINGRU && !p2) ||
      !hstate || !gh || !d0 || !d1 || (kind != GATE_MINGRU && !d2) || !ws ||
      !geometry_ok(B, T, D) || ld < D || !dt != !lam)
    return MG_ERR_ARG;
  return gate_bwd_any<mg_bf16>(kind, {p0, p1, p2, nullptr, ld, 0}, hstate, gh, d0, d1, d2, dh0,
                               GateDecay{dt, lam, dlam, ddt}, B, T, D, ws, ws_bytes, stream);
}

}  // extern "C"
