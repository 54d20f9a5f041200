// fp32 entry points of the elementwise scans (mg_elementwise.h): linear_scan,
// parallel_scan_log and the fused gate scans, and the allocation-free linear_scan.
#include "mg_elementwise.h"

namespace {

// ---------------------------------------------------------------------------
// Static look-back scratch for callers that cannot allocate
// ---------------------------------------------------------------------------
// One array per device, holding the workspace of mg_linear_scan_fwd_noalloc.
// In host code `scratch` names a host-side stand-in, never the device memory:
// every host use goes through the address hipGetSymbolAddress returns for the
// current device, which is looked up once per device and cached.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;  // == MG_NOALLOC_SCRATCH_BYTES
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;

struct NoallocDevice {
  std::mutex mu;                     // serialises the one-time set-up
  std::atomic<void*> ptr{nullptr};   // device address of `scratch`, once set up
};
NoallocDevice g_noalloc[NOALLOC_MAX_DEVICES];

__global__ void zero_fill_kernel(uint4* __restrict__ p, size_t n16) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
    p[i] = make_uint4(0u, 0u, 0u, 0u);
}

int noalloc_device(int* dev) {
  if (hipGetDevice(dev) != hipSuccess || *dev < 0 || *dev >= NOALLOC_MAX_DEVICES)
    return MG_ERR_RUNTIME;
  return MG_OK;
}

// The current device's scratch address, set up by the first call per device:
// the symbol lookup, then one zero fill on `stream` (the look-back workspace
// protocol starts from zeroed memory; later calls ordered on a stream after it
// reuse the contents unchanged).  The set-up is refused while `stream` is being
// captured: a captured fill would not run at capture time and would run again
// on every replay.
int noalloc_scratch(hipStream_t stream, void** out) {
  int dev = -1;
  if (noalloc_device(&dev) != MG_OK) return MG_ERR_RUNTIME;
  NoallocDevice& d = g_noalloc[dev];
  void* p = d.ptr.load(std::memory_order_acquire);
  if (p == nullptr) {
    std::lock_guard<std::mutex> lock(d.mu);
    p = d.ptr.load(std::memory_order_relaxed);
    if (p == nullptr) {
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(stream, &cs) != hipSuccess) return MG_ERR_RUNTIME;
      if (cs != hipStreamCaptureStatusNone) return MG_ERR_CAPTURE;
      if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr)
        return MG_ERR_RUNTIME;
      hipLaunchKernelGGL(zero_fill_kernel, dim3(1024), dim3(256), 0, stream, (uint4*)p,
                         NOALLOC_SCRATCH_BYTES / 16);
      if (hipGetLastError() != hipSuccess) return MG_ERR_LAUNCH;
      d.ptr.store(p, std::memory_order_release);
    }
  }
  *out = p;
  return MG_OK;
}

// Workspace of the linear_scan forward alone, whatever lane width it picks.
size_t linear_fwd_ws_bytes(int64_t B, int64_t T, int64_t D) {
  size_t m = 0;
  for (int vec : {1, 2, 4})
    m = std::max(m, ew_plan(B, T, D, vec, EW_TSUB_FWD, EW_WAVES_FWD, 1).total);
  return m;
}

}  // namespace

extern "C" {

size_t mg_linear_scan_workspace_bytes(int64_t B, int64_t T, int64_t D) {
  return ew_ws_bytes(B, T, D);
}

size_t mg_log_scan_workspace_bytes(int64_t B, int64_t T, int64_t D) {
  return log_ws_bytes(B, T, D);
}

size_t mg_log_scan_state_bytes(int64_t B, int64_t T, int64_t D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (size_t)B * (size_t)((T + LOG_TSUB - 1) / LOG_TSUB) * 2 * (size_t)D * sizeof(float);
}

int mg_linear_scan_fwd(const float* a, const float* b, float* A, float* Bc, int64_t B, int64_t T,
                       int64_t D, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!a || !b || !A || !Bc || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return linear_fwd_launch(a, b, A, Bc, (float*)nullptr, B, T, D, ws, ws_bytes, stream);
}

int mg_linear_scan_fwd_noalloc(const float* a, const float* b, float* A, float* Bc, int64_t B,
                               int64_t T, int64_t D, hipStream_t stream) {
  if (!a || !b || !A || !Bc || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  if (linear_fwd_ws_bytes(B, T, D) > NOALLOC_SCRATCH_BYTES) return MG_ERR_TOO_LARGE;
  void* ws = nullptr;
  const int rc = noalloc_scratch(stream, &ws);
  if (rc != MG_OK) return rc;
  return linear_fwd_launch(a, b, A, Bc, (float*)nullptr, B, T, D, ws, NOALLOC_SCRATCH_BYTES,
                           stream);
}

int mg_scan_workspace_errors(const void* ws, unsigned* count, hipStream_t stream) {
  if (!ws || !count) return MG_ERR_ARG;
  unsigned v = 0;
  if (hipMemcpyAsync(&v, (const unsigned*)ws + MG_H_ERROR, sizeof(unsigned),
                     hipMemcpyDeviceToHost, stream) != hipSuccess)
    return MG_ERR_RUNTIME;
  if (hipStreamSynchronize(stream) != hipSuccess) return MG_ERR_RUNTIME;
  *count = v;
  return MG_OK;
}

int mg_linear_scan_noalloc_errors(unsigned* count, hipStream_t stream) {
  if (!count) return MG_ERR_ARG;
  int dev = -1;
  if (noalloc_device(&dev) != MG_OK) return MG_ERR_RUNTIME;
  const void* p = g_noalloc[dev].ptr.load(std::memory_order_acquire);
  if (p == nullptr) {  // never set up on this device: nothing has run
    *count = 0;
    return MG_OK;
  }
  return mg_scan_workspace_errors(p, count, stream);
}

int mg_linear_scan_bwd(const float* a, const float* b, const float* A, const float* Bc,
                       const float* gA, const float* gB, float* da, float* db, int64_t B,
                       int64_t T, int64_t D, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!a || !b || !A || !Bc || !gA || !gB || !da || !db || !ws || !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  const bool v4 = D % 4 == 0 && all_aligned({a, b, A, Bc, gA, gB, da, db}, 16);
  const int vec = ew_vec(B, T, D, v4, EW_WAVES_BWD * EW_TSUB_BWD);
  return by_vec(vec, [&](auto v) {
    constexpr int V = decltype(v)::value;
    EwPlan p = ew_plan(B, T, D, V, EW_TSUB_BWD, EW_WAVES_BWD, 2);
    if (ws_bytes < p.total) return MG_ERR_WORKSPACE;
    return ew_run(ew_two_launch(p, B, T, D, 4), linear_bwd_kernel<V, EW_TSUB_BWD, EW_WAVES_BWD>,
                  linear_bwd_kernel<V, EW_TSUB_BWD, EW_WAVES_BWD, EW_REDUCE>,
                  linear_bwd_kernel<V, EW_TSUB_BWD, EW_WAVES_BWD, EW_FINAL>,
                  linear_bwd_kernel<V, EW_TSUB_BWD, EW_WAVES_BWD, EW_AGG>, p, ws, stream, a, b,
                  A, Bc, gA, gB, da, db);
  });
}

size_t mg_signed_gate_scan_workspace_bytes(int64_t B, int64_t T, int64_t D) {
  return gate_ws_bytes(B, T, D);
}

int mg_signed_gate_scan_fwd(const float* s, const float* z, const float* hpre, const float* h0,
                            float* h, int64_t B, int64_t T, int64_t D, int coupled, void* ws,
                            size_t ws_bytes, hipStream_t stream) {
  if (!s || !z || !hpre || !h0 || !h || !ws || !geometry_ok(B, T, D) || (coupled & ~1))
    return MG_ERR_ARG;
  return gate_fwd_any<float>(coupled, {s, z, hpre, h0, D, 0}, h, nullptr, GateDecay{}, B, T, D, ws,
                             ws_bytes, stream);
}

int mg_signed_gate_scan_bwd(const float* s, const float* z, const float* hpre, const float* h0,
                            const float* h, const float* gh, float* ds, float* dz, float* dhpre,
                            float* dh0, int64_t B, int64_t T, int64_t D, int coupled, void* ws,
                            size_t ws_bytes, hipStream_t stream) {
  if (!s || !z || !hpre || !h0 || !h || !gh || !ds || !dz || !dhpre || !dh0 || !ws ||
      !geometry_ok(B, T, D) || (coupled & ~1))
    return MG_ERR_ARG;
  return gate_bwd_any<float>(coupled, {s, z, hpre, h0, D, 0}, h, gh, ds, dz, dhpre, dh0,
                             GateDecay{}, B, T, D, ws, ws_bytes, stream);
}

int mg_signed_gate_scan_decay_fwd(const float* s, const float* z, const float* hpre,
                                  const float* h0, const float* dt, const float* lam, float* h,
                                  int64_t B, int64_t T, int64_t D, int coupled, void* ws,
                                  size_t ws_bytes, hipStream_t stream) {
  if (!s || !z || !hpre || !h0 || !dt || !lam || !h || !ws || !geometry_ok(B, T, D) ||
      (coupled & ~1))
    return MG_ERR_ARG;
  return gate_fwd_any<float>(coupled, {s, z, hpre, h0, D, 0}, h, nullptr,
                             GateDecay{dt, lam, nullptr, nullptr}, B, T, D, ws, ws_bytes, stream);
}

int mg_signed_gate_scan_decay_bwd(const float* s, const float* z, const float* hpre,
                                  const float* h0, const float* dt, const float* lam,
                                  const float* h, const float* gh, float* ds, float* dz,
                                  float* dhpre, float* dh0, float* dlam, float* ddt, int64_t B,
                                  int64_t T, int64_t D, int coupled, void* ws, size_t ws_bytes,
                                  hipStream_t stream) {
  if (!s || !z || !hpre || !h0 || !dt || !lam || !h || !gh || !ds || !dz || !dhpre || !dh0 ||
      !ws || !geometry_ok(B, T, D) || (coupled & ~1))
    return MG_ERR_ARG;
  return gate_bwd_any<float>(coupled, {s, z, hpre, h0, D, 0}, h, gh, ds, dz, dhpre, dh0,
                             GateDecay{dt, lam, dlam, ddt}, B, T, D, ws, ws_bytes, stream);
}

size_t mg_mingru_gate_scan_workspace_bytes(int64_t B, int64_t T, int64_t D) {
  return gate_ws_bytes(B, T, D);
}

int mg_mingru_gate_scan_fwd(const float* k, const float* hpre, const float* log_h0, float* h,
                            int64_t B, int64_t T, int64_t D, void* ws, size_t ws_bytes,
                            hipStream_t stream) {
  if (!k || !hpre || !log_h0 || !h || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return gate_fwd_any<float>(GATE_MINGRU, {k, hpre, nullptr, log_h0, D, 0}, h, nullptr,
                             GateDecay{}, B, T, D, ws, ws_bytes, stream);
}

int mg_mingru_gate_scan_bwd(const float* k, const float* hpre, const float* log_h0,
                            const float* h, const float* gh, float* dk, float* dhpre,
                            float* dlog_h0, int64_t B, int64_t T, int64_t D, void* ws,
                            size_t ws_bytes, hipStream_t stream) {
  if (!k || !hpre || !log_h0 || !h || !gh || !dk || !dhpre || !dlog_h0 || !ws ||
      !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  return gate_bwd_any<float>(GATE_MINGRU, {k, hpre, nullptr, log_h0, D, 0}, h, gh, dk, dhpre,
                             nullptr, dlog_h0, GateDecay{}, B, T, D, ws, ws_bytes, stream);
}

int mg_mingru_gate_scan_decay_fwd(const float* k, const float* hpre, const float* log_h0,
                                  const float* dt, const float* lam, float* h, int64_t B,
                                  int64_t T, int64_t D, void* ws, size_t ws_bytes,
                                  hipStream_t stream) {
  if (!k || !hpre || !log_h0 || !dt || !lam || !h || !ws || !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  return gate_fwd_any<float>(GATE_MINGRU, {k, hpre, nullptr, log_h0, D, 0}, h, nullptr,
                             GateDecay{dt, lam, nullptr, nullptr}, B, T, D, ws, ws_bytes, stream);
}

int mg_mingru_gate_scan_decay_bwd(const float* k, const float* hpre, const float* log_h0,
                                  const float* dt, const float* lam, const float* h,
                                  const float* gh, float* dk, float* dhpre, float* dlog_h0,
                                  float* dlam, float* ddt, int64_t B, int64_t T, int64_t D,
                                  void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!k || !hpre || !log_h0 || !dt || !lam || !h || !gh || !dk || !dhpre || !dlog_h0 || !ws ||
      !geometry_ok(B, T, D))
    return MG_ERR_ARG;
  return gate_bwd_any<float>(GATE_MINGRU, {k, hpre, nullptr, log_h0, D, 0}, h, gh, dk, dhpre,
                             nullptr, dlog_h0, GateDecay{dt, lam, dlam, ddt}, B, T, D, ws,
                             ws_bytes, stream);
}

int mg_gate_scan_rows_fwd(int kind, const float* p0, const float* p1, const float* p2, int64_t ld,
                          const float* h0, float h0_const, const float* dt, const float* lam,
                          float* h, int64_t B, int64_t T, int64_t D, void* ws, size_t ws_bytes,
                          hipStream_t stream) {
  if (kind < GATE_SIGNED || kind > GATE_MINGRU || !p0 || !p1 || (kind != GATE_MINGRU && !p2) ||
      !h || !ws || !geometry_ok(B, T, D) || ld < D || !dt != !lam)
    return MG_ERR_ARG;
  return gate_fwd_any<float>(kind, {p0, p1, p2, h0, ld, 0, h0_const}, h, nullptr,
                             GateDecay{dt, lam, nullptr, nullptr}, B, T, D, ws, ws_bytes, stream);
}

int mg_gate_scan_rows_bwd(int kind, const float* p0, const float* p1, const float* p2, int64_t ld,
                          const float* h0, float h0_const, const float* dt, const float* lam,
                          const float* h, const float* gh, float* d0, float* d1, float* d2,
                          float* dh0, float* dlam, float* ddt, int64_t B, int64_t T, int64_t D,
                          void* ws, size_t ws_bytes, hipStream_t stream) {
  if (kind < GATE_SIGNED || kind > GATE_MINGRU || !p0 || !p1 || (kind != GATE_MINGRU && !p2) ||
      !h || !gh || !d0 || !d1 || (kind != GATE_MINGRU && !d2) || !ws || !geometry_ok(B, T, D) ||
      ld < D || !dt != !lam)
    return MG_ERR_ARG;
  return gate_bwd_any<float>(kind, {p0, p1, p2, h0, ld, 0, h0_const}, h, gh, d0, d1, d2, dh0,
                             GateDecay{dt, lam, dlam, ddt}, B, T, D, ws, ws_bytes, stream);
}

int64_t mg_gate_decay_dlam_rows(int64_t B, int64_t T, int64_t D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return B * ((T + GATE_WAVES_BWD * GATE_TSUB_BWD - 1) / (GATE_WAVES_BWD * GATE_TSUB_BWD));
}

int64_t mg_gate_decay_ddt_rows(int64_t B, int64_t T, int64_t D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (D + MG_WAVE - 1) / MG_WAVE;
}

int mg_log_scan_fwd(const float* lc, const float* lv, float* h, float* hstate, int64_t B,
                    int64_t T, int64_t D, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!lc || !lv || !h || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return log_fwd_launch(lc, lv, h, hstate, B, T, D, ws, ws_bytes, stream);
}

int mg_log_scan_bwd(const float* lc, const float* lv, const float* h, const float* hstate,
                    const float* gh, float* dlc, float* dlv, int64_t B, int64_t T, int64_t D,
                    void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!lc || !lv || !h || !gh || !dlc || !dlv || !ws || !geometry_ok(B, T, D)) return MG_ERR_ARG;
  return log_bwd_launch(lc, lv, h, hstate, gh, dlc, dlv, B, T, D, ws, ws_bytes, stream);
}

}  // extern "C"
