// Column sums of a dense matrix (gfx950): the bias gradients of joined projections inside a
// captured graph.
//
// torch's sum over rows splits a long column over workgroups that meet through counters it
// clears with a memset.  As a node of a HIP graph that memset has not cleared them on replays
// after the first: rows of 772 or 896 columns, the joined widths of a DeltaMinGRU and a
// GivensMinGRU layer of 256, gave bias gradients off by their own size.  Here nothing is
// cleared and no workgroup waits for another: the first launch writes a partial sum per row
// chunk and column, the second adds a column's partials in order.
//
// Split: a workgroup takes 64 columns and a chunk of rows, a wave every fourth row of it (256
// or 128 consecutive bytes), a lane its column in four fp32 accumulators.  Chunks have at
// least 64 rows, and there are at most 256, so the partials are no more than 1/16 of the
// matrix.  Bound by the read of the matrix.  (8000, 772) fp32 17 us, torch's sum 21, error
// against float64 1.3e-7 and 1.7e-7; (16384, 3072) bf16 38 us, torch 33; (16384, 896) fp32 31
// us, torch 25.  So eager passes keep torch's.
#include "mg_common.h"

namespace {

typedef uint16_t u16;
constexpr int CS_WAVES = 4;
constexpr int CS_NT = CS_WAVES * MG_WAVE;
constexpr int64_t CS_MIN_ROWS = 64, CS_MAX_CHUNKS = 256;

__device__ __forceinline__ float ld1(const float* p) { return *p; }
__device__ __forceinline__ float ld1(const u16* p) { return __uint_as_float((unsigned)*p << 16); }
__device__ __forceinline__ void st1(float* p, float x) { *p = x; }
__device__ __forceinline__ void st1(u16* p, float x) { *p = __builtin_bit_cast(u16, (__bf16)x); }

template <typename E>
__global__ __launch_bounds__(CS_NT) void column_partials(const E* __restrict__ x,
                                                         float* __restrict__ part, int64_t rows,
                                                         int64_t N, int64_t chunk) {
  __shared__ float s[CS_WAVES][MG_WAVE];
  const int lane = threadIdx.x & (MG_WAVE - 1), w = threadIdx.x / MG_WAVE;
  const int64_t col = (int64_t)blockIdx.x * MG_WAVE + lane, c = col < N ? col : N - 1;
  const int64_t r0 = (int64_t)blockIdx.y * chunk;
  const int64_t r1 = r0 + chunk < rows ? r0 + chunk : rows;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  int64_t r = r0 + w;
  for (; r + 3 * CS_WAVES < r1; r += 4 * CS_WAVES) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] += ld1(x + (r + i * CS_WAVES) * N + c);
  }
  for (; r < r1; r += CS_WAVES) a[0] += ld1(x + r * N + c);
  s[w][lane] = (a[0] + a[1]) + (a[2] + a[3]);
  __syncthreads();
  if (w == 0 && col < N)
    part[(int64_t)blockIdx.y * N + col] = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
}

template <typename E>
__global__ __launch_bounds__(CS_NT) void column_totals(const float* __restrict__ part,
                                                       E* __restrict__ out, int64_t N, int chunks) {
  const int64_t col = (int64_t)blockIdx.x * CS_NT + threadIdx.x;
  if (col >= N) return;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  int k = 0;
  for (; k + 4 <= chunks; k += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] += part[(int64_t)(k + i) * N + col];
  }
  for (; k < chunks; ++k) a[0] += part[(int64_t)k * N + col];
  st1(out + col, (a[0] + a[1]) + (a[2] + a[3]));
}

// Row chunks of a launch, and the rows of each: every chunk has at least one row.
struct CsSplit {
  int64_t chunk;
  int chunks;
};
CsSplit cs_split(int64_t rows) {
  int64_t n = (rows + CS_MIN_ROWS - 1) / CS_MIN_ROWS;
  n = n < CS_MAX_CHUNKS ? n : CS_MAX_CHUNKS;
  const int64_t chunk = (rows + n - 1) / n;
  return {chunk, (int)((rows + chunk - 1) / chunk)};
}

// Rows and columns whose launches and offsets stay in range.
bool cs_ok(int64_t rows, int64_t N) {
  return rows >= 1 && N >= 1 && N <= (1 << 24) && rows <= (1ll << 36);
}

template <typename E>
int cs_run(const void* x, void* out, int64_t rows, int64_t N, float* ws, hipStream_t stream) {
  const CsSplit p = cs_split(rows);
  hipLaunchKernelGGL(column_partials<E>, dim3((unsigned)((N + MG_WAVE - 1) / MG_WAVE), p.chunks),
                     dim3(CS_NT), 0, stream, (const E*)x, ws, rows, N, p.chunk);
  hipLaunchKernelGGL(column_totals<E>, dim3((unsigned)((N + CS_NT - 1) / CS_NT)), dim3(CS_NT), 0,
                     stream, ws, (E*)out, N, p.chunks);
  return hipGetLastError() == hipSuccess ? MG_OK : MG_ERR_LAUNCH;
}

}  // namespace

extern "C" {

size_t mg_column_sums_workspace_bytes(int64_t rows, int64_t N) {
  return cs_ok(rows, N) ? (size_t)cs_split(rows).chunks * N * sizeof(float) : 0;
}

int mg_column_sums(const void* x, void* out, int64_t rows, int64_t N, int dtype, void* ws,
                   size_t ws_bytes, hipStream_t stream) {
  if (!x || !out || !ws || !cs_ok(rows, N) || (dtype & ~1)) return MG_ERR_ARG;
  if (ws_bytes < mg_column_sums_workspace_bytes(rows, N)) return MG_ERR_WORKSPACE;
  return dtype ? cs_run<u16>(x, out, rows, N, (float*)ws, stream)
               : cs_run<float>(x, out, rows, N, (float*)ws, stream);
}

}  // extern "C"
