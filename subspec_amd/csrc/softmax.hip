// softmax(logits / temperature) over the vocabulary, in the logits dtype: the draft's probability
// rows that feed the top-k expansion.
//
// Replaces ClassicSDDraftModel.forward(with_softmax=True):
//   torch.softmax(logits / self.draft_params.temperature, dim=-1)
// (specdecodes/models/draft_models/classic_sd.py:10-16).  As there, the quotient is rounded to the
// tensor dtype first (an elementwise tensor op), the softmax is evaluated in fp32 on the rounded
// values (maximum, exp(x - max), sum, quotient) and each probability is rounded once.
//
// Many rows: one workgroup per row, three passes over the row (maximum, sum, write); a 152064-entry
// 16-bit row is 297 KB, so the second and third pass are served by L2.  A draft step has 1 to 16
// rows, far too few workgroups for the chip: then every row is cut into slices, one launch reduces
// each slice to (maximum, sum of exp relative to it) and a second one combines the slices of its row
// and writes its slice (the sums differ from the one-workgroup order only in fp32 rounding).
#include "common.h"
#include <algorithm>

namespace subspec {

constexpr int kSmThreads = 1024;

template <int DT>
__device__ __forceinline__ float scaled(const void* p, int64_t i, const Divisor& t) {
  return Elem<DT>::round(div_rn(Elem<DT>::load(p, i), t));   // IEEE quotient, then one rounding to the row dtype
}

template <int DT>
__global__ __launch_bounds__(kSmThreads) void softmax_temperature_kernel(const void* __restrict__ logits, void* __restrict__ out,
                                                                          int64_t vocab, Divisor temperature) {
  __shared__ float red[kSmThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * vocab;
  const int tid = threadIdx.x;
  float m = -INFINITY;
  for (int64_t i = tid; i < vocab; i += kSmThreads) m = fmaxf(m, scaled<DT>(logits, base + i, temperature));
  m = block_max<kSmThreads>(m, red);
  float s = 0.f;
  for (int64_t i = tid; i < vocab; i += kSmThreads) s += expf(scaled<DT>(logits, base + i, temperature) - m);
  s = block_sum<kSmThreads>(s, red);
  for (int64_t i = tid; i < vocab; i += kSmThreads)
    Elem<DT>::store(out, base + i, expf(scaled<DT>(logits, base + i, temperature) - m) / s);
}

// ---- few rows: slices of kSliceElems elements, grid (slices, rows)
// Two dependent launches of a few dozen workgroups a row: nothing but latency, so a thread has its 16 elements in flight before
// anything else (16-byte pieces; single elements where the row length or an address does not allow them) and no reduction meets a
// second barrier.  8 rows x 152064 bf16: 6.1 + 6.5 us with single elements and two workgroup reductions in each, 4.3 + 5.6 now.
constexpr int kSliceThreads = 256;
constexpr int kSliceElems = 4096;
constexpr int kMaxSlices = 1024;
constexpr int kSlicePer = kSliceElems / kSliceThreads;

// the thread's elements of a slice of `n`, rounded quotients; piece p of VEC elements starts at (p * kSliceThreads + thread) * VEC
template <int DT, int VEC> struct SmElems;
template <int DT> struct SmElems<DT, 1> {
  typename Elem<DT>::storage raw[kSlicePer];
  __device__ __forceinline__ void load(const void* p, int64_t base, int n) {
#pragma unroll
    for (int j = 0; j < kSlicePer; ++j) raw[j] = ((const typename Elem<DT>::storage*)p)[base + min(j * kSliceThreads + (int)threadIdx.x, n - 1)];
  }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int j = 0; j < kSlicePer; ++j) v[j] = Elem<DT>::load(&raw[j], 0);
  }
  static __device__ __forceinline__ void store(void* p, int64_t base, int n, const float* v) {
#pragma unroll
    for (int j = 0; j < kSlicePer; ++j)
      if (j * kSliceThreads + (int)threadIdx.x < n) Elem<DT>::store(p, base + j * kSliceThreads + threadIdx.x, v[j]);
  }
};
template <int DT> struct SmElems<DT, 8> {
  dec_u4 raw[kSlicePer / 8];
  __device__ __forceinline__ void load(const void* p, int64_t base, int n) {
#pragma unroll
    for (int j = 0; j < kSlicePer / 8; ++j)
      raw[j] = *(const dec_u4*)((const uint16_t*)p + base + min((j * kSliceThreads + (int)threadIdx.x) * 8, n - 8));
  }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int j = 0; j < kSlicePer / 8; ++j) unpack8<DT>(raw[j], v + 8 * j);
  }
  static __device__ __forceinline__ void store(void* p, int64_t base, int n, const float* v) {
#pragma unroll
    for (int j = 0; j < kSlicePer / 8; ++j)
      if ((j * kSliceThreads + (int)threadIdx.x) * 8 < n)
        *(dec_u4*)((uint16_t*)p + base + (j * kSliceThreads + threadIdx.x) * 8) = pack8<DT>(v + 8 * j);
  }
};
template <> struct SmElems<SUBSPEC_F32, 4> {
  float4 raw[kSlicePer / 4];
  __device__ __forceinline__ void load(const void* p, int64_t base, int n) {
#pragma unroll
    for (int j = 0; j < kSlicePer / 4; ++j) raw[j] = *(const float4*)((const float*)p + base + min((j * kSliceThreads + (int)threadIdx.x) * 4, n - 4));
  }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int j = 0; j < kSlicePer / 4; ++j) { v[4 * j] = raw[j].x; v[4 * j + 1] = raw[j].y; v[4 * j + 2] = raw[j].z; v[4 * j + 3] = raw[j].w; }
  }
  static __device__ __forceinline__ void store(void* p, int64_t base, int n, const float* v) {
#pragma unroll
    for (int j = 0; j < kSlicePer / 4; ++j)
      if ((j * kSliceThreads + (int)threadIdx.x) * 4 < n)
        *(float4*)((float*)p + base + (j * kSliceThreads + threadIdx.x) * 4) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
  }
};

template <int DT, int VEC>
__global__ __launch_bounds__(kSliceThreads) void softmax_slice_stats_kernel(const void* __restrict__ logits, float2* __restrict__ stats,
                                                                            int64_t vocab, Divisor temperature) {
  __shared__ float red_m[kSliceThreads / kWave], red_s[kSliceThreads / kWave];
  const int64_t i0 = (int64_t)blockIdx.x * kSliceElems, base = (int64_t)blockIdx.y * vocab + i0;
  const int n = (int)min((int64_t)kSliceElems, vocab - i0);
  SmElems<DT, VEC> e;
  e.load(logits, base, n);
  float v[kSlicePer];
  e.get(v);
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < kSlicePer; ++j) {
    const int i = (j / VEC * kSliceThreads + (int)threadIdx.x) * VEC + j % VEC;
    v[j] = i < n ? Elem<DT>::round(div_rn(v[j], temperature)) : -INFINITY;
    m = fmaxf(m, v[j]);
  }
  m = wave_max(m);
  if ((threadIdx.x & (kWave - 1)) == 0) red_m[threadIdx.x / kWave] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSliceThreads / kWave; ++w) m = fmaxf(m, red_m[w]);
  float s = 0.f;
  if (m != -INFINITY) {
#pragma unroll
    for (int j = 0; j < kSlicePer; ++j) s += expf(v[j] - m);
  }
  s = wave_sum(s);
  if ((threadIdx.x & (kWave - 1)) == 0) red_s[threadIdx.x / kWave] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    s = red_s[0];
#pragma unroll
    for (int w = 1; w < kSliceThreads / kWave; ++w) s += red_s[w];
    stats[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = make_float2(m, s);
  }
}

// Every wavefront combines all slices of its row by itself (38 of a 152064-entry row: one request a lane).
template <int DT, int VEC>
__global__ __launch_bounds__(kSliceThreads) void softmax_slice_write_kernel(const void* __restrict__ logits, void* __restrict__ out,
                                                                            const float2* __restrict__ stats, int64_t vocab,
                                                                            Divisor temperature) {
  const int slices = gridDim.x, lane = threadIdx.x & (kWave - 1);
  const float2* st = stats + (int64_t)blockIdx.y * slices;
  const int64_t i0 = (int64_t)blockIdx.x * kSliceElems, base = (int64_t)blockIdx.y * vocab + i0;
  const int n = (int)min((int64_t)kSliceElems, vocab - i0);
  SmElems<DT, VEC> e;
  e.load(logits, base, n);
  float m = -INFINITY, s = 0.f;
  for (int c = lane; c < slices; c += kWave) m = fmaxf(m, st[c].x);
  m = wave_max(m);
  for (int c = lane; c < slices; c += kWave)
    if (st[c].x != -INFINITY) s += st[c].y * expf(st[c].x - m);
  s = wave_sum(s);
  float v[kSlicePer];
  e.get(v);
#pragma unroll
  for (int j = 0; j < kSlicePer; ++j) v[j] = expf(Elem<DT>::round(div_rn(v[j], temperature)) - m) / s;
  SmElems<DT, VEC>::store(out, base, n, v);
}

// TemperatureLogitsWarper as a stand-alone elementwise pass: out = logits / temperature in the logits dtype
template <int DT>
__global__ __launch_bounds__(256) void temperature_warp_kernel(const void* __restrict__ logits, void* __restrict__ out,
                                                               int64_t n, Divisor temperature) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    Elem<DT>::store(out, i, div_rn(Elem<DT>::load(logits, i), temperature));
}

}  // namespace subspec

using namespace subspec;

extern "C" int subspec_temperature_warp(const void* logits, void* out, int dtype, int64_t n, float temperature,
                                        void* stream) {
  if (!dtype_ok(dtype)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "temperature_warp: unknown dtype %d", dtype);
  if (!logits || !out) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "temperature_warp: null pointer argument");
  if (n <= 0) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "temperature_warp: n=%lld must be positive", (long long)n);
  if (!(temperature > 0.f) || temperature == INFINITY)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "temperature_warp: temperature must be positive and finite");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)std::min<int64_t>((n + 255) / 256, 8192));
  const Divisor t = make_divisor(temperature);
  if (dtype == SUBSPEC_F32)
    hipLaunchKernelGGL((temperature_warp_kernel<SUBSPEC_F32>), grid, dim3(256), 0, st, logits, out, n, t);
  else if (dtype == SUBSPEC_F16)
    hipLaunchKernelGGL((temperature_warp_kernel<SUBSPEC_F16>), grid, dim3(256), 0, st, logits, out, n, t);
  else
    hipLaunchKernelGGL((temperature_warp_kernel<SUBSPEC_BF16>), grid, dim3(256), 0, st, logits, out, n, t);
  SUBSPEC_CHECK_HIP(hipGetLastError());
  return SUBSPEC_OK;
}

extern "C" size_t subspec_softmax_temperature_workspace(int64_t rows, int64_t vocab) {
  const int64_t slices = (vocab + kSliceElems - 1) / kSliceElems;
  if (rows <= 0 || rows >= 256 || slices <= 1 || slices > kMaxSlices) return 0;
  return align_up((size_t)rows * slices * sizeof(float2), 256);
}

extern "C" int subspec_softmax_temperature(const void* logits, void* out, int dtype, int64_t rows, int64_t vocab,
                                           float temperature, void* workspace, size_t workspace_bytes, void* stream) {
  if (!dtype_ok(dtype)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "softmax_temperature: unknown dtype %d", dtype);
  if (!logits || !out) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "softmax_temperature: null pointer argument");
  if (rows <= 0 || vocab <= 0) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "softmax_temperature: rows=%lld vocab=%lld", (long long)rows, (long long)vocab);
  if (!(temperature > 0.f)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "softmax_temperature: temperature must be positive");
  if (rows > 0x7fffffff) SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "softmax_temperature: too many rows");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)rows);
  const Divisor t = make_divisor(temperature);
  const int64_t slices = (vocab + kSliceElems - 1) / kSliceElems;
  if (workspace && rows < 256 && slices > 1 && slices <= kMaxSlices) {
    if (workspace_bytes < subspec_softmax_temperature_workspace(rows, vocab))
      SUBSPEC_FAIL(SUBSPEC_ERR_WORKSPACE, "softmax_temperature: workspace of %zu bytes is smaller than the %zu required",
                   workspace_bytes, subspec_softmax_temperature_workspace(rows, vocab));
    if ((uintptr_t)workspace % 8 != 0) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "softmax_temperature: workspace must be 8-byte aligned");
    const dim3 g2((unsigned)slices, (unsigned)rows);
    float2* stats = (float2*)workspace;
    const int vec = 16 / (int)dtype_size(dtype);
    const bool wide = vocab % vec == 0 && ((uintptr_t)logits | (uintptr_t)out) % 16 == 0;
#define SUBSPEC_SM_SLICED(DT, VEC)                                                                                   \
    hipLaunchKernelGGL((softmax_slice_stats_kernel<DT, VEC>), g2, dim3(kSliceThreads), 0, st, logits, stats, vocab, t);     \
    hipLaunchKernelGGL((softmax_slice_write_kernel<DT, VEC>), g2, dim3(kSliceThreads), 0, st, logits, out, stats, vocab, t)
    if (dtype == SUBSPEC_F32) { if (wide) { SUBSPEC_SM_SLICED(SUBSPEC_F32, 4); } else { SUBSPEC_SM_SLICED(SUBSPEC_F32, 1); } }
    else if (dtype == SUBSPEC_F16) { if (wide) { SUBSPEC_SM_SLICED(SUBSPEC_F16, 8); } else { SUBSPEC_SM_SLICED(SUBSPEC_F16, 1); } }
    else { if (wide) { SUBSPEC_SM_SLICED(SUBSPEC_BF16, 8); } else { SUBSPEC_SM_SLICED(SUBSPEC_BF16, 1); } }
#undef SUBSPEC_SM_SLICED
    SUBSPEC_CHECK_HIP(hipGetLastError());
    return SUBSPEC_OK;
  }
  if (dtype == SUBSPEC_F32)
    hipLaunchKernelGGL((softmax_temperature_kernel<SUBSPEC_F32>), grid, dim3(kSmThreads), 0, st, logits, out, vocab, t);
  else if (dtype == SUBSPEC_F16)
    hipLaunchKernelGGL((softmax_temperature_kernel<SUBSPEC_F16>), grid, dim3(kSmThreads), 0, st, logits, out, vocab, t);
  else
    hipLaunchKernelGGL((softmax_temperature_kernel<SUBSPEC_BF16>), grid, dim3(kSmThreads), 0, st, logits, out, vocab, t);
  SUBSPEC_CHECK_HIP(hipGetLastError());
  return SUBSPEC_OK;
}
