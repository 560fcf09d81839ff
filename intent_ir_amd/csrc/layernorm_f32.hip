// LayerNorm forward in float32 over the last axis: x, y f32 [M, N]; w, b f32 [N]; mean, rstd
// f32 [M] (null: not written).  The op order of the reference LayerNorm IR
// (pipeline/tilelang/core.py:1322-1384, pipeline/cuda/core.py:496-546) and of its CUDA
// kernel (backends/cuda/runtime/kernels/layernorm.cuh:11-98):
//   mean = sum(x) / N;  d = x - mean;  var = sum(d * d) / N;  rstd = 1 / sqrt(var + eps);
//   y = ((d * rstd) * w) + b
// with every step a separately rounded f32 operation (no fused multiply-adds: the kernels
// below are compiled with contraction off), so y differs from numpy's only through the order
// in which the two row sums are accumulated.
//
// Forms, all but the last reading x from HBM once with the row held in registers:
//  * 4 <= N <= 256: 2-64 lanes per row, one vector each (layernorm_rows_f32_grouped);
//  * N <= 4099: a wave per row (kVpl 16-byte vectors per lane), 4 rows per 256-thread workgroup
//    with w and b staged in LDS once per workgroup (instead of once per row from L2);
//  * 4099 < N <= 65539: kW waves per row, the wave sums exchanged through LDS and folded in a
//    fixed order, w and b from L2;
//    these two come twice: kU = false for N % 4 == 0 and 16-byte aligned tensors; kU = true for rows
//    that start at any 4-byte boundary (odd N, unaligned views): the same 16-byte accesses, of
//    which gfx950 asks 4-byte alignment only, from the row's own start, and the last N % 4
//    elements on the row's first lanes;
//  * longer rows, and bases that are not 4-byte aligned: a 256-thread workgroup per row that
//    reads x three times (the second and third reads of a row come from L2).
#include <type_traits>

#include "common.hpp"

namespace ihip {

#pragma clang fp contract(off)

// Rows (waves) per workgroup of the one-wave-per-row form: 4 ran [8192, 4096] 2% ahead of 16
// (45.7 against 46.8 us, graph replays, rotated buffers) and of 2 or 8.
constexpr int kLn32Rows = 4;

// A 16-byte vector of a row, streamed past the caches: 16-byte aligned, or (kU) at any 4-byte
// boundary.  At [8192, 4099] the kU form runs 52.4 us (5.13 TB/s; 47.9 aligned at N = 4096, and
// 107.9 for the three-pass form that these rows took before); through the caches, which could
// merge the lines that neighbouring stores and rows share, its loads and stores took 54.1, its
// stores alone 52.1, and at [4096, 8195] 56.7 streamed against 61.2 and 58.1.
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
template <bool kU>
using ln32_vec = std::conditional_t<kU, f32x4_u, f32x4>;

template <bool kU>
__device__ __forceinline__ f32x4 ln32_load(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const ln32_vec<kU>*>(p));
}
template <bool kU>
__device__ __forceinline__ f32x4 ln32_load_wb(const float* p) {
  return *reinterpret_cast<const ln32_vec<kU>*>(p);
}
template <bool kU>
__device__ __forceinline__ void ln32_store(float* p, f32x4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<ln32_vec<kU>*>(p));
}

// n4 = N / 4 whole vectors per row; kU: the N % 4 elements after them are on lanes 0..2.
template <int kVpl, bool kU>
__global__ __launch_bounds__(64 * kLn32Rows) void layernorm_rows_f32_wave(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, float* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t M, int n4, int N, float eps) {
  __shared__ f32x4 w_lds[kVpl * kWave], b_lds[kVpl * kWave];
  const int lane = threadIdx.x & 63;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kLn32Rows + (threadIdx.x >> 6);
  const bool live = row0 < M;  // waves past the last row read row M - 1 and store nothing
  const int64_t row = live ? row0 : M - 1;
  const float* xr = x + row * N + 4 * lane;
  f32x4 xv[kVpl];
#pragma unroll
  for (int i = 0; i < kVpl; ++i)
    xv[i] = lane + i * kWave < n4 ? ln32_load<kU>(xr + 4 * i * kWave) : f32x4{0.f, 0.f, 0.f, 0.f};
  const int te = 4 * n4 + lane;  // this lane's element of the tail
  const bool tail = kU && te < N;
  float xt = 0.f, wt = 0.f, bt = 0.f;
  if (tail) {
    xt = x[row * N + te];
    wt = w[te];
    bt = b[te];
  }
  for (int t = threadIdx.x; t < n4; t += 64 * kLn32Rows) {  // staged after the row loads are issued
    w_lds[t] = ln32_load_wb<kU>(w + 4 * t);
    b_lds[t] = ln32_load_wb<kU>(b + 4 * t);
  }
  float s = xt;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) s += (xv[i][0] + xv[i][1]) + (xv[i][2] + xv[i][3]);  // padding holds +0
  const float mean = wave_sum(s) / static_cast<float>(N);
  const float dt = xt - mean;
  float q = tail ? dt * dt : 0.f;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) {
    const bool in = lane + i * kWave < n4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = xv[i][j] - mean;
      q += in ? d * d : 0.f;
    }
  }
  const float rstd = 1.0f / sqrtf(wave_sum(q) / static_cast<float>(N) + eps);
  __syncthreads();  // w and b staged
  float* yr = y + row * N + 4 * lane;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) {
    const int idx = lane + i * kWave;  // lanes past n4 read LDS entries never staged and store nothing
    const f32x4 wv = w_lds[idx], bv = b_lds[idx];
    f32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = ((xv[i][j] - mean) * rstd) * wv[j] + bv[j];
    if (live && idx < n4) ln32_store<kU>(yr + 4 * i * kWave, o);
  }
  if (live && tail) y[row * N + te] = (dt * rstd) * wt + bt;
  if (live && lane == 0) {
    if (mean_out != nullptr) mean_out[row] = mean;
    if (rstd_out != nullptr) rstd_out[row] = rstd;
  }
}

// Short rows (4 <= N <= 4 G): G lanes per row, one vector each, kR rows per group with every load
// issued before the first is used, any 4-byte boundary.  The row's last vector starts 4 before its
// end: the elements it shares with the one before it (the first `dup`) are left out of the sums and
// stored twice with the same value.
template <int G, int kR>
__global__ __launch_bounds__(256) void layernorm_rows_f32_grouped(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, float* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t M, int N, float eps) {
  const int lig = threadIdx.x & (G - 1);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * (256 / G) * kR + threadIdx.x / G;
  const bool in = 4 * lig < N;  // lanes past the row hold its last vector and leave all of it out
  const int start = 4 * lig < N - 4 ? 4 * lig : N - 4, dup = in ? 4 * lig - start : 4;
  f32x4 xv[kR];
#pragma unroll
  for (int rr = 0; rr < kR; ++rr) {
    const int64_t row = row0 + rr * (256 / G);
    xv[rr] = ln32_load<true>(x + (row < M ? row : M - 1) * N + start);
  }
  const f32x4 wv = ln32_load_wb<true>(w + start), bv = ln32_load_wb<true>(b + start);
#pragma unroll
  for (int rr = 0; rr < kR; ++rr) {
    const int64_t row = row0 + rr * (256 / G);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) s += j >= dup ? xv[rr][j] : 0.f;
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
    const float mean = s / static_cast<float>(N);
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = xv[rr][j] - mean;
      q += j >= dup ? d * d : 0.f;
    }
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) q += __shfl_xor(q, off, kWave);
    const float rstd = 1.0f / sqrtf(q / static_cast<float>(N) + eps);
    if (row < M) {
      f32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = ((xv[rr][j] - mean) * rstd) * wv[j] + bv[j];
      if (in) ln32_store<true>(y + row * N + start, o);
      if (lig == 0) {
        if (mean_out != nullptr) mean_out[row] = mean;
        if (rstd_out != nullptr) rstd_out[row] = rstd;
      }
    }
  }
}

// kW waves per row, one row per workgroup: wave v holds the vectors (v * 64 + lane) + i * 64 * kW.
template <int kVpl, int kW, bool kU>
__global__ __launch_bounds__(64 * kW) void layernorm_rows_f32_multi(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, float* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int n4, int N, float eps) {
  __shared__ float part_s[kW], part_q[kW];
  const int lane = threadIdx.x & 63, v = threadIdx.x >> 6;
  const int64_t row = blockIdx.x;
  const int base = v * kWave + lane;
  const float* xr = x + row * N + 4 * base;
  f32x4 xv[kVpl];
#pragma unroll
  for (int i = 0; i < kVpl; ++i)
    xv[i] = base + i * kWave * kW < n4 ? ln32_load<kU>(xr + 4 * i * kWave * kW) : f32x4{0.f, 0.f, 0.f, 0.f};
  const int te = 4 * n4 + base;  // this thread's element of the tail
  const bool tail = kU && te < N;
  const float xt = tail ? x[row * N + te] : 0.f;
  float s = xt;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) s += (xv[i][0] + xv[i][1]) + (xv[i][2] + xv[i][3]);
  s = wave_sum(s);
  if (lane == 0) part_s[v] = s;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int k = 0; k < kW; ++k) tot += part_s[k];
  const float mean = tot / static_cast<float>(N);
  const float dt = xt - mean;
  float q = tail ? dt * dt : 0.f;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) {
    const bool in = base + i * kWave * kW < n4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = xv[i][j] - mean;
      q += in ? d * d : 0.f;
    }
  }
  q = wave_sum(q);
  if (lane == 0) part_q[v] = q;
  __syncthreads();
  float qt = 0.f;
#pragma unroll
  for (int k = 0; k < kW; ++k) qt += part_q[k];
  const float rstd = 1.0f / sqrtf(qt / static_cast<float>(N) + eps);
  float* yr = y + row * N + 4 * base;
#pragma unroll
  for (int i = 0; i < kVpl; ++i) {
    const int idx = base + i * kWave * kW;
    if (idx < n4) {
      const f32x4 wv = ln32_load_wb<kU>(w + 4 * idx), bv = ln32_load_wb<kU>(b + 4 * idx);
      f32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = ((xv[i][j] - mean) * rstd) * wv[j] + bv[j];
      ln32_store<kU>(yr + 4 * i * kWave * kW, o);
    }
  }
  if (tail) y[row * N + te] = (dt * rstd) * w[te] + b[te];
  if (v == 0 && lane == 0) {
    if (mean_out != nullptr) mean_out[row] = mean;
    if (rstd_out != nullptr) rstd_out[row] = rstd;
  }
}

// Any N and alignment: one row per 256-thread workgroup, element-wise, three passes over x.
constexpr int kLn32AnyThreads = 256;

__global__ __launch_bounds__(kLn32AnyThreads) void layernorm_rows_f32_any(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, float* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t N, float eps) {
  __shared__ float scratch[kLn32AnyThreads / kWave];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const float* xr = x + row * N;
  float* yr = y + row * N;
  float s = 0.f;
  for (int64_t i = tid; i < N; i += kLn32AnyThreads) s += xr[i];
  const float mean = block_sum(s, scratch) / static_cast<float>(N);
  float q = 0.f;
  for (int64_t i = tid; i < N; i += kLn32AnyThreads) {
    const float d = xr[i] - mean;
    q += d * d;
  }
  const float rstd = 1.0f / sqrtf(block_sum(q, scratch) / static_cast<float>(N) + eps);
  for (int64_t i = tid; i < N; i += kLn32AnyThreads) yr[i] = ((xr[i] - mean) * rstd) * w[i] + b[i];
  if (tid == 0) {
    if (mean_out != nullptr) mean_out[row] = mean;
    if (rstd_out != nullptr) rstd_out[row] = rstd;
  }
}

template <int kVpl, bool kU>
static void launch_ln32_wave(const float* x, const float* w, const float* b, float* y, float* mean, float* rstd,
                             int64_t M, int n4, int N, float eps, hipStream_t s) {
  const int64_t blocks = (M + kLn32Rows - 1) / kLn32Rows;
  layernorm_rows_f32_wave<kVpl, kU><<<dim3(static_cast<unsigned>(blocks)), dim3(64 * kLn32Rows), 0, s>>>(
      x, w, b, y, mean, rstd, M, n4, N, eps);
}

// Two rows per group, or one where that would leave fewer than 1024 workgroups ([768, 128]: 2.8
// against 3.4 us).  us, wave per row (aligned) or three passes (other N) -> grouped: [400000, 16] 89.1
// -> 11.7, [100000, 128] 31.0 -> 20.2, [100000, 256] 39.7 -> 36.5, [205114, 75] 249.4 -> 27.7 (four rows
// 26.1), [1000000, 17] 1069 -> 29.8, [242880, 201] 343.6 -> 71.8 (four rows 74.6).
template <int G>
static void launch_ln32_grouped(const float* x, const float* w, const float* b, float* y, float* mean, float* rstd,
                                int64_t M, int N, float eps, hipStream_t s) {
  const int64_t rows = 256 / G, two = (M + 2 * rows - 1) / (2 * rows);
  if (two >= 1024)
    layernorm_rows_f32_grouped<G, 2><<<dim3(static_cast<unsigned>(two)), dim3(256), 0, s>>>(x, w, b, y, mean, rstd, M,
                                                                                           N, eps);
  else
    layernorm_rows_f32_grouped<G, 1><<<dim3(static_cast<unsigned>((M + rows - 1) / rows)), dim3(256), 0, s>>>(
        x, w, b, y, mean, rstd, M, N, eps);
}

template <int kW, bool kU>
static void launch_ln32_multi(const float* x, const float* w, const float* b, float* y, float* mean, float* rstd,
                              int64_t M, int n4, int N, float eps, hipStream_t s) {
  layernorm_rows_f32_multi<16, kW, kU><<<dim3(static_cast<unsigned>(M)), dim3(64 * kW), 0, s>>>(x, w, b, y, mean, rstd,
                                                                                               n4, N, eps);
}

// N / 4 <= 16384 whole vectors per row.
template <bool kU>
static void launch_ln32_held(const float* x, const float* w, const float* b, float* y, float* mean, float* rstd,
                             int64_t M, int N, float eps, hipStream_t s) {
  const int n4 = N / 4, nv = (N + 3) / 4;
  if (N >= 4 && nv <= 64) {
    if (nv <= 2) launch_ln32_grouped<2>(x, w, b, y, mean, rstd, M, N, eps, s);
    else if (nv <= 4) launch_ln32_grouped<4>(x, w, b, y, mean, rstd, M, N, eps, s);
    else if (nv <= 8) launch_ln32_grouped<8>(x, w, b, y, mean, rstd, M, N, eps, s);
    else if (nv <= 16) launch_ln32_grouped<16>(x, w, b, y, mean, rstd, M, N, eps, s);
    else if (nv <= 32) launch_ln32_grouped<32>(x, w, b, y, mean, rstd, M, N, eps, s);
    else launch_ln32_grouped<64>(x, w, b, y, mean, rstd, M, N, eps, s);
    return;
  }
  if constexpr (kU) {
    if (n4 <= 64) {  // N < 4, or 257-259
      launch_ln32_wave<1, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
      return;
    }
  }
  if (n4 <= 128) launch_ln32_wave<2, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 256) launch_ln32_wave<4, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 512) launch_ln32_wave<8, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 1024) launch_ln32_wave<16, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 2048) launch_ln32_multi<2, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 4096) launch_ln32_multi<4, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else if (n4 <= 8192) launch_ln32_multi<8, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
  else launch_ln32_multi<16, kU>(x, w, b, y, mean, rstd, M, n4, N, eps, s);
}

// True when every tensor starts at a multiple of `a` bytes.
static bool ln32_aligned(const void* x, const void* w, const void* b, const void* y, uintptr_t a) {
  const auto al = [a](const void* p) { return reinterpret_cast<uintptr_t>(p) % a == 0; };
  return al(x) && al(w) && al(b) && al(y);
}

hipError_t launch_layernorm_rows_f32(const float* x, const float* w, const float* b, float* y, float* mean,
                                     float* rstd, int64_t M, int64_t N, float eps, hipStream_t s) {
  if (M == 0) return hipSuccess;
  if (M > 0x7fffffffLL) return hipErrorInvalidValue;
  // N = 0: the mean of an empty row is 0 / 0 (NaN), as numpy's sum / N; y is empty
  if (N > 0 && N / 4 <= 16384 && ln32_aligned(x, w, b, y, 4)) {
    if (N % 4 == 0 && ln32_aligned(x, w, b, y, 16))
      launch_ln32_held<false>(x, w, b, y, mean, rstd, M, static_cast<int>(N), eps, s);
    else
      launch_ln32_held<true>(x, w, b, y, mean, rstd, M, static_cast<int>(N), eps, s);
    return hipGetLastError();
  }
  layernorm_rows_f32_any<<<dim3(static_cast<unsigned>(M)), dim3(kLn32AnyThreads), 0, s>>>(x, w, b, y, mean, rstd, N,
                                                                                          eps);
  return hipGetLastError();
}

}  // namespace ihip
