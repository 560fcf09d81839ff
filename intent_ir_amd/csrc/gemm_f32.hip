// C = act(op(A) @ op(B) + bias) in float32 throughout: A [M, K] (or [K, M] with transpose_a),
// B [K, N] (or [N, K] with transpose_b), bias f32 [N] or null, C f32 [M, N], on gfx950's fp32
// matrix cores (v_mfma_f32_32x32x2_f32: exact f32 products, f32 accumulation; no reduced-
// precision inputs).  Any M, N, K and any alignment.
//
// Schedule (one MFMA instruction is 32x32x2 = 4096 flops in 16 passes, so a CU needs only
// 8 bytes of operands per clock at full rate: the kernel stages through registers and is
// built to keep the matrix pipe fed, not to save copy instructions):
//  * workgroup tile TB x TB (TB = 128, or 64 when 128-tiles would leave most CUs idle), k step
//    32; 256 threads = 4 waves in a 2x2 grid, each owning (TB/2)^2 = (TB/64)^2 blocks of 32x32;
//  * LDS double buffer, one barrier per k step; the next step's global loads are issued before
//    the current step's MFMAs so their latency hides behind ~4096 cycles of matrix work;
//  * each operand is copied into LDS in its own memory order with 16-byte accesses: a
//    K-contiguous operand (A as [M, K], B as [N, K]) as [row][k] rows of 36 floats, a
//    row-contiguous one (A as [K, M], B as [K, N]) as [k][row] rows of TB + 8 floats.  Both
//    paddings keep the MFMA operand reads free of bank conflicts;
//  * k order: within each 8-k slab, lane half h (lane / 32) feeds k = 4h + t to the t-th MFMA
//    (t < 4), so a lane's four k values are contiguous in a [row][k] tile (one 16-byte read)
//    and four rows apart in a [k][row] tile;
//  * the MFMA computes C^T (B as the first operand), so each lane ends with 4 consecutive
//    columns of one C row: 16-byte stores in the epilogue, which adds bias and applies ReLU
//    (numpy's maximum(x, 0): NaN and -0.0 pass through);
//  * tiles are ordered XCD-contiguously, then grouped 8 tile-rows at a time (L2 reuse).
// Edges: a 16-byte chunk that lies wholly inside the operand (and whose row stride allows it)
// is one vector load; any other chunk is loaded element by element with zeros outside, so
// ragged M, N, K and unaligned operands need no copies and no second kernel.
#include "common.hpp"

namespace ihip {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kF32Bk = 32;   // k per LDS tile
constexpr int kF32GroupM = 8;  // tile-rows per raster group

// LDS tile of one operand: kKMajor = [k][row] (row-contiguous operand), else [row][k].
template <int TB, bool kKMajor>
struct F32Tile {
  static constexpr int kPitch = kKMajor ? TB + 8 : kF32Bk + 4;
  static constexpr int kFloats = kKMajor ? kF32Bk * kPitch : TB * kPitch;
  static constexpr int kChunks = TB * kF32Bk / 4 / 256;  // 16-byte chunks per thread
};

// Chunk i of this thread for the tile at (row r0, k k0) of an operand with `rows` rows and K
// columns of k, stored in memory as [rows][K] (kKMajor = false) or [K][rows] (true) with
// leading dimension ld.  vec: rows of the memory layout start 16-byte aligned.
template <int TB, bool kKMajor>
__device__ __forceinline__ void f32_load_tile(const float* __restrict__ X, int64_t rows, int64_t K, int64_t ld,
                                              int64_t r0, int64_t k0, bool vec, int tid,
                                              f32x4 (&v)[F32Tile<TB, kKMajor>::kChunks]) {
#pragma unroll
  for (int i = 0; i < F32Tile<TB, kKMajor>::kChunks; ++i) {
    const int c = tid + 256 * i;
    int64_t outer, inner, outer_lim, inner_lim;
    if (kKMajor) {  // memory [K][rows]: a chunk is 4 consecutive rows at one k
      outer = k0 + c / (TB / 4);
      inner = r0 + (c % (TB / 4)) * 4;
      outer_lim = K;
      inner_lim = rows;
    } else {  // memory [rows][K]: a chunk is 4 consecutive k of one row
      outer = r0 + c / (kF32Bk / 4);
      inner = k0 + (c % (kF32Bk / 4)) * 4;
      outer_lim = rows;
      inner_lim = K;
    }
    const float* p = X + outer * ld + inner;
    if (vec && outer < outer_lim && inner + 4 <= inner_lim) {
      v[i] = *reinterpret_cast<const f32x4*>(p);
    } else {
      f32x4 t = {0.f, 0.f, 0.f, 0.f};
      if (outer < outer_lim) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (inner + e < inner_lim) t[e] = p[e];
      }
      v[i] = t;
    }
  }
}

template <int TB, bool kKMajor>
__device__ __forceinline__ void f32_store_tile(float* lds, int tid, const f32x4 (&v)[F32Tile<TB, kKMajor>::kChunks]) {
  constexpr int P = F32Tile<TB, kKMajor>::kPitch;
#pragma unroll
  for (int i = 0; i < F32Tile<TB, kKMajor>::kChunks; ++i) {
    const int c = tid + 256 * i;
    const int off = kKMajor ? (c / (TB / 4)) * P + (c % (TB / 4)) * 4 : (c / (kF32Bk / 4)) * P + (c % (kF32Bk / 4)) * 4;
    *reinterpret_cast<f32x4*>(lds + off) = v[i];
  }
}

// The four k values (4h + t, t < 4, of slab kk) of row `r` of the tile for this lane.
template <int TB, bool kKMajor>
__device__ __forceinline__ f32x4 f32_frag(const float* lds, int r, int kk, int h) {
  constexpr int P = F32Tile<TB, kKMajor>::kPitch;
  if (kKMajor) {
    const float* p = lds + (kk * 8 + 4 * h) * P + r;
    return f32x4{p[0], p[P], p[2 * P], p[3 * P]};
  }
  return *reinterpret_cast<const f32x4*>(lds + r * P + kk * 8 + 4 * h);
}

__device__ __forceinline__ float relu_keep_nan(float v) { return v < 0.0f ? 0.0f : v; }

// kSplit: workgroup (segment, tile) multiplies k in [seg * kseg, seg * kseg + kseg) only (kseg a
// multiple of kF32Bk) and writes its sums to plane seg of P (M rows of ldp floats).
template <int TB, bool kTA, bool kTB, bool kSplit>
__global__ __launch_bounds__(256) void gemm_f32_bias_relu_kernel(const float* __restrict__ A,
                                                                 const float* __restrict__ B,
                                                                 const float* __restrict__ bias, float* __restrict__ C,
                                                                 int64_t M, int64_t N, int64_t K, int relu,
                                                                 int tiles_m, int tiles_n, int flags, int64_t kseg,
                                                                 float* __restrict__ P, int64_t ldp) {
  static_assert(TB == 128 || TB == 64, "tile extents");
  using TA = F32Tile<TB, kTA>;  // A as [K, M] is row-contiguous: a [k][m] tile
  using TBt = F32Tile<TB, !kTB>;  // B as [K, N] is row-contiguous: a [k][n] tile
  constexpr int kBlk = TB / 64;
  __shared__ __attribute__((aligned(16))) float lds[2 * (TA::kFloats + TBt::kFloats)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1, h = lane >> 5;
  const bool vec_a = flags & 1, vec_b = flags & 2, vec_c = flags & 4;

  const int wg = xcd_contiguous(blockIdx.x, gridDim.x);
  const int seg = kSplit ? wg / (tiles_m * tiles_n) : 0, bid = kSplit ? wg % (tiles_m * tiles_n) : wg;
  const int per_group = kF32GroupM * tiles_n;
  const int g = bid / per_group, first_m = g * kF32GroupM;
  const int gsz = (tiles_m - first_m) < kF32GroupM ? (tiles_m - first_m) : kF32GroupM;
  const int tm = first_m + (bid % per_group) % gsz, tn = (bid % per_group) / gsz;
  const int64_t m0 = static_cast<int64_t>(tm) * TB, n0 = static_cast<int64_t>(tn) * TB;
  const int64_t lda = kTA ? M : K, ldb = kTB ? K : N;

  f32x16_t acc[kBlk][kBlk];
#pragma unroll
  for (int i = 0; i < kBlk; ++i)
#pragma unroll
    for (int j = 0; j < kBlk; ++j) acc[i][j] = f32x16_t{};

  const int64_t kb = kSplit ? seg * kseg : 0, ke = kSplit && kb + kseg < K ? kb + kseg : K;
  const int KT = static_cast<int>((ke - kb + kF32Bk - 1) / kF32Bk);
  f32x4 ra[TA::kChunks], rb[TBt::kChunks];
  if (KT > 0) {
    f32_load_tile<TB, kTA>(A, M, ke, lda, m0, kb, vec_a, tid, ra);
    f32_load_tile<TB, !kTB>(B, N, ke, ldb, n0, kb, vec_b, tid, rb);
    f32_store_tile<TB, kTA>(lds, tid, ra);
    f32_store_tile<TB, !kTB>(lds + TA::kFloats, tid, rb);
  }
  __syncthreads();

  const int ra0 = wm * (TB / 2) + (lane & 31), rb0 = wn * (TB / 2) + (lane & 31);
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < KT;
    if (more) {
      const int64_t k1 = kb + static_cast<int64_t>(kt + 1) * kF32Bk;
      f32_load_tile<TB, kTA>(A, M, ke, lda, m0, k1, vec_a, tid, ra);
      f32_load_tile<TB, !kTB>(B, N, ke, ldb, n0, k1, vec_b, tid, rb);
    }
    const float* la = lds + cur * (TA::kFloats + TBt::kFloats);
    const float* lb = la + TA::kFloats;
#pragma unroll
    for (int kk = 0; kk < kF32Bk / 8; ++kk) {
      f32x4 af[kBlk], bf[kBlk];
#pragma unroll
      for (int i = 0; i < kBlk; ++i) {
        af[i] = f32_frag<TB, kTA>(la, ra0 + i * 32, kk, h);
        bf[i] = f32_frag<TB, !kTB>(lb, rb0 + i * 32, kk, h);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ni = 0; ni < kBlk; ++ni)
#pragma unroll
          for (int mi = 0; mi < kBlk; ++mi)
            acc[ni][mi] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[ni][t], af[mi][t], acc[ni][mi], 0, 0, 0);
    }
    if (more) {
      float* nxt = lds + (cur ^ 1) * (TA::kFloats + TBt::kFloats);
      f32_store_tile<TB, kTA>(nxt, tid, ra);
      f32_store_tile<TB, !kTB>(nxt + TA::kFloats, tid, rb);
    }
    __syncthreads();
  }

  // ---- epilogue: lane holds C[m][n..n+3], m = lane & 31 (+block), n = 8*g4 + 4*h (+block)
#pragma unroll
  for (int ni = 0; ni < kBlk; ++ni) {
#pragma unroll
    for (int mi = 0; mi < kBlk; ++mi) {
      const int64_t m = m0 + wm * (TB / 2) + mi * 32 + (lane & 31);
      if (m >= M) continue;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int64_t n = n0 + wn * (TB / 2) + ni * 32 + g4 * 8 + h * 4;
        if constexpr (kSplit) {
          if (n < N)  // ldp covers n .. n + 3
            *reinterpret_cast<f32x4*>(P + (seg * M + m) * ldp + n) =
                f32x4{acc[ni][mi][g4 * 4], acc[ni][mi][g4 * 4 + 1], acc[ni][mi][g4 * 4 + 2], acc[ni][mi][g4 * 4 + 3]};
          continue;
        }
        f32x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float t = acc[ni][mi][g4 * 4 + q];
          if (bias != nullptr && n + q < N) t = t + bias[n + q];
          v[q] = relu ? relu_keep_nan(t) : t;
        }
        float* p = C + m * N + n;
        if (vec_c && n + 4 <= N) {
          *reinterpret_cast<f32x4*>(p) = v;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (n + q < N) p[q] = v[q];
        }
      }
    }
  }
}

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// C = act(sum of the S planes of P + bias), planes added in order; a thread per 4 columns of a row.
__global__ __launch_bounds__(256) void gemm_f32_reduce(const float* __restrict__ P, int S, int64_t M, int64_t N,
                                                       int64_t ldp, const float* __restrict__ bias, int relu,
                                                       float* __restrict__ C) {
  const int64_t groups = ldp / 4;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= M * groups) return;
  const int64_t m = t / groups, n = (t % groups) * 4, plane = M * ldp / 4;
  const f32x4* src = reinterpret_cast<const f32x4*>(P + m * ldp + n);
  f32x4 sum = src[0];
  int s = 1;
  for (; s + 3 < S; s += 4) {  // loads four planes ahead of the additions
    const f32x4 p1 = src[s * plane], p2 = src[(s + 1) * plane], p3 = src[(s + 2) * plane], p4 = src[(s + 3) * plane];
    sum += p1;
    sum += p2;
    sum += p3;
    sum += p4;
  }
  for (; s < S; ++s) sum += src[s * plane];
  f32x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float u = bias != nullptr && n + q < N ? sum[q] + bias[n + q] : sum[q];
    v[q] = relu ? relu_keep_nan(u) : u;
  }
  float* p = C + m * N + n;
  if (n + 4 <= N) {
    *reinterpret_cast<f32x4_any*>(p) = v;
  } else {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (n + q < N) p[q] = v[q];
  }
}

// 128x128 tiles, or 64x64 when fewer than 256 tiles of 128x128 (the CU count) would run.
int gemm_f32_tile_extent(int64_t M, int64_t N) {
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  return t128 < 256 ? 64 : 128;
}

// Segments of K (1: none) and k per segment.
struct F32Split {
  int S;
  int64_t kseg;
};

template <int TB, bool kTA, bool kTB>
static hipError_t launch_f32_tb(const float* A, const float* B, const float* bias, float* C, int64_t M, int64_t N,
                                int64_t K, int relu, int flags, const F32Split& sp, float* P, hipStream_t s) {
  const int64_t tm = (M + TB - 1) / TB, tn = (N + TB - 1) / TB, ldp = (N + 3) / 4 * 4;
  if (tm * tn * sp.S > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(tm * tn * sp.S));
  if constexpr (TB == 64) {
    if (sp.S > 1) {
      gemm_f32_bias_relu_kernel<TB, kTA, kTB, true><<<grid, dim3(256), 0, s>>>(
          A, B, bias, C, M, N, K, relu, static_cast<int>(tm), static_cast<int>(tn), flags, sp.kseg, P, ldp);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      gemm_f32_reduce<<<dim3(static_cast<unsigned>((M * (ldp / 4) + 255) / 256)), dim3(256), 0, s>>>(
          P, sp.S, M, N, ldp, bias, relu, C);
      return hipGetLastError();
    }
  }
  gemm_f32_bias_relu_kernel<TB, kTA, kTB, false><<<grid, dim3(256), 0, s>>>(
      A, B, bias, C, M, N, K, relu, static_cast<int>(tm), static_cast<int>(tn), flags, K, nullptr, ldp);
  return hipGetLastError();
}

template <int TB>
static hipError_t launch_f32_layout(const float* A, const float* B, const float* bias, float* C, int64_t M, int64_t N,
                                    int64_t K, bool ta, bool tb, int relu, int flags, const F32Split& sp, float* P,
                                    hipStream_t s) {
  if (!ta && !tb) return launch_f32_tb<TB, false, false>(A, B, bias, C, M, N, K, relu, flags, sp, P, s);
  if (!ta) return launch_f32_tb<TB, false, true>(A, B, bias, C, M, N, K, relu, flags, sp, P, s);
  if (!tb) return launch_f32_tb<TB, true, false>(A, B, bias, C, M, N, K, relu, flags, sp, P, s);
  return launch_f32_tb<TB, true, true>(A, B, bias, C, M, N, K, relu, flags, sp, P, s);
}

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The split rule: a grid of 64x64 tiles (fewer than 256 tiles of 128x128) is cut along K into the S
// segments (128 k or more, at most 32) of least estimated time, in ns: k per segment times what
// 1 to 4 workgroups that share a CU need per k, per round of 1024, plus for S > 1 the second launch
// and the partials' round trip.  Ties go to the smaller S.  A workgroup alone on a CU cannot hide
// its loads: 32-37 ns per k measured (1024^3, 1920 x 241 x 14144), two of them 50 (2048 x 1000 x 2048).
// us, unsplit -> split: 46 x 704 x 8512 220 -> 23.4 (23 segments), 1920 x 241 x 14144 354 -> 169 (17), 1984
// x 256 x 8128 218 -> 98.7 (8), 1000 x 1001 x 4096 152 -> 111 (4), 512^3 18.8 -> 10.5 (4), 32 x 4096 x 4096
// 111 -> 34.7 (8); 1024^3 33.3 -> 32.1 (2).
constexpr int64_t kF32NsPerK[5] = {0, 34, 50, 73, 95};
constexpr int64_t kF32SplitFixedNs = 4000;
constexpr int64_t kF32SplitBytesPerNs = 6000;

static int64_t f32_tiles_ns(int64_t wgs, int64_t k) {
  return (wgs / 1024 * kF32NsPerK[4] + kF32NsPerK[(wgs % 1024 + 255) / 256]) * k;
}

static F32Split f32_split_plan(int64_t M, int64_t N, int64_t K) {
  F32Split best = {1, K};
  if (M <= 0 || N <= 0 || gemm_f32_tile_extent(M, N) != 64) return best;
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64), ldp = (N + 3) / 4 * 4;
  int64_t best_ns = f32_tiles_ns(tiles, K);
  for (int64_t S = 2; S <= 32 && S * 128 <= K; ++S) {
    const int64_t kseg = ((K + S - 1) / S + 31) / 32 * 32, segs = (K + kseg - 1) / kseg;
    const int64_t ns = f32_tiles_ns(tiles * segs, kseg) + kF32SplitFixedNs + segs * M * ldp * 8 / kF32SplitBytesPerNs;
    if (ns < best_ns) best = {static_cast<int>(segs), kseg}, best_ns = ns;
  }
  return best;
}

// Workspace bytes of ihip_gemm_f32_bias_relu_ws: the planes of partial sums, 0 where K is not split.
int64_t gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  const F32Split sp = f32_split_plan(M, N, K);
  return sp.S > 1 ? sp.S * M * ((N + 3) / 4 * 4) * 4 : 0;
}

// tile: 0 = automatic (gemm_f32_tile_extent), else 64 or 128.  Unsplit results do not depend on the
// tile: every C element sums its k in the same order (8-k slabs in ascending order, each slab as
// four MFMAs in the same lane pairing).  K is split (the f32 summation order changes) only with the
// automatic tile and a workspace that holds the partials.
hipError_t launch_gemm_f32_bias_relu(const float* A, const float* B, const float* bias, float* C, int64_t M,
                                     int64_t N, int64_t K, bool ta, bool tb, int relu, int tile, void* ws,
                                     int64_t ws_bytes, hipStream_t s) {
  if (M == 0 || N == 0) return hipSuccess;
  const int64_t lda = ta ? M : K, ldb = tb ? K : N;
  const int flags = ((lda % 4 == 0 && al16(A)) ? 1 : 0) | ((ldb % 4 == 0 && al16(B)) ? 2 : 0) |
                    ((N % 4 == 0 && al16(C)) ? 4 : 0);
  const int tb_ext = tile != 0 ? tile : gemm_f32_tile_extent(M, N);
  F32Split sp = {1, K};
  if (tile == 0 && ws != nullptr && al16(ws)) {
    sp = f32_split_plan(M, N, K);
    if (sp.S * M * ((N + 3) / 4 * 4) * 4 > ws_bytes) sp = {1, K};
  }
  float* P = static_cast<float*>(ws);
  return tb_ext == 64 ? launch_f32_layout<64>(A, B, bias, C, M, N, K, ta, tb, relu, flags, sp, P, s)
                      : launch_f32_layout<128>(A, B, bias, C, M, N, K, ta, tb, relu, flags, sp, P, s);
}

}  // namespace ihip
