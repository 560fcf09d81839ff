// C = act(A @ op(B) + bias) in bf16 for products of few rows (the step of a decode): A [M, K], M up to
// 128, B [K, N] or [N, K], any alignment, f32 accumulation on v_mfma_f32_16x16x32_bf16, C bf16 (RNE).
//
// Such a product is bound by reading its long operand once (32 x 32000 x 4096: 262 MB of B for 8
// GFLOP), and the tiled kernels spend it on rows they do not store, on a copy of ragged operands
// and on barriers between short K slices.  Here a wave owns a 16 MF x 16 NF block of C and a
// range of K, walks it in slabs of KS k, and shares nothing until its sums are done:
//  * an operand with K contiguous (A; B as [N, K]) is read in whole KS-long pieces of rows, 16
//    bytes per lane at the row's own 2-byte boundary, and goes through the wave's own LDS to
//    become MFMA fragments (rows padded by 16 bytes: conflict-free).  Fragments loaded straight
//    from memory (64 bytes of each of 16 rows per instruction) ran at 1.7-2.9 TB/s;
//  * B as [K, N] is read 8 k-rows at a time, NF consecutive columns per lane (2 NF bytes), and the
//    8 x NF values of a lane are transposed in its registers, one v_perm per pair: lane i of a
//    group then holds 8 k of column NF i + j for the j-th MFMA, so the block's columns are dealt
//    out to the MFMAs in that order;
//  * the next slab is in flight while the wave multiplies this one: (MF + NF) KS 32 bytes per wave,
//    8 or more waves per CU, no barrier;
//  * the waves of a workgroup that share a block take consecutive ranges of K, add their sums in
//    LDS in order, and each thread rounds and stores 4 consecutive columns.  (Taking the slabs in
//    turn instead ran 32 x 32000 x 4096 10% slower: every wave then walks the same few channels.)
//    Where the blocks are at most half the CUs, segments of K go to workgroups of their own, as many
//    as keep them all in one round of 256, and their f32 sums, through a workspace, to the split-K
//    reduction: one CU takes in 16-30 GB/s whatever its waves, so a product needs all of them.
// Kernel times in us (graph replays), tiled (packed, split) kernels -> this one: B as [N, K]
// 32 x 32000 x 4096 63.2 -> 51.8 (5.1 TB/s), 16 x 4096 x 4096 13.4 -> 10.8, 16 x 1024 x 8192 13.0 ->
// 9.9, 1 x 8192 x 8192 38.0 -> 24.8; B as [K, N] 16 x 32000 x 4096 53.1 -> 49.0, 16 x 16384 x 2048 16.9
// -> 14.2, 16 x 1024 x 8192 13.2 -> 10.5; ragged: 1 x 40274 x 4311 362.5 -> 82.4, 2 x 24482 x 4991
// ([N, K]) 212.9 -> 66.2, 16 x 4097 x 4095 38.2 -> 12.6, 64 x 32001 x 1001 66.8 -> 27.4, 2 x 117 x
// 1209 16.2 -> 7.8.
// Every C element sums its k in ascending slabs of 32 as the tiled kernels do: with one wave along
// K the bits are theirs, with more the result differs by the f32 summation order only.  The split
// depends on M, N, K and B's layout, so alignment does not change a bit.
#include "common.hpp"

namespace ihip {

hipError_t launch_splitk_reduce(const float* P, int S, int64_t M, int64_t N, int64_t ldp, const float* bias, int relu,
                                uint16_t* C, hipStream_t s);

// 16-row and 16-column fragments per wave, waves along K, segments of K over workgroups.
struct DirectPlan {
  int mf, nf, wk, S;
};

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kStep = 32;  // k per MFMA

// 2 * NF bytes (NF = 4 or 8) from any 2-byte boundary into NF / 2 dwords.
template <int NF>
__device__ __forceinline__ void load_cols(const uint16_t* p, uint32_t* d) {
  if constexpr (NF == 4) {
    const u32x2 v = *reinterpret_cast<const u32x2_b2*>(p);
    d[0] = v.x;
    d[1] = v.y;
  } else {
    const u32x4 v = *reinterpret_cast<const u32x4_b2*>(p);
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q] = v[q];
  }
}

template <int MF, int NF, bool kNT>
struct Direct {
  static constexpr int KS = 64;                            // k per slab
  static constexpr int kRows = 16 * (kNT ? MF + NF : MF);  // rows staged: A's, then B's as [N, K]
  static constexpr int kPerRow = KS / 8;                   // lanes (16-byte chunks) per row of a slab
  static constexpr int kAtOnce = 64 / kPerRow;             // rows per load instruction
  static constexpr int kLoads = kRows / kAtOnce;
  static constexpr int kPitch = KS + 8;                    // halves per staged row
  static constexpr int kSums = 16 * MF * (16 * NF + 4) * 4;
  static constexpr int kLdsBytes = kRows * kPitch * 2 > kSums ? kRows * kPitch * 2 : kSums;  // per wave
  static constexpr int kSteps = KS / kStep;

  struct Slab {
    u32x4 rows[kLoads];
    uint32_t b[kNT ? 1 : kSteps][4 * NF];  // B as [K, N]: k-row r of the lane's 8 at b[step][r * NF / 2]
  };

  const uint16_t* A;
  const uint16_t* B;
  uint32_t off[kLoads];  // element offset of this lane's chunk of each row, from A (or B) at k = 0
  uint32_t boff;         // B as [K, N]: element offset of the lane's first k-row and columns at k = 0
  int64_t N;

  __device__ __forceinline__ static bool from_b(int t) { return kNT && t * kAtOnce >= 16 * MF; }

  // rows past the last one, and columns past N, read the last ones (their results are not stored)
  __device__ __forceinline__ void init(int64_t M, int64_t K, int64_t m0, int64_t n0, int lane) {
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const int r = t * kAtOnce + lane / kPerRow;
      const int64_t lim = from_b(t) ? N : M;
      int64_t row = from_b(t) ? n0 + r - 16 * MF : m0 + r;
      if (row >= lim) row = lim - 1;
      off[t] = static_cast<uint32_t>(row * K + (lane % kPerRow) * 8);
    }
    if constexpr (!kNT) {
      const int64_t n = n0 + NF * (lane & 15);
      boff = static_cast<uint32_t>(8 * (lane >> 4) * N + (n + NF <= N ? n : N - NF));
    }
  }

  // the slab at k; kTail: it may reach past K, zeros there
  template <bool kTail>
  __device__ __forceinline__ void load(Slab& s, int64_t k, int64_t K, int lane) const {
    const uint16_t* a = A + k;
    const uint16_t* b = kNT ? B + k : B + k * N;
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const uint16_t* p = (from_b(t) ? b : a) + off[t];
      if constexpr (kTail) {
        const int c = (lane % kPerRow) * 8;
        s.rows[t] = load_tail8(p - c, c, K - k);
      } else {
        s.rows[t] = *reinterpret_cast<const u32x4_b2*>(p);
      }
    }
    if constexpr (!kNT) {
      const int n = static_cast<int>(N);
#pragma unroll
      for (int st = 0; st < kSteps; ++st)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          uint32_t* d = &s.b[st][r * (NF / 2)];
          if constexpr (kTail) {  // k-rows past K: the last one is read and zeros are used
            const int64_t past = k + st * kStep + 8 * (lane >> 4) + r - (K - 1);
            load_cols<NF>(b + (static_cast<int64_t>(st * kStep + r) - (past > 0 ? past : 0)) * n + boff, d);
#pragma unroll
            for (int q = 0; q < NF / 2; ++q) d[q] = past > 0 ? 0u : d[q];
          } else {
            load_cols<NF>(b + static_cast<int64_t>(st * kStep + r) * n + boff, d);
          }
        }
    }
  }

  __device__ __forceinline__ static void stage(const Slab& s, uint16_t* lds, int lane) {
#pragma unroll
    for (int t = 0; t < kLoads; ++t)
      *reinterpret_cast<u32x4*>(lds + (t * kAtOnce + lane / kPerRow) * kPitch + (lane % kPerRow) * 8) = s.rows[t];
  }

  __device__ __forceinline__ static void multiply(const uint32_t (&b)[kNT ? 1 : kSteps][4 * NF], const uint16_t* lds,
                                                  int lane, f32x4 (&acc)[MF][NF]) {
    const uint16_t* frag = lds + (lane & 15) * kPitch + 8 * (lane >> 4);
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      bf16x8_t a[MF];
#pragma unroll
      for (int i = 0; i < MF; ++i) a[i] = *reinterpret_cast<const bf16x8_t*>(frag + 16 * i * kPitch + st * kStep);
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        bf16x8_t w;
        if constexpr (kNT) {
          w = *reinterpret_cast<const bf16x8_t*>(frag + 16 * (MF + j) * kPitch + st * kStep);
        } else {  // column j of the lane's 8 x NF values: k pairs from one half of two k-rows' dwords
          u32x4 d;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            d[q] = __builtin_amdgcn_perm(b[st][(2 * q + 1) * (NF / 2) + j / 2], b[st][2 * q * (NF / 2) + j / 2],
                                         (j & 1) ? 0x07060302u : 0x05040100u);
          w = __builtin_bit_cast(bf16x8_t, d);
        }
#pragma unroll
        for (int i = 0; i < MF; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a[i], acc[i][j], 0, 0, 0);
      }
    }
  }
};

// Workgroup: wk waves along K x (W / wk) blocks along N.  mb fastest, so that neighbouring
// workgroups of an XCD share their columns of B.
template <int MF, int NF, bool kNT, int W>
__global__ __launch_bounds__(64 * W) void gemm_bf16_direct(const uint16_t* __restrict__ A,
                                                           const uint16_t* __restrict__ B,
                                                           const float* __restrict__ bias, uint16_t* __restrict__ C,
                                                           int64_t M, int64_t N, int64_t K, int relu, int mblocks,
                                                           int nblocks, int wk, int S, float* __restrict__ P,
                                                           int64_t ldp) {
  using D = Direct<MF, NF, kNT>;
  constexpr int KS = D::KS;
  constexpr int TM = 16 * MF, TN = 16 * NF, kPitch = TN + 4;
  __shared__ __attribute__((aligned(16))) char lds_raw[W * D::kLdsBytes];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i16 = lane & 15, g = lane >> 4;
  const int wn = wave / wk, kw = wave % wk;
  const int bid = xcd_contiguous(blockIdx.x, gridDim.x);
  const int64_t m0 = static_cast<int64_t>(bid % mblocks) * TM;
  const int seg = bid / mblocks / nblocks;  // nblocks workgroups along N
  const int64_t n0 = (static_cast<int64_t>(bid / mblocks % nblocks) * (W / wk) + wn) * TN;
  uint16_t* stage = reinterpret_cast<uint16_t*>(lds_raw + wave * D::kLdsBytes);

  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int64_t slabs = (K + KS - 1) / KS, per = (slabs + wk * S - 1) / (wk * S);
  const int64_t s0 = (seg * wk + kw) * per, s1 = s0 + per < slabs ? s0 + per : slabs;
  if (n0 < N && s0 < s1) {
    D d;
    d.A = A;
    d.B = B;
    d.N = N;
    d.init(M, K, m0, n0, lane);
    const int64_t whole = K / KS;  // slabs before it are wholly inside K
    const auto load = [&](typename D::Slab& slab, int64_t i) {
      if (i < whole)
        d.template load<false>(slab, i * KS, K, lane);
      else
        d.template load<true>(slab, i * KS, K, lane);
    };
    typename D::Slab slab;
    load(slab, s0);
    for (int64_t i = s0; i < s1; ++i) {
      D::stage(slab, stage, lane);
      __builtin_amdgcn_wave_barrier();  // rows staged by other lanes; a wave's LDS accesses stay in order
      if constexpr (kNT) {
        if (i + 1 < s1) load(slab, i + 1);
      }
      D::multiply(slab.b, stage, lane, acc);
      __builtin_amdgcn_wave_barrier();  // before the next slab, or the sums, take their place
      if constexpr (!kNT) {
        if (i + 1 < s1) load(slab, i + 1);
      }
    }
  }

  // acc[i][j] of this lane: row m = 16 i + i16; rows 4 g + q of the MFMA are the block's columns
  // 16 j + 4 g + q (B as [N, K]) or NF (4 g + q) + j, the last lanes' moved back inside N.
  float* mine = reinterpret_cast<float*>(stage);
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      if constexpr (kNT) {
        *reinterpret_cast<f32x4*>(mine + (16 * i + i16) * kPitch + 16 * j + 4 * g) = acc[i][j];
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t n = n0 + NF * (4 * g + q);
          const int64_t c = (n + NF <= N ? n : N - NF) + j - n0;
          if (n < N && c >= 0) mine[(16 * i + i16) * kPitch + c] = acc[i][j][q];
        }
      }
    }
  __syncthreads();
  const float floor_v = relu ? 0.0f : -__builtin_inff();
  const char* block = lds_raw + wn * wk * D::kLdsBytes;
  for (int t = kw * 64 + lane; t < TM * TN / 4; t += wk * 64) {
    const int r = t / (TN / 4), c = (t % (TN / 4)) * 4;
    const int64_t m = m0 + r, n = n0 + c;
    if (m >= M || n >= N) continue;
    const char* p = block + (r * kPitch + c) * 4;
    f32x4 sum = *reinterpret_cast<const f32x4*>(p);
    for (int w = 1; w < wk; ++w) sum += *reinterpret_cast<const f32x4*>(p + w * D::kLdsBytes);
    if (S > 1) {  // this segment's sums: gemm_splitk_reduce adds the segments (ldp covers n .. n + 3)
      *reinterpret_cast<f32x4*>(P + (seg * M + m) * ldp + n) = sum;
      continue;
    }
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = __builtin_elementwise_maximum(sum[q] + (bias != nullptr && n + q < N ? bias[n + q] : 0.0f), floor_v);
    const u32x2 pk = {pack_bf16x2_rne(v[0], v[1]), pack_bf16x2_rne(v[2], v[3])};
    uint16_t* dst = C + m * N + n;
    if (n + 4 <= N) {
      *reinterpret_cast<u32x2_b2*>(dst) = pk;
    } else {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        if (n + q < N) dst[q] = static_cast<uint16_t>(pk[q >> 1] >> (16 * (q & 1)));
    }
  }
}

template <int MF, int NF, bool kNT, int W>
hipError_t launch(const uint16_t* A, const uint16_t* B, const float* bias, uint16_t* C, int64_t M, int64_t N, int64_t K,
                  int relu, const DirectPlan& p, float* P, int64_t ldp, hipStream_t s) {
  const int64_t mblocks = (M + 16 * MF - 1) / (16 * MF), groups = W / p.wk;
  const int64_t nblocks = ((N + 16 * NF - 1) / (16 * NF) + groups - 1) / groups, grid = mblocks * nblocks * p.S;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  gemm_bf16_direct<MF, NF, kNT, W><<<dim3(static_cast<unsigned>(grid)), dim3(64 * W), 0, s>>>(
      A, B, bias, C, M, N, K, relu, static_cast<int>(mblocks), static_cast<int>(nblocks), p.wk, p.S, P, ldp);
  return hipGetLastError();
}

template <int MF, bool kNT>
hipError_t launch_nf(const uint16_t* A, const uint16_t* B, const float* bias, uint16_t* C, int64_t M, int64_t N,
                     int64_t K, int relu, const DirectPlan& p, float* P, int64_t ldp, hipStream_t s) {
  if constexpr (kNT) {
    if (p.nf == 2) return p.wk == 8 ? launch<MF, 2, kNT, 8>(A, B, bias, C, M, N, K, relu, p, P, ldp, s)
                                    : launch<MF, 2, kNT, 4>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
  } else if constexpr (MF <= 2) {
    if (p.nf == 8) return p.wk == 8 ? launch<MF, 8, kNT, 8>(A, B, bias, C, M, N, K, relu, p, P, ldp, s)
                                    : launch<MF, 8, kNT, 4>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
  }
  return p.wk == 8 ? launch<MF, 4, kNT, 8>(A, B, bias, C, M, N, K, relu, p, P, ldp, s)
                   : launch<MF, 4, kNT, 4>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
}

template <bool kNT>
hipError_t launch_mf(const uint16_t* A, const uint16_t* B, const float* bias, uint16_t* C, int64_t M, int64_t N,
                     int64_t K, int relu, const DirectPlan& p, float* P, int64_t ldp, hipStream_t s) {
  switch (p.mf) {
    case 1: return launch_nf<1, kNT>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
    case 2: return launch_nf<2, kNT>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
    default: return launch_nf<4, kNT>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
  }
}

}  // namespace

// Waves along K and segments of a product whose blocks are 64 columns wide: waves until 2048 run
// (8 per CU) or each has two slabs; then, where the launch and the round trip of a reduction (3-4
// us) are less than what idle CUs cost, as many segments as 256 workgroups allow.  (Rounded up they
// made 257 to 300, a second round for a few: 3 x 3200 x 12736 23.9 us, now 17.9; 16 x 1856 x 14024
// ([N, K]) 25.7, now 16.5.)  B as [N, K] with more than 64 blocks runs 32-column blocks on every CU
// instead (1 x 8192 x 8192: 26.5 us, in two segments 30.0); columns of B as [K, N] that narrow would
// be read half a line at a time (40.3 against 32.7).
DirectPlan gemm_direct_plan(int64_t M, int64_t N, int64_t K, bool transpose_b) {
  DirectPlan p;
  p.mf = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int64_t blocks = (M + 16 * p.mf - 1) / (16 * p.mf) * ((N + 63) / 64);
  p.wk = 1;
  while (p.wk < 8 && blocks * p.wk < 2048 && K >= 256 * p.wk) p.wk *= 2;
  p.S = 1;
  if (blocks <= (transpose_b ? 64 : 128) && K >= 2048) {
    const int64_t fill = 256 / blocks, most = K / 512;
    p.S = static_cast<int>(fill < most ? (fill < 16 ? fill : 16) : (most < 16 ? most : 16));
  }
  p.nf = 4;
  return p;
}

// Where this kernel is taken: K above two slabs, 16 to 65536 columns, A and B below 2^31 elements
// (offsets are 32 bits), and the side of the lines below on which it was the faster one.  The lines
// come from 5900 shapes drawn over M <= 128, N <= 65536, K <= 20000 in both layouts and 700 of round
// sizes, each timed here and on the kernels that run otherwise (tiled, packed or split) by graph
// replays of both on the same buffers.  The 4500 drawn ones that are taken ran 1.69x faster (geometric
// mean), nine of them slower by more than 3% (aligned ones by at most 8%); the others would have run
// 1.15x slower here.  What the lines follow:
//  * blocks of 64 columns (with the rows' blocks) against the 256 CUs: up to 256 run in one round (of
//    half as wide ones, two); the second round of 257 to 512 is partly empty and pays for few rows or
//    long K only;
//  * K: a wave needs some slabs to hide its latency, the more the more rows it multiplies (B as [K, N],
//    17 x 13888 x 136 9.0 against 5.3 us, 28 x 912 x 176 9.4 against 5.5);
//  * operands off 16-byte alignment by their length, which the other kernels copy first: up to 128 rows.
bool gemm_direct_takes(int64_t M, int64_t N, int64_t K, bool transpose_a, bool transpose_b) {
  if (transpose_a || M < 1 || N < 16 || N > 65536 || K <= 128) return false;
  if (N * K >= (int64_t(1) << 31) || M * K >= (int64_t(1) << 31)) return false;
  const bool ragged = K % 8 != 0 || (!transpose_b && N % 8 != 0);
  if (M > (ragged ? 128 : transpose_b ? 64 : 32) || (!ragged && N > 49152)) return false;
  const DirectPlan p = gemm_direct_plan(M, N, K, transpose_b);
  const int64_t b = (M + 16 * p.mf - 1) / (16 * p.mf) * ((N + 63) / 64), w = b * p.S;
  if (ragged && transpose_b) {
    if (M <= 32) return true;
    if (M <= 64) return K < 4096 || b <= 128 || b > 192;
    if (K < 256) return b <= 256;
    return K < 4096 || b <= 64 || b > 256 || (K < 8192 && (b <= 128 || b > 192));
  }
  if (ragged) {
    if (M <= 16) return true;
    if (M <= 32) return K >= 256 || b > 192;
    if (M <= 64) return K >= 384 || b > 512 || (K >= 256 && b > 64);
    return K >= 768 || (K >= 512 && b <= 256);
  }
  if (b > 512) return transpose_b ? M <= 32 || K >= 768 : M <= 16 || K < 2048;
  // rows of B as [N, K] a multiple of 1 KiB apart, which the tiled kernels read more slowly
  const bool pitch = transpose_b && K % 512 == 0;
  if (b > 256) {
    if (pitch && K >= 3072) return M <= 32 || (K >= 4096 && b > 352);
    if (M > 32) return false;
    if (M > 16) return K >= 4096 && b > (transpose_b ? 320 : 448);
    if (K < (transpose_b ? 256 : 512) || (K >= 1024 && K < 2048)) return false;
    return K < 1024 || (b > 320 && (K >= 4096 || !transpose_b));
  }
  if (pitch && M > 32) return K >= 512 && K <= 4096 && (b <= 128 || b > 192);
  if (pitch && M > 16) return K >= 512 && (K < 8192 || b <= 128 || b > 170);
  if (M <= 16) {
    if (!transpose_b && (K < 256 || (K >= 4096 && b > 64 && b <= 85))) return false;
    // workgroups launched, in rounds of 256: long K asks for rounds at least 5/8 full
    const int64_t u = transpose_b && w < 256 ? 2 * w : w, rounds = (u + 255) / 256;
    return K < 8192 || b <= 64 || u * 8 >= rounds * 256 * 5;
  }
  if (M <= 32) {
    if (!transpose_b) return K >= 512 && K <= 4096;
    return K >= 256 && (K < 2048 || b <= 64 || (b <= 128 && K < 8192) || (b > 192 && K < 4096));
  }
  return K >= 384 && (w < 64 || b <= 8 || (w <= 128 && K < 2560) || K < 1024);
}

int gemm_direct_segments(int64_t M, int64_t N, int64_t K, bool transpose_b) {
  return gemm_direct_plan(M, N, K, transpose_b).S;
}

int64_t gemm_direct_ldp(int64_t N) { return (N + 3) / 4 * 4; }

hipError_t launch_gemm_direct(const uint16_t* A, const uint16_t* B, const float* bias, uint16_t* C, int64_t M,
                              int64_t N, int64_t K, bool transpose_b, int relu, void* ws, int64_t ws_bytes,
                              hipStream_t s) {
  DirectPlan p = gemm_direct_plan(M, N, K, transpose_b);
  const int64_t ldp = gemm_direct_ldp(N);
  if (p.S > 1 && (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 15) != 0 || ws_bytes < p.S * M * ldp * 4))
    p.S = 1;
  // block widths (they do not change a sum): 32 columns where 64 leave CUs idle and B's rows are
  // whole either way, 128 where enough blocks remain and K is long (32000 x 4096: 59.3 -> 50.8 us)
  const int64_t wgs = (M + 16 * p.mf - 1) / (16 * p.mf) * ((N + 63) / 64) * p.S;
  if (transpose_b && wgs < 256) p.nf = 2;
  if (!transpose_b && p.mf <= 2 && wgs >= 400 && K >= 2048) p.nf = 8;
  float* P = static_cast<float*>(ws);
  const hipError_t e = transpose_b ? launch_mf<true>(A, B, bias, C, M, N, K, relu, p, P, ldp, s)
                                   : launch_mf<false>(A, B, bias, C, M, N, K, relu, p, P, ldp, s);
  if (e != hipSuccess || p.S == 1) return e;
  return launch_splitk_reduce(P, p.S, M, N, ldp, bias, relu, C, s);
}

}  // namespace ihip
