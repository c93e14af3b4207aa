// Projections of few rows: out[M, N] = x[M, K] . w[N, K]^T in bf16, M <= 64
// (plain decode, the verify of a few sequences, the draft's steps), fp32
// accumulation over the whole of K, one rounding at the end.
//
// What bounds it: the weights' stream from HBM (M <= 16), then the x rows'
// way from L2 into each CU (every workgroup reads all of x).  The library's
// tiles leave CUs idle on the narrow projections, and its host call costs
// ~20 us against ~4.
//
// A workgroup of eight waves owns 16 NT weight rows; wave w takes the 64-wide
// chunks w, w + 8, ... of K, so the workgroup streams 1 KiB of each row side
// by side, three chunks in flight per wave.  Weights load straight into the
// A operand (lane l: row l % 16, 16 bytes at k 8 (l / 16)); x rows load as
// whole 128-byte lines and turn into the B operand through LDS rows of the
// wave's own (36 dwords: 16 rows of 16 bytes cover all banks).  Loaded into
// the operand directly, half lines of 16 rows, x cost more the more rows it
// has (M 32, N 4096, K 4096: 14.2 us against 11.7).  The waves' sums meet in
// LDS in wave order (deterministic).
//
// Measured on MI355X against the library (device time, rotating weights, us):
//   N 4096 K 4096:    M 1 9.3 / 15.8   M 16 10.1 / 15.8   M 32 11.9 / 13.3
//   N 24576 K 4096:   M 1 37.0 / 45.4  M 16 42.8 / 45.8
//   N 4096 K 1024:    M 1 4.0 / 6.1    M 32 4.4 / 8.4     M 64 5.9 / 8.7
//   N 1024 K 3072:    M 1 6.0 / 9.3    M 32 7.4 / 7.7
//   N 5120 K 25600:   M 1 68 / 134     M 16 87 / 138      M 64 154 / 157
#include "common.h"

namespace nva {
namespace {

constexpr int kWaves = 8;
constexpr int kChunkK = 64;
constexpr int kDepth = 3;
constexpr int kXPitch = 36;          // dwords per staged x row

template <int MT, int NT>
__global__ void __launch_bounds__(kWave * kWaves, 2)
linear_rows_kernel(const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w,
                   uint16_t* __restrict__ out, int64_t out_stride, int32_t M, int32_t N, int32_t K) {
  constexpr int kStage = MT * 16 * kXPitch;
  constexpr int kSums = NT * MT * kWave * 4;
  constexpr int kOwn = kStage > kSums ? kStage : kSums;   // dwords of LDS a wave
  __shared__ __attribute__((aligned(16))) uint32_t lds[kWaves * kOwn];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int m16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT;
  uint32_t* const stage = lds + wv * kOwn;

  // rows past the end repeat the last one; what they give is not stored
  const uint16_t* wp[NT];
  const uint16_t* xp[2 * MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = n0 + 16 * t + m16;
    wp[t] = w + static_cast<int64_t>(r < N ? r : N - 1) * K + 8 * g;
  }
#pragma unroll
  for (int t = 0; t < 2 * MT; ++t) {
    const int r = 8 * t + (lane >> 3);
    xp[t] = x + static_cast<int64_t>(r < M ? r : M - 1) * x_stride + 8 * (lane & 7);
  }
  struct Chunk {
    uint4 w[NT][2], x[2 * MT];
  };
  auto load = [&](int c, Chunk& b) {
    const int k = c * kChunkK;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) b.w[t][s] = *reinterpret_cast<const uint4*>(wp[t] + k + 32 * s);
#pragma unroll
    for (int t = 0; t < 2 * MT; ++t) b.x[t] = *reinterpret_cast<const uint4*>(xp[t] + k);
  };
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // the stage belongs to this wave: LDS runs its operations in order
  auto compute = [&](const Chunk& b) {
#pragma unroll
    for (int t = 0; t < 2 * MT; ++t)
      *reinterpret_cast<uint4*>(stage + (8 * t + (lane >> 3)) * kXPitch + 4 * (lane & 7)) = b.x[t];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const bf16x8_t xo = *reinterpret_cast<const bf16x8_t*>(stage + (16 * m + m16) * kXPitch +
                                                               16 * s + 4 * g);
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, b.w[t][s]), xo, acc[t][m], 0, 0, 0);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  const int nchunks = K / kChunkK;
  Chunk buf[kDepth];
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
    if (wv + d * kWaves < nchunks) load(wv + d * kWaves, buf[d]);
  for (int c0 = wv; c0 < nchunks; c0 += kDepth * kWaves) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      const int c = c0 + d * kWaves;
      if (c < nchunks) compute(buf[d]);
      if (c + kDepth * kWaves < nchunks) load(c + kDepth * kWaves, buf[d]);
    }
  }

  // the sums of all waves, tile by tile
  __syncthreads();
  f32x4_t* const sums = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) sums[(wv * NT * MT + t * MT + m) * kWave + lane] = acc[t][m];
  __syncthreads();
  for (int it = wv; it < NT * MT; it += kWaves) {
    f32x4_t s = sums[it * kWave + lane];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) {
      const f32x4_t a = sums[(v * NT * MT + it) * kWave + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += a[i];
    }
    // accumulator rows are weight rows: four consecutive columns of out
    const int m = 16 * (it % MT) + m16, n = n0 + 16 * (it / MT) + 4 * g;
    if (m < M && n < N)
      *reinterpret_cast<uint2*>(out + m * out_stride + n) = make_uint2(
          static_cast<uint32_t>(f32_to_bf16(s[0])) | (static_cast<uint32_t>(f32_to_bf16(s[1])) << 16),
          static_cast<uint32_t>(f32_to_bf16(s[2])) | (static_cast<uint32_t>(f32_to_bf16(s[3])) << 16));
  }
}

}  // namespace
}  // namespace nva

using namespace nva;

// Where the lines lie (device time, us here / library, rotating weights):
//   * K > 4096: every workgroup reads x whole, 16 rows of N 6144 K 8192 26.7 /
//     23.8, N 4096 K 12288 26.7 / 23.4.  Past K 16384, though, the library's
//     time jumps where N is small against K (N 512-6144, K 17408-32768: 43-190
//     us), and this kernel's does not: N 5120 K 25600, M 1 68 / 134, M 32 106 /
//     146; N 2048 K 20480, M 16 35 / 61.  At K 16384 itself the library splits
//     K and wins (N 4096, M 16 34.7 / 31.7), below N 512 too few workgroups
//     stream (N 64 K 49152, M 1 54 / 34), past K 32768 it is mixed (N 1024, M
//     24 66 / 62), and from 33 rows x costs more: N from 2048, K to 25600 (N
//     2048 K 25600, M 64 79 / 80; N 5120 K 27648, M 64 164 / 158);
//   * up to 12 rows, every N (N 16 K 64, M 1 2.1 / 4.2; N 8192 K 4096 level);
//   * more rows where the last round of workgroups is nearly empty (N between
//     4096 and 6144): M 16 K 2560 11.4 / 10.7 (N 6144 K 4096 15.7 / 14.7), M 32
//     K 3072 16.1 / 12.6, K 2048 11.1 / 12.6 still; M 64 K 64 4.1 / 3.9, K 2048
//     17.2 / 13.2;
//   * 17-32 rows: N to 4096 (K 4096, M 32 11.9 / 13.3), and to 8192 for K to
//     2048 (N 6144 K 3072, M 32 14.0 / 13.0), past N 7168, where the library's
//     time jumps, to 3072 (N 8192, M 32 14.9 / 17.9; K 4096 18.5 / 17.4);
//     wider N loses (N 9216 K 2560, M 24 20.8 / 15.3);
//   * 33-64 rows: N 4096 and N 6144-8192 for K to 2048 (N 4096, M 64 10.3 /
//     12.6; N 6144 12.6 / 13.5; K 4096 21.0 / 18.3); N 1024 K 2048 8.5 / 8.2.
extern "C" int nva_linear_preferred(int32_t rows, int32_t n, int32_t k) {
  if (rows < 1 || rows > 64 || k < kChunkK || k % kChunkK || n < 16 || n % 4) return 0;
  if (k > 4096)
    return k > 16384 && k <= 32768 && n >= 512 && n <= 6144 && k >= 4 * static_cast<int64_t>(n) &&
           (rows <= 32 || (n >= 2048 && k <= 25600));
  const bool part_round = n > 4096 && n < 6144;
  if (rows <= 12) return 1;
  if (rows <= 16) return n <= 4096 || n >= 7168 || k <= (part_round ? 2048 : 3584);
  if (rows <= 32) return n <= 4096 || (n <= 8192 && k <= (n > 7168 ? 3072 : 2048));
  return n >= 4096 && n <= 8192 && !part_round && k <= 2048;
}

extern "C" int nva_linear(const void* x, int64_t x_row_stride, const void* w, void* out,
                          int64_t out_row_stride, int32_t rows, int32_t n, int32_t k, void* stream) {
  if (rows < 0 || n <= 0 || k <= 0) return NVA_ERR_ARG;
  if (rows == 0) return NVA_OK;
  if (!x || !w || !out || x_row_stride < k || out_row_stride < n) return NVA_ERR_ARG;
  if (rows > 64 || k % kChunkK || n % 4 || x_row_stride % 8 || out_row_stride % 4 || !aligned16(x) ||
      !aligned16(w) || !aligned16(out))
    return NVA_ERR_UNSUPPORTED;
  // 32 weight rows a workgroup halve x's traffic; 16 where that would leave
  // CUs empty (N 4096 K 4096, M 16: 10.7 / 13.6 us) or where few x rows make
  // it cheap (N 24576, M 1: 36.7 / 41.8, M 8 38.8 / 41.5, M 12 42.2 / 41.5)
  const bool two = n >= 6144 && (rows > 8 || n < 12288);
  auto launch = [&](auto* kern) {
    const int per = two ? 32 : 16;
    kern<<<(n + per - 1) / per, kWave * kWaves, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const uint16_t*>(x), x_row_stride, static_cast<const uint16_t*>(w),
        static_cast<uint16_t*>(out), out_row_stride, rows, n, k);
  };
  if (rows <= 16)
    launch(two ? linear_rows_kernel<1, 2> : linear_rows_kernel<1, 1>);
  else if (rows <= 32)
    launch(two ? linear_rows_kernel<2, 2> : linear_rows_kernel<2, 1>);
  else
    launch(two ? linear_rows_kernel<4, 2> : linear_rows_kernel<4, 1>);
  return launch_status();
}
