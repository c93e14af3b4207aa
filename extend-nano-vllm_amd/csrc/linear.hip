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
// Measured on MI355X against the library (rotating weights, us):
//   N 4096 K 4096:    M 1 9.3 / 15.3   M 16 10.7 / 15.5   M 32 11.7 / 13.6
//   N 24576 K 4096:   M 1 36.7 / 45.1  M 16 42.2 / 45.3
//   N 151936 K 4096:  M 1 200 / 250    M 16 225 / 253     M 32 280 / 264
//   N 4096 K 1024:    M 1 4.4 / 6.5    M 32 4.9 / 8.8     M 64 6.3 / 9.3
//   N 1024 K 3072:    M 1 6.4 / 9.3    M 32 7.8 / 8.0     M 64 10.8 / 10.5
//   N 6144 K 8192:    M 1 25.3 / 22.4  M 16 26.7 / 23.8
//   N 5120 K 25600:   M 1 64 / 134     M 64 106 / 157
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

// Where the lines lie (us here / library, both sides of each):
//   * K > 4096: every workgroup reads x whole, 16 rows of N 6144 K 8192 26.7 /
//     23.8, N 4096 K 12288 26.7 / 23.4; but where N is small against K the
//     library leaves most CUs idle (N 5120 K 25600, M 16: 66 / 138);
//   * M > 16: wide N loses (M 24, N 151936: 267 / 259, N 24576 48.1 / 48.5),
//     N 6144 K 4096 is level at M 32 (16.1 / 15.9);
//   * M > 32: N 6144 K 1024 7.4 / 9.4 and N 4096 K 2048 10.1 / 11.4 at M 64,
//     but N 6144 K 4096 20.2 / 17.8 and N 1024 K 2048 8.5 / 8.2.
extern "C" int nva_linear_preferred(int32_t rows, int32_t n, int32_t k) {
  if (rows < 1 || rows > 64 || k < kChunkK || k % kChunkK || n < 16 || n % 4) return 0;
  if (k >= 4 * static_cast<int64_t>(n) && k >= 16384) return 1;
  if (rows <= 16) return k <= 4096;
  if (rows <= 32) return k <= 4096 && n <= 8192;
  return k <= 2048 && n >= 4096 && n <= 8192;
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
