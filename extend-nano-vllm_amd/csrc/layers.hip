// Supporting per-token kernels of the target/draft forward that sit between
// the projection GEMMs: RMSNorm (optionally fused with the residual add),
// per-head q/k RMSNorm fused with neox RoPE, and SiLU-and-mul.  They are
// memory bound and replace chains of small eager torch ops; rounding follows
// the reference's eager formulas step by step (see each kernel).
#include "common.h"

namespace nva {
namespace {

constexpr int kNormThreads = 256;
constexpr int kMaxHidden = 1 << 20;
constexpr int kRowVecs = 4;    // 16-byte vectors per thread a register-resident row may use

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < kNormThreads / kWave; ++i) s += red[i];
  __syncthreads();
  return s;
}

// RMSNorm of one row, optionally after adding a residual row:
//   s = f32(x) (+ f32(residual));  residual_out = bf16(s)
//   out = bf16( bf16(s * rsqrt(mean(s^2) + eps)) * weight )
// (nanovllm/layers/layernorm.py:70-82 and :91-107: the fp32 sum is normalised,
// rounded to bf16, then multiplied by the bf16 weight in bf16.)  ROUND
// normalises the bf16-rounded sum instead: a bf16 tensor add followed by
// RMSNorm without residual (the EAGLE3 draft layer, eagle3.py:141-146).
template <bool ADD, bool ROUND = false>
__global__ void __launch_bounds__(kNormThreads)
rms_norm_kernel(const uint16_t* __restrict__ x, int64_t x_stride,
                const uint16_t* __restrict__ residual, int64_t res_stride,
                const uint16_t* __restrict__ weight, uint16_t* __restrict__ out,
                int64_t out_stride, uint16_t* __restrict__ residual_out, int64_t res_out_stride,
                int32_t hidden, float eps, bool vec) {
  __shared__ float red[kNormThreads / kWave];
  const int64_t r = blockIdx.x;
  const uint16_t* xr = x + r * x_stride;
  const uint16_t* rr = ADD ? residual + r * res_stride : nullptr;
  uint16_t* o = out + r * out_stride;
  uint16_t* ro = ADD ? residual_out + r * res_out_stride : nullptr;
  float ss = 0.0f;
  if (vec && hidden <= 8 * kNormThreads * kRowVecs) {
    // Rows of up to 8 * kNormThreads * kRowVecs elements stay in registers:
    // every load (x, residual, weight) is issued up front and the second
    // pass normalises the values held, instead of re-reading them after the
    // reduction.  The per-thread sums run in the same order as the loop
    // below, so the result is bit-identical to it.
    float s[kRowVecs][8];
    uint4 w[kRowVecs];
#pragma unroll
    for (int i = 0; i < kRowVecs; ++i) {
      const int v = threadIdx.x + i * kNormThreads;
      if (v < hidden / 8) {
        const uint4 a = reinterpret_cast<const uint4*>(xr)[v];
        uint4 b = make_uint4(0, 0, 0, 0);
        if (ADD) b = reinterpret_cast<const uint4*>(rr)[v];
        w[i] = reinterpret_cast<const uint4*>(weight)[v];
        const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
        uint32_t so[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float lo = bf16_to_f32(aw[e] & 0xFFFFu), hi = bf16_to_f32(aw[e] >> 16);
          if (ADD) {
            lo += bf16_to_f32(bw[e] & 0xFFFFu);
            hi += bf16_to_f32(bw[e] >> 16);
            so[e] = static_cast<uint32_t>(f32_to_bf16(lo)) | (static_cast<uint32_t>(f32_to_bf16(hi)) << 16);
            if (ROUND) {
              lo = bf16_to_f32(so[e] & 0xFFFFu);
              hi = bf16_to_f32(so[e] >> 16);
            }
          }
          s[i][2 * e] = lo;
          s[i][2 * e + 1] = hi;
          ss += lo * lo + hi * hi;
        }
        if (ADD) reinterpret_cast<uint4*>(ro)[v] = make_uint4(so[0], so[1], so[2], so[3]);
      }
    }
    const float inv = rsqrtf(block_sum(ss, red) / static_cast<float>(hidden) + eps);
#pragma unroll
    for (int i = 0; i < kRowVecs; ++i) {
      const int v = threadIdx.x + i * kNormThreads;
      if (v < hidden / 8) {
        const uint32_t ww[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
        uint32_t ov[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float nl = bf16_to_f32(f32_to_bf16(s[i][2 * e] * inv)) * bf16_to_f32(ww[e] & 0xFFFFu);
          const float nh = bf16_to_f32(f32_to_bf16(s[i][2 * e + 1] * inv)) * bf16_to_f32(ww[e] >> 16);
          ov[e] = static_cast<uint32_t>(f32_to_bf16(nl)) | (static_cast<uint32_t>(f32_to_bf16(nh)) << 16);
        }
        reinterpret_cast<uint4*>(o)[v] = make_uint4(ov[0], ov[1], ov[2], ov[3]);
      }
    }
    return;
  }
  // pass 1: sum of squares of the fp32 (residual-added) row
  if (vec) {
    for (int v = threadIdx.x; v < hidden / 8; v += kNormThreads) {
      const uint4 a = reinterpret_cast<const uint4*>(xr)[v];
      uint4 b = make_uint4(0, 0, 0, 0);
      if (ADD) b = reinterpret_cast<const uint4*>(rr)[v];
      const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
      uint32_t so[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float lo = bf16_to_f32(aw[e] & 0xFFFFu), hi = bf16_to_f32(aw[e] >> 16);
        if (ADD) {
          lo += bf16_to_f32(bw[e] & 0xFFFFu);
          hi += bf16_to_f32(bw[e] >> 16);
          so[e] = static_cast<uint32_t>(f32_to_bf16(lo)) | (static_cast<uint32_t>(f32_to_bf16(hi)) << 16);
          if (ROUND) {
            lo = bf16_to_f32(so[e] & 0xFFFFu);
            hi = bf16_to_f32(so[e] >> 16);
          }
        }
        ss += lo * lo + hi * hi;
      }
      if (ADD) reinterpret_cast<uint4*>(ro)[v] = make_uint4(so[0], so[1], so[2], so[3]);
    }
  } else {
    for (int c = threadIdx.x; c < hidden; c += kNormThreads) {
      float v = bf16_to_f32(xr[c]);
      if (ADD) {
        v += bf16_to_f32(rr[c]);
        ro[c] = f32_to_bf16(v);
        if (ROUND) v = bf16_to_f32(f32_to_bf16(v));
      }
      ss += v * v;
    }
  }
  const float inv = rsqrtf(block_sum(ss, red) / static_cast<float>(hidden) + eps);
  // pass 2: recompute the fp32 row (exactly the same sums) and normalise
  if (vec) {
    for (int v = threadIdx.x; v < hidden / 8; v += kNormThreads) {
      const uint4 a = reinterpret_cast<const uint4*>(xr)[v];
      uint4 b = make_uint4(0, 0, 0, 0);
      if (ADD) b = reinterpret_cast<const uint4*>(rr)[v];
      const uint4 w = reinterpret_cast<const uint4*>(weight)[v];
      const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
      uint32_t ov[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float lo = bf16_to_f32(aw[e] & 0xFFFFu), hi = bf16_to_f32(aw[e] >> 16);
        if (ADD) {
          lo += bf16_to_f32(bw[e] & 0xFFFFu);
          hi += bf16_to_f32(bw[e] >> 16);
          if (ROUND) {
            lo = bf16_to_f32(f32_to_bf16(lo));
            hi = bf16_to_f32(f32_to_bf16(hi));
          }
        }
        const float nl = bf16_to_f32(f32_to_bf16(lo * inv)) * bf16_to_f32(ww[e] & 0xFFFFu);
        const float nh = bf16_to_f32(f32_to_bf16(hi * inv)) * bf16_to_f32(ww[e] >> 16);
        ov[e] = static_cast<uint32_t>(f32_to_bf16(nl)) | (static_cast<uint32_t>(f32_to_bf16(nh)) << 16);
      }
      reinterpret_cast<uint4*>(o)[v] = make_uint4(ov[0], ov[1], ov[2], ov[3]);
    }
  } else {
    for (int c = threadIdx.x; c < hidden; c += kNormThreads) {
      float v = bf16_to_f32(xr[c]);
      if (ADD) v += bf16_to_f32(rr[c]);
      if (ROUND) v = bf16_to_f32(f32_to_bf16(v));
      const float n = bf16_to_f32(f32_to_bf16(v * inv));
      o[c] = f32_to_bf16(n * bf16_to_f32(weight[c]));
    }
  }
}

// Per-head RMSNorm (optional) + neox rotary embedding for the q and k heads of
// a fused QKV row, and (STORE) the write of the rotated keys and of the value
// heads to the paged cache in the same launch:
//   norm:  x = bf16(bf16(x * rsqrt(mean(x^2) + eps)) * w)   (qwen3.py:87-96)
//   rope:  y1 = x1*cos - x2*sin, y2 = x2*cos + x1*sin in fp32, rounded to bf16
//          with cos/sin = cos_sin[pos][i], cos_sin[pos][64 + i]
//          (rotary_embedding.py:6-48)
// Heads [0, hq) are queries (to q_out), [hq, hq + hkv) keys (to k_out, or
// rounded to bf16 and then to the cache at the token's slot, e4m3(bf16 /
// k_scale) for FP8), [hq + hkv, hq + 2 hkv) values (copied to the cache, e4m3(
// bf16 / v_scale) for FP8); a slot that is negative or past the cache is
// skipped.  Every value written is the one store_kvcache would write.
//
// Memory bound at prefill sizes, latency bound below.  16 lanes take a head:
// lane i the elements 4 i .. 4 i + 3 and 64 + 4 i .. (the two halves the
// rotation pairs) as 8-byte loads and stores, four heads a wave.  Against a head
// a wave with 2-byte accesses, us (20 launches in a graph): 384 tokens of 48
// heads 6.6 -> 4.4, 1024 of 32 heads 10.7 -> 4.7, 16384 of 48 heads 174 (2.3
// TB/s) -> 65.6 (6.1); FP8 pages 7.5 -> 5.0, 13.5 -> 6.4, 194 -> 74.
enum class KeyTo { kTensor, kCacheBf16, kCacheFp8 };

struct SlotPages {
  int64_t blk_stride, tok_stride, head_stride;  // elements
  int32_t block_size;
  int64_t num_slots;
};

// The sum of p over the 64 element pairs of a head, in the order of a 64-lane
// butterfly (32, 16, 8, 4, 2, 1) over pairs 4 i + e: a row rotation by n takes
// the place of the exchange with lane i ^ n, since the sums so far repeat
// every 2 n lanes.
template <int N>
__device__ __forceinline__ float row_ror_add(float v) {
  const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, false);
  return v + __builtin_bit_cast(float, r);
}
__device__ __forceinline__ float head_sum(float (&p)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    p[e] = row_ror_add<1>(row_ror_add<2>(row_ror_add<4>(row_ror_add<8>(p[e]))));
  return (p[0] + p[2]) + (p[1] + p[3]);
}

template <bool VEC>
__device__ __forceinline__ void load4(const uint16_t* p, float (&v)[4]) {
  if constexpr (VEC) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    v[0] = bf16_to_f32(w.x & 0xFFFFu);
    v[1] = bf16_to_f32(w.x >> 16);
    v[2] = bf16_to_f32(w.y & 0xFFFFu);
    v[3] = bf16_to_f32(w.y >> 16);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bf16_to_f32(p[e]);
  }
}
template <bool VEC>
__device__ __forceinline__ void load4(const float* p, float (&v)[4]) {
  if constexpr (VEC) {
    const float4 w = *reinterpret_cast<const float4*>(p);
    v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p[e];
  }
}
template <bool VEC>
__device__ __forceinline__ void put4(uint16_t* p, const uint16_t (&v)[4]) {
  if constexpr (VEC) {
    store_streamed(reinterpret_cast<uint2*>(p),
                   make_uint2(v[0] | (static_cast<uint32_t>(v[1]) << 16),
                              v[2] | (static_cast<uint32_t>(v[3]) << 16)));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) store_streamed(p + e, v[e]);
  }
}
// f32_to_e4m3 of two values in the low half of the result, by gfx950's
// conversion (round to nearest even, subnormals included).  What is too large,
// where f32_to_e4m3 saturates, it makes NaN, and NaN loses its sign.  Eight of
// the software conversions in a lane cost ~1 us a launch.
__device__ __forceinline__ uint32_t e4m3_pair(float a, float b) {
  const uint32_t w = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(
      __builtin_amdgcn_fmed3f(a, -448.0f, 448.0f), __builtin_amdgcn_fmed3f(b, -448.0f, 448.0f), 0, false));
  auto pick = [](float x, uint32_t byte) {
    return x != x ? ((__float_as_uint(x) >> 24) & 0x80u) | 0x7Fu : byte;
  };
  return pick(a, w & 0xFFu) | (pick(b, (w >> 8) & 0xFFu) << 8);
}
template <bool VEC>
__device__ __forceinline__ void put4_e4m3(uint8_t* p, const uint16_t (&v)[4], float scale) {
  float x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = bf16_to_f32(v[e]) / scale;
  const uint32_t w = e4m3_pair(x[0], x[1]) | (e4m3_pair(x[2], x[3]) << 16);
  if constexpr (VEC) {
    *reinterpret_cast<uint32_t*>(p) = w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = static_cast<uint8_t>(w >> (8 * e));
  }
}

template <KeyTo TO, bool VEC>
__global__ void __launch_bounds__(kNormThreads)
qk_norm_rope_kernel(const uint16_t* __restrict__ qkv, int64_t row_stride,
                    const int64_t* __restrict__ positions, const uint16_t* __restrict__ q_w,
                    const uint16_t* __restrict__ k_w, const float* __restrict__ cos_sin,
                    int32_t max_pos, int32_t hq, int32_t hkv, float eps,
                    uint16_t* __restrict__ q_out, void* __restrict__ k_out,
                    void* __restrict__ v_cache, SlotPages pages,
                    const int32_t* __restrict__ slot_mapping,
                    const float* __restrict__ k_scale_p, const float* __restrict__ v_scale_p) {
  constexpr bool STORE = TO != KeyTo::kTensor;
  const int t = blockIdx.y;
  const int place = blockIdx.x * (kNormThreads / 16) + threadIdx.x / 16;
  const int d0 = 4 * (threadIdx.x & 15);
  // a wave's four heads are of one kind: the queries' and the keys' places are
  // padded to fours (with one kv head, keys and values in one wave took turns
  // in the FP8 conversion: 3.6 us a launch, 3.2 apart)
  const int qp = (hq + 3) & ~3, kp = (hkv + 3) & ~3;
  const int kind = place < qp ? 0 : place < qp + kp ? 1 : 2;
  const int h = place - (kind == 0 ? 0 : kind == 1 ? qp : qp + kp);
  if (h >= (kind == 0 ? hq : hkv) || (kind == 2 && !STORE)) return;
  const int head = h + (kind == 0 ? 0 : kind == 1 ? hq : hq + hkv);
  const uint16_t* src = qkv + static_cast<int64_t>(t) * row_stride + static_cast<int64_t>(head) * 128 + d0;
  int64_t dst = 0;
  if (STORE && kind > 0) {
    const int64_t slot = slot_mapping[t];
    if (slot < 0 || slot >= pages.num_slots) return;
    dst = (slot / pages.block_size) * pages.blk_stride + (slot % pages.block_size) * pages.tok_stride +
          h * pages.head_stride + d0;
  }
  // every load is issued before the first use (the position's cos/sin row
  // behind the position itself, both ahead of the norm's reduction)
  int64_t pos = positions[t];
  float x1[4], x2[4];
  load4<VEC>(src, x1);
  load4<VEC>(src + 64, x2);
  uint16_t y1[4], y2[4];
  if (STORE && kind == 2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {   // the bits as they were
      y1[e] = static_cast<uint16_t>(__float_as_uint(x1[e]) >> 16);
      y2[e] = static_cast<uint16_t>(__float_as_uint(x2[e]) >> 16);
    }
    if constexpr (TO == KeyTo::kCacheFp8) {
      const float scale = v_scale_p ? *v_scale_p : 1.0f;
      put4_e4m3<VEC>(static_cast<uint8_t*>(v_cache) + dst, y1, scale);
      put4_e4m3<VEC>(static_cast<uint8_t*>(v_cache) + dst + 64, y2, scale);
    } else {
      put4<VEC>(static_cast<uint16_t*>(v_cache) + dst, y1);
      put4<VEC>(static_cast<uint16_t*>(v_cache) + dst + 64, y2);
    }
    return;
  }
  const bool is_q = kind == 0;
  const uint16_t* w = is_q ? q_w : k_w;
  float w1[4], w2[4], c[4], s[4];
  if (w) {
    load4<VEC>(w + d0, w1);
    load4<VEC>(w + d0 + 64, w2);
  }
  pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
  load4<VEC>(cos_sin + pos * 128 + d0, c);
  load4<VEC>(cos_sin + pos * 128 + 64 + d0, s);
  if (w) {
    float p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = x1[e] * x1[e] + x2[e] * x2[e];
    const float inv = rsqrtf(head_sum(p) / 128.0f + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x1[e] = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(x1[e] * inv)) * w1[e]));
      x2[e] = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(x2[e] * inv)) * w2[e]));
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y1[e] = f32_to_bf16(x1[e] * c[e] - x2[e] * s[e]);
    y2[e] = f32_to_bf16(x2[e] * c[e] + x1[e] * s[e]);
  }
  if (is_q) {
    uint16_t* q = q_out + (static_cast<int64_t>(t) * hq + h) * 128 + d0;
    put4<VEC>(q, y1);
    put4<VEC>(q + 64, y2);
  } else if constexpr (TO == KeyTo::kTensor) {
    uint16_t* k = static_cast<uint16_t*>(k_out) + (static_cast<int64_t>(t) * hkv + h) * 128 + d0;
    put4<VEC>(k, y1);
    put4<VEC>(k + 64, y2);
  } else if constexpr (TO == KeyTo::kCacheFp8) {
    const float scale = k_scale_p ? *k_scale_p : 1.0f;
    put4_e4m3<VEC>(static_cast<uint8_t*>(k_out) + dst, y1, scale);
    put4_e4m3<VEC>(static_cast<uint8_t*>(k_out) + dst + 64, y2, scale);
  } else {
    put4<VEC>(static_cast<uint16_t*>(k_out) + dst, y1);
    put4<VEC>(static_cast<uint16_t*>(k_out) + dst + 64, y2);
  }
}

// out = bf16( bf16(silu(a)) * b ) for a row [a | b] (activation.py:11-14:
// F.silu in bf16, then a bf16 product).  The division stays IEEE: with the
// hardware reciprocal in its place silu(a)'s bf16 rounding flips next to
// rounding midpoints, and the product's second rounding then leaves the
// one-ulp bound against torch.
__device__ __forceinline__ uint16_t silu_mul_one(uint16_t a, uint16_t b) {
  const float av = bf16_to_f32(a);
  const float sv = bf16_to_f32(f32_to_bf16(av / (1.0f + __expf(-av))));
  return f32_to_bf16(sv * bf16_to_f32(b));
}

// vec: 16-byte vectors of 8 elements (rows and strides multiples of 8,
// 16-byte aligned); grid.x covers a row in kNormThreads * 8 elements
__global__ void __launch_bounds__(kNormThreads)
silu_mul_kernel(const uint16_t* __restrict__ x, int64_t x_stride, uint16_t* __restrict__ out,
                int64_t out_stride, int32_t inter, bool vec) {
  const int64_t r = blockIdx.y;
  const uint16_t* a = x + r * x_stride;
  const uint16_t* b = a + inter;
  uint16_t* o = out + r * out_stride;
  if (vec) {
    const int v = blockIdx.x * kNormThreads + threadIdx.x;
    if (v >= inter / 8) return;
    const uint4 av = reinterpret_cast<const uint4*>(a)[v];
    const uint4 bv = reinterpret_cast<const uint4*>(b)[v];
    const uint32_t aw[4] = {av.x, av.y, av.z, av.w}, bw[4] = {bv.x, bv.y, bv.z, bv.w};
    uint32_t ow[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      ow[e] = static_cast<uint32_t>(silu_mul_one(aw[e] & 0xFFFFu, bw[e] & 0xFFFFu)) |
              (static_cast<uint32_t>(silu_mul_one(aw[e] >> 16, bw[e] >> 16)) << 16);
    reinterpret_cast<uint4*>(o)[v] = make_uint4(ow[0], ow[1], ow[2], ow[3]);
    return;
  }
  for (int c = blockIdx.x * kNormThreads + threadIdx.x; c < inter; c += gridDim.x * kNormThreads)
    o[c] = silu_mul_one(a[c], b[c]);
}

}  // namespace
}  // namespace nva

using namespace nva;

extern "C" int nva_rms_norm(const void* x, int64_t x_row_stride, const void* weight, void* out,
                            int64_t out_row_stride, int32_t rows, int32_t hidden, float eps,
                            void* stream) {
  if (rows < 0 || hidden <= 0 || hidden > kMaxHidden) return NVA_ERR_ARG;
  if (rows == 0) return NVA_OK;
  if (!x || !weight || !out || x_row_stride < hidden || out_row_stride < hidden) return NVA_ERR_ARG;
  const bool vec = hidden % 8 == 0 && x_row_stride % 8 == 0 && out_row_stride % 8 == 0 &&
                   aligned16(x) && aligned16(weight) && aligned16(out);
  rms_norm_kernel<false><<<rows, kNormThreads, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(x), x_row_stride, nullptr, 0,
      static_cast<const uint16_t*>(weight), static_cast<uint16_t*>(out), out_row_stride, nullptr,
      0, hidden, eps, vec);
  return launch_status();
}

namespace {

template <bool ROUND>
int launch_add_rms_norm(const void* x, int64_t x_row_stride, const void* residual,
                        int64_t residual_row_stride, const void* weight, void* out,
                        int64_t out_row_stride, void* residual_out,
                        int64_t residual_out_row_stride, int32_t rows, int32_t hidden, float eps,
                        void* stream) {
  if (rows < 0 || hidden <= 0 || hidden > kMaxHidden) return NVA_ERR_ARG;
  if (rows == 0) return NVA_OK;
  if (!x || !residual || !weight || !out || !residual_out || x_row_stride < hidden ||
      residual_row_stride < hidden || out_row_stride < hidden || residual_out_row_stride < hidden)
    return NVA_ERR_ARG;
  // pass 2 re-reads x and residual: residual_out must not overwrite them
  if (residual_out == x || residual_out == residual) return NVA_ERR_ARG;
  const bool vec = hidden % 8 == 0 && x_row_stride % 8 == 0 && residual_row_stride % 8 == 0 &&
                   out_row_stride % 8 == 0 && residual_out_row_stride % 8 == 0 && aligned16(x) &&
                   aligned16(residual) && aligned16(weight) && aligned16(out) &&
                   aligned16(residual_out);
  rms_norm_kernel<true, ROUND><<<rows, kNormThreads, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(x), x_row_stride, static_cast<const uint16_t*>(residual),
      residual_row_stride, static_cast<const uint16_t*>(weight), static_cast<uint16_t*>(out),
      out_row_stride, static_cast<uint16_t*>(residual_out), residual_out_row_stride, hidden, eps,
      vec);
  return launch_status();
}

}  // namespace

extern "C" int nva_add_rms_norm(const void* x, int64_t x_row_stride, const void* residual,
                                int64_t residual_row_stride, const void* weight, void* out,
                                int64_t out_row_stride, void* residual_out,
                                int64_t residual_out_row_stride, int32_t rows, int32_t hidden,
                                float eps, void* stream) {
  return launch_add_rms_norm<false>(x, x_row_stride, residual, residual_row_stride, weight, out,
                                    out_row_stride, residual_out, residual_out_row_stride, rows,
                                    hidden, eps, stream);
}

extern "C" int nva_add_then_rms_norm(const void* x, int64_t x_row_stride, const void* residual,
                                     int64_t residual_row_stride, const void* weight, void* out,
                                     int64_t out_row_stride, void* sum_out,
                                     int64_t sum_out_row_stride, int32_t rows, int32_t hidden,
                                     float eps, void* stream) {
  return launch_add_rms_norm<true>(x, x_row_stride, residual, residual_row_stride, weight, out,
                                   out_row_stride, sum_out, sum_out_row_stride, rows, hidden, eps,
                                   stream);
}

namespace {

bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

// qk_norm_rope_kernel's workgroups of 16 places, each kind of head padded to
// fours (the last kind's padding needs no place)
int head_blocks(int32_t hq, int32_t hkv, int kv_kinds) {
  const int places = ((hq + 3) & ~3) + (kv_kinds - 1) * ((hkv + 3) & ~3) + hkv;
  return (places + kNormThreads / 16 - 1) / (kNormThreads / 16);
}

// the 8- and 16-byte accesses of qk_norm_rope_kernel's inputs
bool rows_aligned(const void* qkv, int64_t row_stride, const void* q_w, const void* k_w,
                  const void* cos_sin) {
  return aligned8(qkv) && row_stride % 4 == 0 && aligned8(q_w) && aligned8(k_w) && aligned16(cos_sin);
}

}  // namespace

extern "C" int nva_qk_norm_rope(const void* qkv, int64_t row_stride, const int64_t* positions,
                                const void* q_norm_weight, const void* k_norm_weight,
                                const float* cos_sin, int32_t max_position, int32_t num_tokens,
                                int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                float eps, void* q_out, void* k_out, void* stream) {
  if (head_dim != 128) return NVA_ERR_UNSUPPORTED;
  if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || max_position <= 0)
    return NVA_ERR_ARG;
  if (num_tokens == 0) return NVA_OK;
  if (!qkv || !positions || !cos_sin || !q_out || !k_out ||
      row_stride < static_cast<int64_t>(num_q_heads + num_kv_heads) * head_dim)
    return NVA_ERR_ARG;
  if ((q_norm_weight == nullptr) != (k_norm_weight == nullptr)) return NVA_ERR_ARG;
  dim3 grid(head_blocks(num_q_heads, num_kv_heads, 1), num_tokens);
  const bool vec = rows_aligned(qkv, row_stride, q_norm_weight, k_norm_weight, cos_sin) &&
                   aligned8(q_out) && aligned8(k_out);
  auto* kern = vec ? qk_norm_rope_kernel<KeyTo::kTensor, true> : qk_norm_rope_kernel<KeyTo::kTensor, false>;
  kern<<<grid, kNormThreads, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(qkv), row_stride, positions,
      static_cast<const uint16_t*>(q_norm_weight), static_cast<const uint16_t*>(k_norm_weight),
      cos_sin, max_position, num_q_heads, num_kv_heads, eps, static_cast<uint16_t*>(q_out), k_out,
      nullptr, SlotPages{}, nullptr, nullptr, nullptr);
  return launch_status();
}

extern "C" int nva_qk_norm_rope_store(
    const void* qkv, int64_t row_stride, const int64_t* positions, const void* q_norm_weight,
    const void* k_norm_weight, const float* cos_sin, int32_t max_position, int32_t num_tokens,
    int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, float eps, void* q_out,
    void* k_cache, void* v_cache, int kv_dtype, int64_t cache_block_stride,
    int64_t cache_token_stride, int64_t cache_head_stride, int32_t num_blocks, int32_t block_size,
    const int32_t* slot_mapping, const float* k_scale, const float* v_scale, void* stream) {
  if (head_dim != 128) return NVA_ERR_UNSUPPORTED;
  if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || max_position <= 0 ||
      num_blocks < 0 || block_size <= 0 || cache_block_stride < 0 || cache_token_stride < 0 ||
      cache_head_stride < 0)
    return NVA_ERR_ARG;
  if (kv_dtype != NVA_KV_BF16 && kv_dtype != NVA_KV_FP8_E4M3) return NVA_ERR_ARG;
  if (num_tokens == 0) return NVA_OK;
  if (!qkv || !positions || !cos_sin || !q_out || !k_cache || !v_cache || !slot_mapping ||
      row_stride < static_cast<int64_t>(num_q_heads + 2 * num_kv_heads) * head_dim)
    return NVA_ERR_ARG;
  if ((q_norm_weight == nullptr) != (k_norm_weight == nullptr)) return NVA_ERR_ARG;
  const SlotPages pages{cache_block_stride, cache_token_stride, cache_head_stride, block_size,
                        static_cast<int64_t>(num_blocks) * block_size};
  dim3 grid(head_blocks(num_q_heads, num_kv_heads, 2), num_tokens);
  const bool vec = rows_aligned(qkv, row_stride, q_norm_weight, k_norm_weight, cos_sin) &&
                   aligned8(q_out) && aligned8(k_cache) && aligned8(v_cache) &&
                   cache_block_stride % 4 == 0 && cache_token_stride % 4 == 0 &&
                   cache_head_stride % 4 == 0;
  auto* kern = kv_dtype == NVA_KV_BF16
                   ? (vec ? qk_norm_rope_kernel<KeyTo::kCacheBf16, true>
                          : qk_norm_rope_kernel<KeyTo::kCacheBf16, false>)
                   : (vec ? qk_norm_rope_kernel<KeyTo::kCacheFp8, true>
                          : qk_norm_rope_kernel<KeyTo::kCacheFp8, false>);
  kern<<<grid, kNormThreads, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(qkv), row_stride, positions,
      static_cast<const uint16_t*>(q_norm_weight), static_cast<const uint16_t*>(k_norm_weight),
      cos_sin, max_position, num_q_heads, num_kv_heads, eps, static_cast<uint16_t*>(q_out), k_cache,
      v_cache, pages, slot_mapping, k_scale, v_scale);
  return launch_status();
}

extern "C" int nva_silu_mul(const void* x, int64_t x_row_stride, void* out, int64_t out_row_stride,
                            int32_t rows, int32_t intermediate, void* stream) {
  if (rows < 0 || intermediate <= 0) return NVA_ERR_ARG;
  if (rows == 0) return NVA_OK;
  if (!x || !out || x_row_stride < 2 * static_cast<int64_t>(intermediate) ||
      out_row_stride < intermediate)
    return NVA_ERR_ARG;
  const bool vec = intermediate % 8 == 0 && x_row_stride % 8 == 0 && out_row_stride % 8 == 0 &&
                   aligned16(x) && aligned16(out);
  const int per_block = kNormThreads * (vec ? 8 : 4);
  dim3 grid((intermediate + per_block - 1) / per_block, rows);
  silu_mul_kernel<<<grid, kNormThreads, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(x), x_row_stride, static_cast<uint16_t*>(out), out_row_stride,
      intermediate, vec);
  return launch_status();
}
