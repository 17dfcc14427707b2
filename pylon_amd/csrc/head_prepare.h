// One wavefront prepares one head of a token's q/k/v projection: per-head RMSNorm (if a
// weight is given) and the rotation of element i with element i + head_dim/2 (if
// frequencies are given), in float.  Head sizes are multiples of 64; a lane owns
// head_dim/64 consecutive elements and finds its rotation partner in lane + 32.
#pragma once
#include "common.h"

// src: head_dim bf16 values (4-byte aligned for EPL >= 2).  On return v[e] is element
// lane*EPL + e.
template <int EPL>
__device__ __forceinline__ void load_head_bf16(const uint16_t* __restrict__ src, int lane, float v[EPL]) {
  if (EPL == 1) {
    v[0] = __uint_as_float(static_cast<uint32_t>(src[lane]) << 16);
  } else {
#pragma unroll
    for (int e = 0; e < EPL; e += 2) {
      const uint32_t two = *reinterpret_cast<const uint32_t*>(src + lane * EPL + e);
      v[e] = __uint_as_float(two << 16);
      v[e + 1 < EPL ? e + 1 : e] = __uint_as_float(two & 0xffff0000u);
    }
  }
}

template <int EPL>
__device__ __forceinline__ void norm_rotate_head(float v[EPL], int lane, const float* __restrict__ weight,
                                                 float eps, const float* __restrict__ inv_freq, float pos) {
  constexpr int HD = EPL * 64;
  if (weight != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) ss += v[e] * v[e];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(HD) + eps);
#pragma unroll
    for (int e = 0; e < EPL; ++e) v[e] = (v[e] * inv) * weight[lane * EPL + e];
  }
  if (inv_freq != nullptr) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float other = __shfl_xor(v[e], 32, PYLON_WAVE);
      const int pair = (lane & 31) * EPL + e;  // index of the (i, i + HD/2) pair
      const float angle = pos * inv_freq[pair];
      const float c = cosf(angle), sn = sinf(angle);
      v[e] = (lane < 32) ? v[e] * c - other * sn : v[e] * c + other * sn;
    }
  }
}

// dst: head_dim bf16 values (4-byte aligned for EPL >= 2).
template <int EPL>
__device__ __forceinline__ void store_head_bf16(uint16_t* __restrict__ dst, int lane, const float v[EPL]) {
  if (EPL == 1) {
    dst[lane] = float_to_bf16_bits(v[0]);
  } else {
#pragma unroll
    for (int e = 0; e < EPL; e += 2) {
      *reinterpret_cast<uint32_t*>(dst + lane * EPL + e) = floats_to_bf16_pair(v[e], v[e + 1 < EPL ? e + 1 : e]);
    }
  }
}

// ---- the same for bfloat16 with 16-byte accesses -----------------------------------------
// head_dim/8 lanes share a head, 8 consecutive elements each, so a wavefront prepares
// 512/head_dim heads at once.  j is the lane's index within its head (lane % (HD/8)).
// Every lane of the wave must call these together (they exchange values inside a head).

__device__ __forceinline__ void load8_bf16(const uint16_t* __restrict__ src, float v[8]) {
  const uint4 raw = *reinterpret_cast<const uint4*>(src);
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(w[i] << 16);
    v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

// Eight elements of a projection's row, sent for (load) some time before they are needed (sum): bfloat16
// ones, or with PARTS the sum of n_parts float vectors (32-byte aligned), stride elements apart, added in
// order and rounded to bfloat16 once.  The first four parts are on their way together.
template <bool PARTS>
struct RawHead {
  uint4 bits;
  __device__ __forceinline__ void load(const void* src, size_t at, int, long long) {
    bits = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(src) + at);
  }
  __device__ __forceinline__ void sum(const void*, size_t, int, long long, float v[8]) const {
    const uint32_t w[4] = {bits.x, bits.y, bits.z, bits.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};
template <>
struct RawHead<true> {
  float4 lo[4], hi[4];
  __device__ __forceinline__ void load(const void* src, size_t at, int n_parts, long long stride) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float4* from = reinterpret_cast<const float4*>(static_cast<const float*>(src) + at + (p < n_parts ? p : 0) * stride);
      lo[p] = from[0], hi[p] = from[1];
    }
  }
  __device__ __forceinline__ void sum(const void* src, size_t at, int n_parts, long long stride, float v[8]) const {
    float4 a = lo[0], b = hi[0];
    auto add = [&](const float4& c, const float4& d) __attribute__((always_inline)) {
      a.x += c.x, a.y += c.y, a.z += c.z, a.w += c.w;
      b.x += d.x, b.y += d.y, b.z += d.z, b.w += d.w;
    };
    if (n_parts > 1) add(lo[1], hi[1]);
    if (n_parts > 2) add(lo[2], hi[2]);
    if (n_parts > 3) add(lo[3], hi[3]);
    for (int p = 4; p < n_parts; ++p) {
      const float4* from = reinterpret_cast<const float4*>(static_cast<const float*>(src) + at + p * stride);
      add(from[0], from[1]);
    }
    const float sums[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(static_cast<__bf16>(sums[e]));
  }
};

__device__ __forceinline__ void store8_bf16(uint16_t* __restrict__ dst, const float v[8]) {
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  bf16x8_t w;
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = static_cast<__bf16>(v[e]);  // the hardware's: to nearest, ties to even
  *reinterpret_cast<bf16x8_t*>(dst) = w;
}

// Sum over the LPH (8, 16 or 32) lanes that share a head, in every lane: neighbours, pairs, quads, halves of a row
// of 16, rows change places (the additions of a butterfly over lane ^ 1, 2, 4, 8, 16, without a trip through LDS).
template <int LPH>
__device__ __forceinline__ float head_sum(float v) {
  static_assert(LPH == 8 || LPH == 16 || LPH == 32, "head sizes 64, 128, 256");
  v += lanes_turned<0xB1>(v);
  v += lanes_turned<0x4E>(v);
  v += lanes_turned<0x141>(v);
  if constexpr (LPH >= 16) v += lanes_turned<0x140>(v);
  if constexpr (LPH >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return v;
}

// v: elements 8j .. 8j+7 of a head.  weight: those of the head's RMSNorm weight, if it is `weighted`;
// `rotated`: whether the head is (both per lane: heads in one wave may differ).  cs: the token's rotation
// table, or null for the whole wave.
template <int HD>
__device__ __forceinline__ void norm_rotate8_with(float v[8], int j, bool weighted, const float weight[8], float eps,
                                                  bool rotated, const float* __restrict__ cs) {
  constexpr int LPH = HD / 8;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
  ss = head_sum<LPH>(ss);
  if (weighted) {
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(HD) + eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (v[e] * inv) * weight[e];
  }
  if (cs != nullptr) {
    const bool low = j < LPH / 2;
    const int pair0 = 8 * (j & (LPH / 2 - 1));
    float other[8], c[8], sn[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (LPH == 16)
        other[e] = lanes_turned<0x128>(v[e]);  // eight lanes further on in the row of 16
      else
        other[e] = __shfl_xor(v[e], LPH / 2, PYLON_WAVE);
      c[e] = cs[pair0 + e], sn[e] = cs[HD / 2 + pair0 + e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float turned = low ? v[e] * c[e] - other[e] * sn[e] : v[e] * c[e] + other[e] * sn[e];
      v[e] = rotated ? turned : v[e];
    }
  }
}
