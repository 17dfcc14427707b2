// Rows of float or bfloat16 elements through buffer descriptors, four elements a lane at a time: what lies beyond the
// row is read as zeros and written nowhere, so that no lane asks for its bounds.  Rows begin at multiples of 16
// bytes (float) or 8 (bfloat16) and are whole fours of elements.
#pragma once

#include "common.h"

typedef unsigned int row_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int row_u2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_view(const T* row, int elements) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(row), 0, elements * static_cast<int>(sizeof(T)), 0x00020000);
}

// Elements i .. i + 3.
template <typename T>
__device__ __forceinline__ float4 row_four(__amdgpu_buffer_rsrc_t row, int i) {
  if constexpr (sizeof(T) == 4) {
    const row_u4 v = __builtin_amdgcn_raw_buffer_load_b128(row, i * 4, 0, 0);
    return float4{__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
  } else {
    const row_u2 v = __builtin_amdgcn_raw_buffer_load_b64(row, i * 2, 0, 0);
    return float4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                  __uint_as_float(v.y & 0xffff0000u)};
  }
}

template <typename T>
__device__ __forceinline__ void row_store(__amdgpu_buffer_rsrc_t row, int i, const float4 v) {
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b128(
        row_u4{__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)}, row, i * 4, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b64(row_u2{floats_to_bf16_pair(v.x, v.y), floats_to_bf16_pair(v.z, v.w)}, row, i * 2,
                                          0, 0);
}

// The same of a row that begins anywhere, by a check a four instead of a descriptor.
template <typename T>
struct LooseRow {
  T* p;
  int elements;
};
typedef float loose_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned short loose_h4 __attribute__((ext_vector_type(4), aligned(2)));

template <typename T>
__device__ __forceinline__ float4 row_four(const LooseRow<T>& row, int i) {
  if (i >= row.elements) return float4{0.f, 0.f, 0.f, 0.f};
  if constexpr (sizeof(T) == 4) {
    const loose_f4 v = *reinterpret_cast<const loose_f4*>(row.p + i);
    return float4{v.x, v.y, v.z, v.w};
  } else {
    const loose_h4 v = *reinterpret_cast<const loose_h4*>(row.p + i);
    return float4{bf16_bits_to_float(v.x), bf16_bits_to_float(v.y), bf16_bits_to_float(v.z), bf16_bits_to_float(v.w)};
  }
}

template <typename T>
__device__ __forceinline__ void row_store(const LooseRow<T>& row, int i, const float4 v) {
  if (i >= row.elements) return;
  if constexpr (sizeof(T) == 4)
    *reinterpret_cast<loose_f4*>(row.p + i) = loose_f4{v.x, v.y, v.z, v.w};
  else
    *reinterpret_cast<loose_h4*>(row.p + i) =
        loose_h4{float_to_bf16_bits(v.x), float_to_bf16_bits(v.y), float_to_bf16_bits(v.z), float_to_bf16_bits(v.w)};
}

template <bool LOOSE, typename T>
__device__ __forceinline__ auto row_of(const T* row, int elements) {
  if constexpr (LOOSE)
    return LooseRow<T>{const_cast<T*>(row), elements};
  else
    return row_view(row, elements);
}

// Whether rows `apart` elements apart from here on are such rows.
template <typename T>
static inline bool row_aligned(const T* p, long long apart = 0) {
  return (reinterpret_cast<uintptr_t>(p) & (4 * sizeof(T) - 1)) == 0 && (apart & 3) == 0;
}

// The sum of squares of four elements.  (Spelled out: which product of a sum becomes the fused one is else the
// compiler's choice, kernel by kernel.)
__device__ __forceinline__ float row_squares(const float4 v) {
  return fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, v.x * v.x)));
}

// Sum over a workgroup of THREADS; `scratch` has a place a wavefront and is nobody else's.  Waits for no load or store.
template <int THREADS>
__device__ __forceinline__ float row_block_sum(float v, float* scratch) {
  v = wave_sum(v);
  if ((threadIdx.x & (PYLON_WAVE - 1)) == 0) scratch[threadIdx.x / PYLON_WAVE] = v;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < THREADS / PYLON_WAVE; ++i) total += scratch[i];
  return total;
}

// d[n] = the sum over `parts` rows, `fours` fours of elements apart, of elements 4 (threadIdx.x + n THREADS) .. + 3, in
// order; of 1, 2, 4 and 8 rows (bfloat16: 1 and 2) all loads are sent before the first sum.
template <typename TD, int NV, int THREADS, bool LOOSE = false>
__device__ __forceinline__ void row_sum_parts(float4 (&d)[NV], const TD* row, int dim, int parts, unsigned fours) {
  auto part = [&](int p, float4* e) __attribute__((always_inline)) {
    const auto view = row_of<LOOSE>(row + static_cast<size_t>(p) * fours * 4, dim);
#pragma unroll
    for (int n = 0; n < NV; ++n) e[n] = row_four<TD>(view, 4 * (threadIdx.x + n * THREADS));
  };
  auto add = [&](const float4* e) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      d[n].x += e[n].x; d[n].y += e[n].y; d[n].z += e[n].z; d[n].w += e[n].w;
    }
  };
  float4 e1[NV];
  // Registers for them.  Partial sums are float: with room for eight bfloat16 rows a residual norm of 6,148 to 8,192 elements
  // holds 169 registers, one workgroup a unit, without it 80 and three (600, 1,024 and 2,048 rows of 8,192, a bfloat16 product, 11.7,
  // 20.3 and 36.6 us -> 10.2, 18.5 and 34.2).
  constexpr bool ROOM = THREADS <= 512 && sizeof(TD) == 4;
  if (ROOM && parts == 4) {
    float4 e2[NV], e3[NV];
    part(0, d); part(1, e1); part(2, e2); part(3, e3);
    add(e1); add(e2); add(e3);
  } else if (parts == 2) {
    part(0, d); part(1, e1);
    add(e1);
  } else if (ROOM && parts == 8) {
    float4 e2[NV], e3[NV], e4[NV], e5[NV], e6[NV], e7[NV];
    part(0, d); part(1, e1); part(2, e2); part(3, e3); part(4, e4); part(5, e5); part(6, e6); part(7, e7);
    add(e1); add(e2); add(e3); add(e4); add(e5); add(e6); add(e7);
  } else {
    part(0, d);
    for (int p = 1; p < parts; ++p) {
      part(p, e1);
      add(e1);
    }
  }
}
