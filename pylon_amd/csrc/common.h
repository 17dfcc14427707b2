// Shared helpers of the gfx950 kernels: element types, wave-level reductions, and the
// error convention of the C entry points (0 = launched, non-zero = refused, with the
// reason in pylon_last_error()).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#define PYLON_WAVE 64

// Element type codes shared with the Python side.
enum PylonDtype { PYLON_F32 = 0, PYLON_BF16 = 1 };

// bfloat16 is carried as its raw 16 bits; all arithmetic is done in float.
struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float bf16_bits_to_float(uint16_t b) {
  return __uint_as_float(static_cast<uint32_t>(b) << 16);
}

// Round to nearest, ties to even; NaN stays NaN.  By the hardware's conversion: the same in integer arithmetic, with a
// branch for NaN, was ten instructions a value, 0.4 us of a residual norm's 4.7.
__device__ __forceinline__ uint16_t float_to_bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}
// Two of them in one word, `low` in its low half.
__device__ __forceinline__ uint32_t floats_to_bf16_pair(float low, float high) {
  typedef float pair_f __attribute__((ext_vector_type(2)));
  typedef __bf16 pair_b __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((pair_f{low, high}), pair_b));
}

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16_t v) { return bf16_bits_to_float(v.bits); }

template <typename T>
__device__ __forceinline__ T from_float(float v);
template <>
__device__ __forceinline__ float from_float<float>(float v) {
  return v;
}
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float v) {
  bf16_t r;
  r.bits = float_to_bf16_bits(v);
  return r;
}

// The activations of gated feed-forwards.  gelu is its tanh form, 0.5 z (1 + tanh(c (z + 0.044715 z^3)))
// with c = sqrt(2 / pi); because (1 + tanh(u)) / 2 = 1 / (1 + exp(-2u)) it costs one exponential.
#define PYLON_ACT_SILU 0
#define PYLON_ACT_GELU 1
__device__ __forceinline__ float pylon_silu(float z) { return z / (1.0f + expf(-z)); }
// For results that are about to be rounded to bfloat16: the hardware's exponential and reciprocal (about one
// part in 2^22 each).
__device__ __forceinline__ float pylon_silu_for_bf16(float z) {
  return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
__device__ __forceinline__ float pylon_gelu_tanh(float z) {
  return z / (1.0f + expf(-1.5957691216057308f * fmaf(0.044715f * z * z, z, z)));
}
__device__ __forceinline__ float pylon_gate_act(float z, int act) {
  return act == PYLON_ACT_GELU ? pylon_gelu_tanh(z) : pylon_silu(z);
}

// v of another lane of the same row of 16, by a DPP control.
template <int CTRL>
__device__ __forceinline__ float lanes_turned(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), CTRL, 0xf, 0xf, true));
}

// Over the 64 lanes of a wavefront; every lane gets the result, and the same bits: a butterfly over neighbours,
// pairs, quads, halves of a row of 16, rows, halves of the wave, on the vector unit (six trips through LDS with
// shuffles, about 130 clocks each).
template <typename OP>
__device__ __forceinline__ float wave_over(float v, OP op) {
  v = op(v, lanes_turned<0xB1>(v));   // lane ^ 1
  v = op(v, lanes_turned<0x4E>(v));   // lane ^ 2
  v = op(v, lanes_turned<0x141>(v));  // lane ^ 7, whose quad holds the same
  v = op(v, lanes_turned<0x140>(v));  // lane ^ 15, whose half of the row holds the same
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(h[0]), __uint_as_float(h[1]));
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_over(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_over(v, [](float a, float b) { return fmaxf(a, b); });
}

// The first key that a token at position pos sees, for the one integer by which the attention
// kernels are told their mask: window > 0, the last `window` keys (itself included);
// window < 0, the keys of its own chunk of -window positions, chunks counted from position 0;
// 0, every key from the request's first on.
__host__ __device__ __forceinline__ int first_visible(int pos, int window) {
  if (window > 0) return pos - window + 1 > 0 ? pos - window + 1 : 0;
  if (window < 0) return pos <= 0 ? 0 : pos / (-window) * (-window);
  return 0;
}

// Sum over a workgroup of up to 1024 threads. `scratch` holds >= 16 floats of LDS.
// Every thread gets the result; the order of additions depends only on blockDim.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = threadIdx.x / PYLON_WAVE;
  const int nwaves = (blockDim.x + PYLON_WAVE - 1) / PYLON_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int i = 0; i < nwaves; ++i) total += scratch[i];
  return total;
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = threadIdx.x / PYLON_WAVE;
  const int nwaves = (blockDim.x + PYLON_WAVE - 1) / PYLON_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int i = 1; i < nwaves; ++i) total = fmaxf(total, scratch[i]);
  return total;
}

// ---- host side -------------------------------------------------------------------

extern thread_local char pylon_error_text[512];

#define PYLON_REFUSE(...)                                              \
  do {                                                                 \
    snprintf(pylon_error_text, sizeof(pylon_error_text), __VA_ARGS__); \
    return 1;                                                          \
  } while (0)

#define PYLON_REQUIRE(cond, ...)       \
  do {                                 \
    if (!(cond)) PYLON_REFUSE(__VA_ARGS__); \
  } while (0)

// After a launch: report a launch error (bad configuration and the like) as a refusal.
#define PYLON_LAUNCHED(name)                                                          \
  do {                                                                                \
    hipError_t e_ = hipGetLastError();                                                \
    if (e_ != hipSuccess) {                                                           \
      snprintf(pylon_error_text, sizeof(pylon_error_text), "%s: launch failed: %s",   \
               name, hipGetErrorString(e_));                                          \
      return 2;                                                                       \
    }                                                                                 \
    return 0;                                                                         \
  } while (0)

// The cache policy of a buffer load whose line nobody reads again (the nt bit).  A unit has some 115 lines on their way from
// memory at any time, so a stream's rate is what one line's way allows: so marked 6.06 -> 6.90 TB/s from memory (319 MB,
// three in turn), 6.85 -> 7.54 from the memory-side cache (84 MB).  Products whose matrices all stay in that cache (256 MB) gain
// or lose by it: 60 to 200 MB of 1,024-wide ones 4 to 10 % less time, of 2,560-wide ones 2 to 10 % more (65 to 128 rows, whose
// halves read w twice, up to 15).  Lines that other workgroups read too are lost to them (prompt products 15 to 25 % slower).
#define PYLON_STREAMED 2

// Compute units of the current device (0 if there is none); asked of the runtime once per device.
extern "C" int pylon_compute_units();

static inline bool pylon_valid_dtype(int d) { return d == PYLON_F32 || d == PYLON_BF16; }
static inline size_t pylon_dtype_size(int d) { return d == PYLON_F32 ? 4 : 2; }
