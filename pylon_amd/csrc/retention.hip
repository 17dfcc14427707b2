// Retention: linear attention with one fixed decay per head, no softmax and no denominator.
// Per request and head a state S [dim, vdim] of floats is carried from token to token:
//
//   S_t = decay * S_{t-1} + k_t v_t^T,     o_t = S_t^T q_t,
//   out_t = o_t / sqrt(mean(o_t^2) + eps) * silu(g_t)
//
// q and k are first rotated by the token's position (the first rot_dims elements of a head,
// element i paired with i + rot_dims/2, angle = position * inv_freq[i]); k is then multiplied
// by k_scale.  Everything but the loads of the projection and the store of the result is float.
//
// This file holds the recurrent form: one workgroup per (row of the step, head) walks the
// row's tokens in order with S in registers: in retention_rows_kernel four neighbouring columns a
// thread and every IP-th row of them; in the general kernel, for the sizes which that does not take, column j
// in the threads j, j + vdim, ....  The order of every sum is fixed by the head's sizes,
// so a request's results do not depend on how it was cut into steps or what shared a step.
#include "common.h"

// FORM 1 (lightning attention): q, k and v pass through silu (rounded to the model's type) instead of being
// rotated and scaled, and o_t leaves as floats, unnormed and ungated.
template <typename T, int NI, int THREADS, int FORM>
__global__ __launch_bounds__(THREADS) void retention_recurrent_kernel(void* __restrict__ out_any, const T* __restrict__ proj, long long ld,
                                           int q_off, int k_off, int v_off, int g_off, float* state,
                                           const float* __restrict__ decay, const float* __restrict__ inv_freq,
                                           int rot_dims, const int* __restrict__ positions,
                                           const int* __restrict__ row_start, const int* __restrict__ row_slots,
                                           int heads, int dim, int vdim, int ip_count, float eps, float k_scale) {
  extern __shared__ float lds[];
  float* qs = lds;                 // [dim]
  float* ks = qs + dim;            // [dim]
  float* part = ks + dim;          // [ip_count * vdim]
  float* red = part + ip_count * vdim;  // [16]
  const int row = blockIdx.x, head = blockIdx.y;
  const int tid = threadIdx.x;
  const int j = tid % vdim, ip = tid / vdim;  // column of S, and which rows of it
  const bool owner = ip < ip_count;           // the workgroup is padded to whole wavefronts
  const int begin = row_start[row], end = row_start[row + 1];
  float* st = state + ((static_cast<size_t>(row_slots[row]) * heads + head) * dim) * vdim;
  const float lam = decay[head];
  float s[NI];
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int i = ip + n * ip_count;
    s[n] = (owner && i < dim) ? st[static_cast<size_t>(i) * vdim + j] : 0.f;
  }
  const int half = rot_dims / 2;
  for (int t = begin; t < end; ++t) {
    const T* pr = proj + static_cast<size_t>(t) * ld;
    const float pos = FORM == 0 ? static_cast<float>(positions[t]) : 0.f;
    for (int e = tid; e < 2 * dim; e += blockDim.x) {
      const bool is_k = e >= dim;
      const int d = is_k ? e - dim : e;
      const T* src = pr + (is_k ? k_off : q_off) + head * dim;
      float v = to_float(src[d]);
      if (FORM == 1) {
        v = sizeof(T) == 2 ? to_float(from_float<T>(pylon_silu_for_bf16(v))) : pylon_silu(v);
      } else if (d < rot_dims) {
        const int pair = d < half ? d : d - half;
        const float angle = pos * inv_freq[pair];
        float sn, cs;
        sincosf(angle, &sn, &cs);
        const float other = to_float(src[d < half ? d + half : d - half]);
        v = d < half ? v * cs - other * sn : v * cs + other * sn;
      }
      if (is_k) ks[d] = v * k_scale;
      else qs[d] = v;
    }
    __syncthreads();
    float vj = to_float(pr[v_off + head * vdim + j]);
    if (FORM == 1) vj = sizeof(T) == 2 ? to_float(from_float<T>(pylon_silu_for_bf16(vj))) : pylon_silu(vj);
    float acc = 0.f;
    if (owner) {
#pragma unroll
      for (int n = 0; n < NI; ++n) {
        const int i = ip + n * ip_count;
        if (i < dim) {
          s[n] = fmaf(lam, s[n], ks[i] * vj);
          acc = fmaf(s[n], qs[i], acc);
        }
      }
      part[ip * vdim + j] = acc;
    }
    __syncthreads();
    float o = 0.f, sq = 0.f;
    if (ip == 0) {
      for (int p = 0; p < ip_count; ++p) o += part[p * vdim + j];
      sq = o * o;
    }
    if (FORM == 1) {
      // (the next token's q and k are written behind the barrier above, its parts behind the next one)
      if (ip == 0) static_cast<float*>(out_any)[(static_cast<size_t>(t) * heads + head) * vdim + j] = o;
      continue;
    }
    T* out = static_cast<T*>(out_any);
    const float total = block_sum(sq, red);  // two barriers inside: qs, ks and part are free again after it
    if (ip == 0) {
      const float inv = 1.0f / sqrtf(total / static_cast<float>(vdim) + eps);
      const float g = to_float(pr[g_off + head * vdim + j]);
      out[(static_cast<size_t>(t) * heads + head) * vdim + j] = from_float<T>((o * inv) * (g / (1.0f + expf(-g))));
    }
  }
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int i = ip + n * ip_count;
    if (owner && i < dim) st[static_cast<size_t>(i) * vdim + j] = s[n];
  }
}

// A decode step brings one token a row: 64 KB of state a head go through a compute unit for a few thousand
// operations, and what bounds it is the number of loads and their chain.  So: 512 threads with 16-byte pieces
// of S, contiguous over the workgroup; the first token's elements are sent for ahead of S (loads come back
// in order: behind it they would wait for all of it) and are rotated while S is on its way; k, q and v in LDS.
// One token a row, 20 heads of 128 x 128: 4 rows 17.5 us with 64 loads of 4 bytes by 256 threads, 6.4 so; 64 rows
// 89.9 and 42.8 (168 MB through the chip: 3.9 TB/s); 2 rows of 16 heads of 256 x 256 52.3 and 13.0; 2 rows of 50
// float32 tokens 243 and 109.
#define RT_THREADS 512
template <typename T, int NI, int FORM>
__global__ __launch_bounds__(RT_THREADS) void retention_rows_kernel(
    void* __restrict__ out_any, const T* __restrict__ proj, long long ld, int q_off, int k_off, int v_off, int g_off,
    float* state, const float* __restrict__ decay, const float* __restrict__ inv_freq, int rot_dims,
    const int* __restrict__ positions, const int* __restrict__ row_start, const int* __restrict__ row_slots, int heads,
    int dim, int vdim, int ip_count, float eps, float k_scale) {
  extern __shared__ __attribute__((aligned(16))) float rows_lds[];
  float* vs = rows_lds;                 // [vdim]
  float* part = vs + vdim;              // [ip_count * vdim]
  float* ks = part + ip_count * vdim;   // [dim]
  float* qs = ks + dim;                 // [dim]
  float* red = qs + dim;                // [16]
  const int row = blockIdx.x, head = blockIdx.y;
  const int tid = threadIdx.x;
  const int quads = vdim / 4;
  const int ip = tid / quads, j = 4 * (tid - ip * quads);
  const bool owner = ip < ip_count;
  const int begin = row_start[row], end = row_start[row + 1];
  float* st = state + ((static_cast<size_t>(row_slots[row]) * heads + head) * dim) * vdim;
  const float lam = decay[head];
  const int half = rot_dims / 2;
  const int elements = 2 * dim + vdim;  // q, k and v, at most two a thread

  float raw[2], other[2], freq[2], pos = 0.f, gate = 0.f;
  auto fetch = [&](int t) {
    const T* pr = proj + static_cast<size_t>(t) * ld;
    if (FORM == 0) pos = static_cast<float>(positions[t]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = tid + u * RT_THREADS;
      raw[u] = other[u] = freq[u] = 0.f;
      if (e >= elements) continue;
      if (e >= 2 * dim) {
        raw[u] = to_float(pr[v_off + head * vdim + e - 2 * dim]);
        continue;
      }
      const int d = e >= dim ? e - dim : e;
      const T* src = pr + (e >= dim ? k_off : q_off) + head * dim;
      raw[u] = to_float(src[d]);
      if (FORM == 0 && d < rot_dims) {
        other[u] = to_float(src[d < half ? d + half : d - half]);
        freq[u] = inv_freq[d < half ? d : d - half];
      }
    }
    if (FORM == 0 && tid < vdim) gate = to_float(pr[g_off + head * vdim + tid]);
  };
  auto stage = [&]() {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = tid + u * RT_THREADS;
      if (e >= elements) continue;
      float v = raw[u];
      if (FORM == 1) v = sizeof(T) == 2 ? to_float(from_float<T>(pylon_silu_for_bf16(v))) : pylon_silu(v);
      if (e >= 2 * dim) {
        vs[e - 2 * dim] = v;
        continue;
      }
      const int d = e >= dim ? e - dim : e;
      if (FORM == 0 && d < rot_dims) {
        float sn, cs;
        sincosf(pos * freq[u], &sn, &cs);
        v = d < half ? v * cs - other[u] * sn : v * cs + other[u] * sn;
      }
      if (e >= dim) ks[d] = v * k_scale;
      else qs[d] = v;
    }
  };

  if (begin < end) fetch(begin);
  float4 s[NI];
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int i = ip + n * ip_count;
    s[n] = float4{0.f, 0.f, 0.f, 0.f};
    if (owner && i < dim) s[n] = *reinterpret_cast<const float4*>(st + static_cast<size_t>(i) * vdim + j);
  }
  for (int t = begin; t < end; ++t) {
    stage();
    const float g = gate;
    if (t + 1 < end) fetch(t + 1);
    __syncthreads();
    if (owner) {
      const float4 v = *reinterpret_cast<const float4*>(vs + j);
      float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NI; ++n) {
        const int i = ip + n * ip_count;
        if (i < dim) {
          const float k = ks[i], q = qs[i];
          s[n].x = fmaf(lam, s[n].x, k * v.x), acc.x = fmaf(s[n].x, q, acc.x);
          s[n].y = fmaf(lam, s[n].y, k * v.y), acc.y = fmaf(s[n].y, q, acc.y);
          s[n].z = fmaf(lam, s[n].z, k * v.z), acc.z = fmaf(s[n].z, q, acc.z);
          s[n].w = fmaf(lam, s[n].w, k * v.w), acc.w = fmaf(s[n].w, q, acc.w);
        }
      }
      *reinterpret_cast<float4*>(part + ip * vdim + j) = acc;
    }
    __syncthreads();
    float o = 0.f;
    if (tid < vdim)
      for (int p = 0; p < ip_count; ++p) o += part[p * vdim + tid];
    const size_t at = (static_cast<size_t>(t) * heads + head) * vdim + tid;
    if (FORM == 1) {
      // (the next token's q, k and v are written behind the barrier above, its parts behind the next one)
      if (tid < vdim) static_cast<float*>(out_any)[at] = o;
      continue;
    }
    const float total = block_sum(tid < vdim ? o * o : 0.f, red);  // two barriers inside: all of LDS is free after it
    if (tid < vdim) {
      const float inv = 1.0f / sqrtf(total / static_cast<float>(vdim) + eps);
      static_cast<T*>(out_any)[at] = from_float<T>((o * inv) * (g / (1.0f + expf(-g))));
    }
  }
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int i = ip + n * ip_count;
    if (owner && i < dim) *reinterpret_cast<float4*>(st + static_cast<size_t>(i) * vdim + j) = s[n];
  }
}

// proj: [tokens, ld] of dtype, one row per token holding q (heads * dim elements from q_off),
// k (from k_off), v (heads * vdim from v_off) and the gate g (heads * vdim from g_off).
// out: [tokens, heads * vdim] of dtype (form 1: of float; no gate, no rotation, k_scale 1).  state: float [slots, heads, dim, vdim].
// decay: float [heads]; inv_freq: float [rot_dims / 2] (null when rot_dims is 0).
// The host guarantees row_slots < slots, one position per token and row_start[rows] <= tokens.
extern "C" int pylon_retention_recurrent(void* out, const void* proj, int dtype, long long ld, int q_off, int k_off,
                                         int v_off, int g_off, float* state, const float* decay,
                                         const float* inv_freq, int rot_dims, const int* positions,
                                         const int* row_start, const int* row_slots, int rows, int heads, int dim,
                                         int vdim, float eps, float k_scale, int form, hipStream_t stream) {
  PYLON_REQUIRE(form == 0 || (form == 1 && rot_dims == 0 && k_scale == 1.0f),
                "retention: form %d, or a rotation or a scale of k in the form that has none", form);
  PYLON_REQUIRE(pylon_valid_dtype(dtype), "retention: unknown dtype");
  PYLON_REQUIRE(rows >= 0 && heads > 0 && dim > 0 && vdim > 0, "retention: bad sizes");
  PYLON_REQUIRE(vdim <= 256 && dim <= 1024, "retention: heads of up to 1024 key and 256 value elements, got %d and %d",
                dim, vdim);
  PYLON_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= dim, "retention: rot_dims %d does not fit a head of %d",
                rot_dims, dim);
  PYLON_REQUIRE(rot_dims == 0 || inv_freq != nullptr, "retention: a rotation needs its frequencies");
  if (rows == 0) return 0;
  // Heads of 16 KB of state and more whose columns come in fours (64 x 64: 6.8 us in the general kernel, 4.6
  // here; 96 x 64 12.5 and 4.9); below that a thread would have less than two pieces, and rows_ip > dim leaves
  // threads without any.
  const int rows_ip = vdim % 4 == 0 ? RT_THREADS / (vdim / 4) : 0;
  if (rows_ip > 0 && static_cast<long long>(dim) * vdim >= 4096 && rows_ip <= dim && dim <= 32 * rows_ip &&
      2 * dim + vdim <= 2 * RT_THREADS && (reinterpret_cast<uintptr_t>(state) & 15) == 0) {
    const dim3 rows_grid(rows, heads), rows_block(RT_THREADS);
    const size_t rows_bytes = sizeof(float) * (vdim + static_cast<size_t>(rows_ip) * vdim + 2 * dim + 16);
#define GO3(T, NI, FORM)                                                                                              \
  hipLaunchKernelGGL((retention_rows_kernel<T, NI, FORM>), rows_grid, rows_block, rows_bytes, stream, out,             \
                     (const T*)proj, ld, q_off, k_off, v_off, g_off, state, decay, inv_freq, rot_dims, positions,      \
                     row_start, row_slots, heads, dim, vdim, rows_ip, eps, k_scale)
#define PICK3(T)                                                        \
  do {                                                                  \
    if (dim <= 8 * rows_ip && form == 0) GO3(T, 8, 0);                  \
    else if (dim <= 8 * rows_ip) GO3(T, 8, 1);                          \
    else if (form == 0) GO3(T, 32, 0);                                  \
    else GO3(T, 32, 1);                                                 \
  } while (0)
    if (dtype == PYLON_F32) PICK3(float);
    else PICK3(bf16_t);
#undef PICK3
#undef GO3
    PYLON_LAUNCHED("retention_recurrent");
  }
  int ip_count = 256 / vdim;
  if (ip_count > dim) ip_count = dim;
  if ((dim + ip_count - 1) / ip_count > 64) {  // a large head: more threads, fewer rows of S each
    ip_count = 1024 / vdim;
    if (ip_count > dim) ip_count = dim;
  }
  const int per = (dim + ip_count - 1) / ip_count;
  PYLON_REQUIRE(per <= 64, "retention: a head of %d x %d does not fit a workgroup's registers", dim, vdim);
  dim3 grid(rows, heads), block((vdim * ip_count + PYLON_WAVE - 1) / PYLON_WAVE * PYLON_WAVE);
  const size_t lds = sizeof(float) * (2 * dim + ip_count * vdim + 16);
#define GO2(T, NI, FORM)                                                                                            \
  if (block.x <= 256)                                                                                          \
    hipLaunchKernelGGL((retention_recurrent_kernel<T, NI, 256, FORM>), grid, block, lds, stream, out, (const T*)proj, ld, \
                       q_off, k_off, v_off, g_off, state, decay, inv_freq, rot_dims, positions, row_start,      \
                       row_slots, heads, dim, vdim, ip_count, eps, k_scale);                                    \
  else                                                                                                         \
    hipLaunchKernelGGL((retention_recurrent_kernel<T, NI, 1024, FORM>), grid, block, lds, stream, out, (const T*)proj, ld, \
                     q_off, k_off, v_off, g_off, state, decay, inv_freq, rot_dims, positions, row_start,        \
                     row_slots, heads, dim, vdim, ip_count, eps, k_scale)
#define GO(T, NI)                     \
  do {                                \
    if (form == 0) { GO2(T, NI, 0); } \
    else { GO2(T, NI, 1); }           \
  } while (0)
#define PICK(T)                 \
  do {                          \
    if (per <= 4) GO(T, 4);     \
    else if (per <= 16) GO(T, 16); \
    else GO(T, 64);             \
  } while (0)
  if (dtype == PYLON_F32) PICK(float);
  else PICK(bf16_t);
#undef PICK
#undef GO
#undef GO2
  PYLON_LAUNCHED("retention_recurrent");
}
