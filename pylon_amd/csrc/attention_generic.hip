// Paged causal grouped-query attention, the exact and general form: any element type,
// any head size up to 1024, values up to 512 (multiples of 8 with 16-byte loads), any number of heads and groups,
// any page size, optional sliding window or chunks (first_visible in common.h).  One wavefront owns one (token, query head):
// it walks that token's visible keys 64 at a time (one key per lane), keeps a running
// maximum and sum in float, and accumulates the weighted values with one lane per
// output element.  The walk starts at the first visible key of the token, so the order
// of every sum depends only on the token's position and never on how the batch was cut.
// Options: values of another size than keys; q rows that lie q_stride elements apart (a slice
// of a fused projection); a learned bias by distance added to the scaled score,
// rel[bucket[min(i - j, bucket_len - 1)] * n_heads + head], or without a table of buckets a bias
// that grows with the logarithm of the distance and is taken off, rel[head] * log(1 + rel[n_heads +
// head] * (i - j)); and a sink, a key of score 0 without a value, which adds one to the softmax's
// denominator, or with sink_logit a learned score per head in its place (exp(sink_logit[head]) is
// added; it is neither scaled nor capped).  softcap > 0: the scaled score s becomes softcap *
// tanh(s / softcap) before anything is added to it.
#include "common.h"

#define ATT_WAVES 4
#define ATT_BATCH 8

template <typename T>
struct Vec8;  // eight consecutive elements, loaded as wide as the type allows

template <>
struct Vec8<float> {
  static __device__ __forceinline__ float dot(const float* __restrict__ q, const float* __restrict__ k, float acc) {
    const float4 a = *reinterpret_cast<const float4*>(k);
    const float4 b = *reinterpret_cast<const float4*>(k + 4);
    acc = fmaf(q[0], a.x, acc);
    acc = fmaf(q[1], a.y, acc);
    acc = fmaf(q[2], a.z, acc);
    acc = fmaf(q[3], a.w, acc);
    acc = fmaf(q[4], b.x, acc);
    acc = fmaf(q[5], b.y, acc);
    acc = fmaf(q[6], b.z, acc);
    acc = fmaf(q[7], b.w, acc);
    return acc;
  }
};

template <>
struct Vec8<bf16_t> {
  static __device__ __forceinline__ float dot(const float* __restrict__ q, const bf16_t* __restrict__ k, float acc) {
    const uint4 raw = *reinterpret_cast<const uint4*>(k);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc = fmaf(q[2 * i], __uint_as_float(w[i] << 16), acc);
      acc = fmaf(q[2 * i + 1], __uint_as_float(w[i] & 0xffff0000u), acc);
    }
    return acc;
  }
};

// Over the 64 lanes of a wavefront.  One instance (bfloat16 values of 129 to 256 elements) has no register left for the
// vector unit's way and spills eight in every block of keys: 600 tokens of 16 heads of 256 745 us, through LDS 697.
template <typename T, int DIMS_PER_LANE, typename OP>
__device__ __forceinline__ float att_over(float v, OP op) {
  if constexpr (sizeof(T) == 2 && DIMS_PER_LANE == 4) {
#pragma unroll
    for (int off = PYLON_WAVE / 2; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, PYLON_WAVE));
    return v;
  } else {
    return wave_over(v, op);
  }
}

// What a score becomes before the softmax: scaled, capped, with the bias by distance.
__device__ __forceinline__ float att_score(float dot, float scale, float softcap, const float* __restrict__ rel,
                                           const int* __restrict__ bucket, int bucket_len, int n_heads, int h, int far) {
  float s = dot * scale;
  if (softcap > 0.f) s = softcap * tanhf(s / softcap);
  if (rel != nullptr) {
    if (bucket != nullptr)
      s += rel[static_cast<size_t>(bucket[far < bucket_len ? far : bucket_len - 1]) * n_heads + h];
    else
      s -= rel[h] * logf(1.0f + rel[n_heads + h] * static_cast<float>(far));
  }
  return s;
}

template <typename T, int DIMS_PER_LANE>
__global__ void paged_attention_kernel(T* __restrict__ out, const T* __restrict__ q,
                                       const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                                       const int* __restrict__ block_table, int table_width,
                                       const int* __restrict__ tok_row, const int* __restrict__ positions,
                                       long long items, int n_heads, int n_kv_heads, int head_dim,
                                       int page_size, int window, float scale, int v_dim, long long q_stride,
                                       const float* __restrict__ rel, const int* __restrict__ bucket,
                                       int bucket_len, int sink, int v_transposed, float softcap,
                                       const float* __restrict__ sink_logit, int v_row) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = threadIdx.x / PYLON_WAVE;
  float* qbuf = lds + wave * head_dim;
  const long long item = static_cast<long long>(blockIdx.x) * ATT_WAVES + wave;
  const bool active = item < items;
  int t = 0, h = 0;
  if (active) {
    t = static_cast<int>(item / n_heads);
    h = static_cast<int>(item - static_cast<long long>(t) * n_heads);
    const T* qr = q + static_cast<size_t>(t) * q_stride + static_cast<size_t>(h) * head_dim;
    for (int i = lane; i < head_dim; i += PYLON_WAVE) qbuf[i] = to_float(qr[i]);
  }
  __syncthreads();
  if (!active) return;

  const int kvh = h / (n_heads / n_kv_heads);
  const int pos = positions[t];
  const int* table = block_table + static_cast<size_t>(tok_row[t]) * table_width;
  const int first = first_visible(pos, window);

  float m = -INFINITY, l = 0.f;
  float acc[DIMS_PER_LANE];
#pragma unroll
  for (int i = 0; i < DIMS_PER_LANE; ++i) acc[i] = 0.f;

  for (int base = first; base <= pos; base += PYLON_WAVE) {
    const int j = base + lane;
    const bool valid = j <= pos;
    int phys = 0;
    float s = -INFINITY;
    if (valid) {
      phys = table[j / page_size] * page_size + (j % page_size);
      const T* kr = k_cache + (static_cast<size_t>(phys) * n_kv_heads + kvh) * head_dim;
      float dot = 0.f;
      if (head_dim & 7) {  // a head that is no whole number of 16-byte pieces: element by element
        for (int d = 0; d < head_dim; ++d) dot = fmaf(qbuf[d], to_float(kr[d]), dot);
      } else {
        // (loads of 64 elements of the key go out together: with the loop rolled a lane waited for memory
        // at every eight)
#pragma unroll 8
        for (int d = 0; d < head_dim; d += 8) dot = Vec8<T>::dot(qbuf + d, kr + d, dot);
      }
      s = att_score(dot, scale, softcap, rel, bucket, bucket_len, n_heads, h, pos - j);
    }
    const float m_new = fmaxf(m, att_over<T, DIMS_PER_LANE>(s, [](float a, float b) { return fmaxf(a, b); }));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);
    l = l * corr + att_over<T, DIMS_PER_LANE>(p, [](float a, float b) { return a + b; });
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) acc[i] *= corr;
    const int count = (pos - base + 1 < PYLON_WAVE) ? pos - base + 1 : PYLON_WAVE;
    // values transposed inside their page: [page, kv head, element, slot in page]
    const size_t vstep = v_transposed ? page_size : 1;
    // Eight keys' values are sent for before the first is used (a wave otherwise waits out a trip to
    // memory per key: float32, 32 heads of 128, steps of 3 and 270 tokens of about 110 keys together 107 -> 36
    // us a launch); the sums keep their order.
    for (int k0 = 0; k0 < count; k0 += ATT_BATCH) {
      float pk[ATT_BATCH], vv[ATT_BATCH][DIMS_PER_LANE];
#pragma unroll
      for (int u = 0; u < ATT_BATCH; ++u) {
        const int kk = k0 + u < count ? k0 + u : count - 1;
        pk[u] = __shfl(p, kk, PYLON_WAVE);
        const int physk = __shfl(phys, kk, PYLON_WAVE);
        const T* vr = v_transposed
                          ? v_cache + (static_cast<size_t>(physk / page_size) * n_kv_heads + kvh) * v_dim * page_size +
                                physk % page_size
                          : v_cache + (static_cast<size_t>(physk) * n_kv_heads + kvh) * v_row;
#pragma unroll
        for (int i = 0; i < DIMS_PER_LANE; ++i) {
          const int d = lane + PYLON_WAVE * i;
          vv[u][i] = d < v_dim ? to_float(vr[d * vstep]) : 0.f;
        }
      }
#pragma unroll
      for (int u = 0; u < ATT_BATCH; ++u)
        if (k0 + u < count)
#pragma unroll
          for (int i = 0; i < DIMS_PER_LANE; ++i) acc[i] = fmaf(pk[u], vv[u][i], acc[i]);
    }
    m = m_new;
  }
  T* orow = out + (static_cast<size_t>(t) * n_heads + h) * v_dim;
  if (sink_logit != nullptr) {
    // the sink joins as one more score: the larger of it and the maximum so far is the new scale
    const float z = sink_logit[h];
    const float m_fin = fmaxf(m, z);
    const float corr = expf(m - m_fin);
    l = l * corr + expf(z - m_fin);
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) acc[i] *= corr;
  } else if (sink) {
    l += expf(-m);  // the sink's weight on the scale of the running maximum
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < DIMS_PER_LANE; ++i) {
    const int d = lane + PYLON_WAVE * i;
    if (d < v_dim) orow[d] = from_float<T>(acc[i] * inv);
  }
}

// The same in float32 for few (token, head) pairs: a workgroup each, where the kernel above has a wavefront that makes
// trip after trip to memory (of 120 keys: 4 for the keys, 16 for their values).  Four wavefronts score a block of 64
// keys each, a key a lane, all of a key's elements under way at once; one or two more (64 elements of the values each)
// have the values of two blocks on their way meanwhile.  Every number is formed as above and in its order: a key's dot
// product along its elements, a block's maximum and sum over the lanes, blocks one after the other on the running
// maximum, an element's products key by key; so the bits are the same, and which kernel runs is a matter of time
// alone.  What bounds it is one trip to memory for the table and one for keys and values a round of 256 keys, and the
// chain of products.  32 heads of 128 over 8, us of the kernel above and of this: 3 tokens of about 100 keys 25.7, 8.0; 16
// of 120 27, 16.5; 8 of 700 142, 41; 1 of 8,000 1,496, 385; 1 of 1 5.9, 4.8.
template <int KD>  // elements of a key: 64 KD
__device__ __forceinline__ void paged_attention_few_body(
    float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ tok_row, const int* __restrict__ positions, int n_heads, int n_kv_heads, int page_size,
    int window, float scale, int v_dim, long long q_stride, const float* __restrict__ rel,
    const int* __restrict__ bucket, int bucket_len, int sink, float softcap, const float* __restrict__ sink_logit,
    int v_row) {
  constexpr int DIM = 64 * KD, BLOCKS = 4;  // blocks of 64 keys a round
  __shared__ __attribute__((aligned(16))) float qbuf[DIM];
  // of a round and the one before: what weighs a block's keys, their sum, the blocks' maxima
  __shared__ float weight[2][BLOCKS][PYLON_WAVE], total[2][BLOCKS], top[2][BLOCKS];
  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int t = blockIdx.x / n_heads, h = blockIdx.x - t * n_heads;
  const int kvh = h / (n_heads / n_kv_heads);
  const int pos = __builtin_amdgcn_readfirstlane(positions[t]);
  const int* table = block_table + static_cast<size_t>(__builtin_amdgcn_readfirstlane(tok_row[t])) * table_width;
  const int first = first_visible(pos, window);
  for (int i = threadIdx.x; i < DIM; i += blockDim.x)
    qbuf[i] = q[static_cast<size_t>(t) * q_stride + static_cast<size_t>(h) * DIM + i];
  __syncthreads();
  auto slot_of = [&](int j) { return table[j / page_size] * page_size + (j % page_size); };

  // The running maximum behind each block of a round, and what the sums so far are multiplied with there.
  float m = -INFINITY;
  auto follow = [&](int parity, int blocks, float (&after)[BLOCKS], float (&corr)[BLOCKS]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b)
      if (b < blocks) {
        after[b] = fmaxf(m, top[parity][b]);
        corr[b] = expf(m - after[b]);
        m = after[b];
      }
  };
  int parity = 0;
  if (wave < BLOCKS) {
    for (int base = first; base <= pos; base += BLOCKS * PYLON_WAVE, parity ^= 1) {
      const int blocks = (pos - base) / PYLON_WAVE + 1 < BLOCKS ? (pos - base) / PYLON_WAVE + 1 : BLOCKS;
      const int j = base + wave * PYLON_WAVE + lane;
      const bool valid = j <= pos;
      float s = -INFINITY;
      if (wave < blocks) {
        if (valid) {
          const float* kr = k_cache + (static_cast<size_t>(slot_of(j)) * n_kv_heads + kvh) * DIM;
          float4 key[DIM / 4];
#pragma unroll
          for (int d = 0; d < DIM / 4; ++d) key[d] = *reinterpret_cast<const float4*>(kr + 4 * d);
          float dot = 0.f;
#pragma unroll
          for (int d = 0; d < DIM / 4; ++d) {
            const float4 e = *reinterpret_cast<const float4*>(qbuf + 4 * d);
            dot = fmaf(e.x, key[d].x, dot);
            dot = fmaf(e.y, key[d].y, dot);
            dot = fmaf(e.z, key[d].z, dot);
            dot = fmaf(e.w, key[d].w, dot);
          }
          s = att_score(dot, scale, softcap, rel, bucket, bucket_len, n_heads, h, pos - j);
        }
        const float most = wave_max(s);
        if (lane == 0) top[parity][wave] = most;
      }
      __syncthreads();
      float after[BLOCKS], corr[BLOCKS];
      follow(parity, blocks, after, corr);
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b)
        if (b == wave && b < blocks) {
          const float p = valid ? expf(s - after[b]) : 0.f;
          const float sum = wave_sum(p);
          weight[parity][b][lane] = p;
          if (lane == 0) total[parity][b] = sum;
        }
      __syncthreads();
    }
    return;
  }

  const int d = (wave - BLOCKS) * PYLON_WAVE + lane;  // this lane's element of the values
  const char* const values = reinterpret_cast<const char*>(v_cache + static_cast<size_t>(kvh) * v_row);
  const unsigned row_bytes = static_cast<unsigned>(n_kv_heads) * v_row * 4u;
  float l = 0.f, acc = 0.f;
  for (int base = first; base <= pos; base += BLOCKS * PYLON_WAVE, parity ^= 1) {
    const int blocks = (pos - base) / PYLON_WAVE + 1 < BLOCKS ? (pos - base) / PYLON_WAVE + 1 : BLOCKS;
    float even[PYLON_WAVE], odd[PYLON_WAVE];
    auto bring = [&](float (&v)[PYLON_WAVE], int b) __attribute__((always_inline)) {
      if (b >= blocks) return;
      const int j = base + b * PYLON_WAVE + lane;
      const int slot = slot_of(j < pos ? j : pos);  // beyond the last key: that one again, not used
      // a view of each row: lanes beyond its elements bring zeros, without a branch; sixteen keys at a time, as many as there are
#pragma unroll
      for (int part = 0; part < PYLON_WAVE; part += 16) {
        if (part > 0 && base + b * PYLON_WAVE + part > pos) break;
#pragma unroll
        for (int k = part; k < part + 16; ++k) {
          const unsigned long long row = static_cast<unsigned long long>(static_cast<unsigned>(__builtin_amdgcn_readlane(slot, k))) * row_bytes;
          v[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(values + row), 0, v_dim * 4, 0x00020000), d * 4, 0, 0));
        }
      }
    };
    bring(even, 0);
    bring(odd, 1);
    __syncthreads();
    float after[BLOCKS], corr[BLOCKS];
    follow(parity, blocks, after, corr);
    __syncthreads();
    auto add = [&](const float (&v)[PYLON_WAVE], int b) __attribute__((always_inline)) {
      if (b >= blocks) return;
      l = l * corr[b] + total[parity][b];
      acc *= corr[b];
      const int count = pos - (base + b * PYLON_WAVE) + 1 < PYLON_WAVE ? pos - (base + b * PYLON_WAVE) + 1 : PYLON_WAVE;
      const float p = weight[parity][b][lane];
      auto weight_of = [&](int k) __attribute__((always_inline)) {
        return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), k));
      };
      if (count == PYLON_WAVE) {
#pragma unroll
        for (int k = 0; k < PYLON_WAVE; ++k) acc = fmaf(weight_of(k), v[k], acc);
      } else {
#pragma unroll
        for (int k = 0; k < PYLON_WAVE; ++k)
          if (k < count) acc = fmaf(weight_of(k), v[k], acc);
      }
    };
    add(even, 0);
    bring(even, 2);
    add(odd, 1);
    bring(odd, 3);
    add(even, 2);
    add(odd, 3);
  }
  if (sink_logit != nullptr) {
    const float z = sink_logit[h];
    const float m_fin = fmaxf(m, z);
    const float corr = expf(m - m_fin);
    l = l * corr + expf(z - m_fin);
    acc *= corr;
  } else if (sink) {
    l += expf(-m);
  }
  if (d < v_dim) out[(static_cast<size_t>(t) * n_heads + h) * v_dim + d] = acc * (1.0f / l);
}

template <int KD>
__global__ __launch_bounds__(6 * PYLON_WAVE) void paged_attention_few_kernel(
    float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ tok_row, const int* __restrict__ positions, int n_heads, int n_kv_heads, int page_size,
    int window, float scale, int v_dim, long long q_stride, const float* __restrict__ rel,
    const int* __restrict__ bucket, int bucket_len, int sink, float softcap, const float* __restrict__ sink_logit,
    int v_row) {
  paged_attention_few_body<KD>(out, q, k_cache, v_cache, block_table, table_width, tok_row, positions, n_heads, n_kv_heads,
                               page_size, window, scale, v_dim, q_stride, rel, bucket, bucket_len, sink, softcap, sink_logit, v_row);
}

// Whether the kernel of a workgroup a pair takes a float32 launch: up to two workgroups a compute unit (beyond, the
// wavefronts of the other hide each other's waits: 48 tokens of 120 keys, 32 heads, 41 us against 35; 16 of them 17
// against 27).  Where the second workgroup of a unit has five keys or fewer there is nothing to win: 9 to 16 tokens of one
// key, heads of 128 and of 64, 6.2 and 5.5 us against 6.0 and 4.9; of ten keys 6.2 and 5.6 against 6.9 and 5.8.
static bool att_few(long long items, int head_dim, int v_dim, int v_transposed) {
  return items <= 2 * pylon_compute_units() && (head_dim == 64 || head_dim == 128) && v_dim <= 128 && !v_transposed;
}

template <typename T>
static int launch_paged_attention(T* out, const T* q, const T* k_cache, const T* v_cache,
                                  const int* block_table, int table_width, const int* tok_row,
                                  const int* positions, int tokens, int n_heads, int n_kv_heads,
                                  int head_dim, int page_size, int window, float scale, int v_dim,
                                  long long q_stride, const float* rel, const int* bucket, int bucket_len,
                                  int sink, int v_transposed, float softcap, const float* sink_logit,
                                  int v_row, hipStream_t stream) {
  const long long items = static_cast<long long>(tokens) * n_heads;
  if constexpr (sizeof(T) == 4) {
    if (att_few(items, head_dim, v_dim, v_transposed)) {
      const dim3 few_grid(static_cast<unsigned>(items)), few_block((4 + (v_dim + 63) / 64) * PYLON_WAVE);
#define FEW(KD)                                                                                                  \
  hipLaunchKernelGGL((paged_attention_few_kernel<KD>), few_grid, few_block, 0, stream, out, q, k_cache, v_cache, \
                     block_table, table_width, tok_row, positions, n_heads, n_kv_heads, page_size, window, scale, \
                     v_dim, q_stride, rel, bucket, bucket_len, sink, softcap, sink_logit, v_row)
      if (head_dim == 64)
        FEW(1);
      else
        FEW(2);
#undef FEW
      return 0;
    }
  }
  const long long blocks = (items + ATT_WAVES - 1) / ATT_WAVES;
  dim3 grid((unsigned)blocks), block(ATT_WAVES * PYLON_WAVE);
  const size_t lds = sizeof(float) * ATT_WAVES * head_dim;
#define LAUNCH(DPL)                                                                                  \
  hipLaunchKernelGGL((paged_attention_kernel<T, DPL>), grid, block, lds, stream, out, q, k_cache,    \
                     v_cache, block_table, table_width, tok_row, positions, items, n_heads,          \
                     n_kv_heads, head_dim, page_size, window, scale, v_dim, q_stride, rel, bucket,   \
                     bucket_len, sink, v_transposed, softcap, sink_logit, v_row)
  if (v_dim <= 64)
    LAUNCH(1);
  else if (v_dim <= 128)
    LAUNCH(2);
  else if (v_dim <= 256)
    LAUNCH(4);
  else
    LAUNCH(8);
#undef LAUNCH
  return 0;
}

// q: [tokens, n_heads, head_dim], rows q_stride elements apart; out: [tokens, n_heads, v_dim].
// Caches: keys [pages*page_size, n_kv_heads, head_dim], values [pages*page_size, n_kv_heads, v_dim].
// v_row: elements from one value row to the next (v_dim, or more where the values are the first
// v_dim elements of wider rows: of the keys themselves, say, with v_cache the keys' cache).
// With v_transposed the values lie as [pages, n_kv_heads, v_dim, page_size].
// rel: null, or float [rows, n_heads] with bucket: int [bucket_len], every entry a row of rel; or,
// with bucket null, float [2, n_heads]: per head the factor and the slope of a logarithmic bias.
// block_table: [rows, table_width] page ids; tok_row[t] names the table row of token t;
// positions[t] is the token's index in its request; keys first(t)..positions[t] are read,
// first(t) = max(0, positions[t] - window + 1) when window > 0; the start of the token's chunk of
// -window positions when window < 0; else 0.
extern "C" int pylon_paged_attention(void* out, const void* q, const void* k_cache, const void* v_cache,
                                     int dtype, const int* block_table, int table_width,
                                     const int* tok_row, const int* positions, int tokens, int n_heads,
                                     int n_kv_heads, int head_dim, int page_size, int window,
                                     float scale, int v_dim, long long q_stride, const float* rel,
                                     const int* bucket, int bucket_len, int sink, int v_transposed,
                                     float softcap, const float* sink_logit, int v_row, hipStream_t stream) {
  PYLON_REQUIRE(pylon_valid_dtype(dtype), "paged_attention: unknown dtype");
  PYLON_REQUIRE(tokens >= 0 && n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0,
                "paged_attention: %d query heads cannot be grouped over %d key/value heads", n_heads,
                n_kv_heads);
  PYLON_REQUIRE(head_dim >= 1 && head_dim <= 1024, "paged_attention: head_dim %d must be between 1 and 1024", head_dim);
  PYLON_REQUIRE(page_size > 0 && table_width > 0, "paged_attention: bad page size or table width");
  PYLON_REQUIRE(v_dim >= 1 && v_dim <= 512, "paged_attention: values of 1 to 512 elements, got %d", v_dim);
  PYLON_REQUIRE(q_stride >= static_cast<long long>(n_heads) * head_dim, "paged_attention: q rows overlap");
  PYLON_REQUIRE(v_row >= v_dim && (v_row == v_dim || !v_transposed), "paged_attention: rows of values overlap, or are transposed and apart");
  PYLON_REQUIRE(rel == nullptr || bucket == nullptr || bucket_len >= 1,
                "paged_attention: a table of buckets holds at least one entry");
  if (tokens == 0) return 0;
  PYLON_REQUIRE(static_cast<long long>(tokens) * n_heads / ATT_WAVES < (1ll << 31),
                "paged_attention: too many (token, head) pairs for one launch");
  if (dtype == PYLON_F32)
    launch_paged_attention<float>((float*)out, (const float*)q, (const float*)k_cache,
                                  (const float*)v_cache, block_table, table_width, tok_row, positions,
                                  tokens, n_heads, n_kv_heads, head_dim, page_size, window, scale, v_dim,
                                  q_stride, rel, bucket, bucket_len, sink, v_transposed, softcap, sink_logit,
                                  v_row, stream);
  else
    launch_paged_attention<bf16_t>((bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache,
                                   (const bf16_t*)v_cache, block_table, table_width, tok_row, positions,
                                   tokens, n_heads, n_kv_heads, head_dim, page_size, window, scale, v_dim,
                                   q_stride, rel, bucket, bucket_len, sink, v_transposed, softcap, sink_logit,
                                  v_row, stream);
  PYLON_LAUNCHED("paged_attention");
}
