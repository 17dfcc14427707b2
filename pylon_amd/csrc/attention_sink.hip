// Paged causal attention with a learned bias by distance and a sink, on the matrix cores, for
// bfloat16 prompt portions and single tokens alike:
//
//   s_ij = scale * q_i.k_j + bias[head, min(i - j, bucket_len - 1)],   j <= i
//   out_i = sum_j exp(s_ij) v_j / (1 + sum_j exp(s_ij))
//
// (the learned table's rows already looked up by distance).  Keys have `dim` elements, values `vdim`.  Keys lie in the cache as [slot, kv head, dim];
// values lie transposed inside every page, [page, kv head, vdim, slot in page], so that the
// eight keys a lane feeds to a matrix instruction are neighbours in memory.
//
// A workgroup owns up to 32 consecutive tokens of one request and the (up to four) query heads of one key/value head;
// each of its eight wavefronts one head and 16 of the tokens (one tile of query columns).  It walks the keys in blocks of
// 32 (which never cross a page: pages are
// multiples of 32).  Scores are computed transposed, S^T = K Q^T (16x16x32 instructions: rows are
// keys, columns are queries), so that everything that belongs to a query (its running maximum,
// its sum, its output) lives in the lanes of that query's column, and the exponentials are
// already laid out as the operand of O^T = V^T P^T.  Scores, bias, maximum, exponentials and
// sums are float; the weights enter the value product as two bfloat16 terms, p = hi + lo, so
// that they carry sixteen bits of mantissa.  The sink is where the walk starts: maximum 0,
// sum 1, output 0.  The waves of a workgroup take heads of one key/value head at the same
// tokens: a block's keys and values are fetched once, with 16-byte loads of whole rows, into LDS
// (two buffers in turns: one barrier a block) and read from there by every wave as operands
// (rows padded against bank conflicts).  Keys
// may be cut over `cuts` workgroups, which then leave float partial results (maximum, sum,
// unnormalised output) for a second small kernel to merge in order; the sink belongs to the
// first cut.  The order of a query's sums: that of its keys, in blocks from the first key that its tile sees, cut at every
// so many blocks of its tile's walk.  A single token is a tile of its own.  A prompt portion's tiles begin where the portion
// does, and the host deals it more cuts the fewer tiles its step has and the longer the step's longest request is: the same
// tokens alone and beside others are other roundings of the same sums, each as near to the exact ones.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_at8 __attribute__((aligned(8)));  // sixteen bytes of a cache of values, which begins at any eighth byte

#define AS_BLOCK 32   // keys per step of the walk
#define AS_MAX_BIAS 4096
// Waves a SIMD of the prompt kernel: two workgroups a compute unit where the outputs and queries leave the registers, at
// values of up to 128 (the host counts on two for keys of up to 192: ops._sink_launch).
#define AS_WAVES(KS, NV) ((NV) <= 8 ? 4 : 2)
// And of the kernel of single tokens, whose largest instance (heads beyond 128 in both) needs more than half of the
// registers: asked for two it had 67 of them in scratch memory (heads of 256, 128 requests of 500 keys: 129 -> 161 us).
#define AS_SINGLE_WAVES(KS, NV) ((KS) > 4 && (NV) > 8 ? 1 : 2)
#define AS_LOG2E 1.4426950408889634f

__device__ __forceinline__ uint32_t as_pack(float a, float b) {
  return floats_to_bf16_pair(a, b);
}

// KS: steps of 32 key elements (dim <= 32 KS); NV: tiles of 16 value elements (vdim <= 16 NV).
// scale * s, or with a cap c > 0: c * tanh(scale * s / c), the tangent as 1 - 2 / (e^(2x) + 1)
// (it ends at 1 and -1 where the exponential overflows or vanishes).
__device__ __forceinline__ float capped_score(float s, float scale, float cap) {
  const float v = s * scale;
  if (!(cap > 0.f)) return v;
  const float e = __expf(2.0f * v / cap);
  return cap * (1.0f - 2.0f / (e + 1.0f));
}

template <bool V>
struct as_flag {
  static constexpr bool value = V;
};

// e to the power of a difference.  (Scores stay as they are and only the differences are multiplied with log2 e: kept
// times log2 e, they saved one multiplication each, but a finite one could become infinite, and beside biases of 60 and
// of 400 the float sums were up to 2.0 and 2.6 times as far from 64 bits.)
__device__ __forceinline__ float as_exp(float v) { return __builtin_amdgcn_exp2f(v * AS_LOG2E); }

// The largest over the four lanes of a query's column, on the vector unit (two trips through LDS with shuffles).
__device__ __forceinline__ float as_column_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// FULL: keys of exactly 32 KS elements and values of exactly 16 NV, the strides in LDS constants.
//
// What bounds it is the issue of a block's vector and matrix instructions (1.1 us a block of 32 keys and compute unit with
// four waves a SIMD, of which the matrix instructions take 0.3), and for the tile with the longest walk that walk's own
// length (1.2 us a block with nothing beside it).  The registers are kept at 128 so that two workgroups share a compute
// unit: with 145 the second one waited for the first to end.  The questions that are the same for a whole wave (does it
// work, is there a cap, are the keys near, far, hidden) are asked once a block: asked inside the loops over the operands
// they had put a branch and a wait for all loads before every matrix instruction.  The loads of the queries are waited
// for before the walk.  Keys are written to LDS in the order that makes a lane's eight weights those of eight neighbours:
// one 16-byte piece of values.  32 heads of 128 over 8, 2,048 tokens, bias over 2,049 distances: 153 -> 90 us; behind
// 952 cached ones 275 -> 134; behind 452 in a window of 1,024 without a bias 143 -> 71; 40 tokens 10.4 -> 9.0.
template <int KS, int NV, bool FULL>
__global__ __launch_bounds__(512, AS_WAVES(KS, NV)) void attention_sink_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, long long q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ tiles, const int* __restrict__ positions, int n_heads, int n_kv_heads, int dim_arg, int vdim_arg, int page_size, float scale,
    const float* __restrict__ bias, int bucket_len, int sink, int cuts, float* __restrict__ partial, int window,
    float softcap, const float* __restrict__ sink_logit) {
  // eight waves: wave & 3 names the head of the group, wave >> 2 which 16 of the tile's 32 tokens
  const int dim = FULL ? 32 * KS : dim_arg, vdim = FULL ? 16 * NV : vdim_arg;
  constexpr int waves_per_group = 4;
  constexpr int KL = (KS + 3) / 4, VL = (NV + 7) / 8;  // 16-byte pieces of a block a thread fetches
  constexpr bool KEYS_FIT = FULL && KS % 4 == 0, VALUES_FIT = FULL && NV % 8 == 0;  // every thread has its pieces
  extern __shared__ float bias_lds[];  // [heads of the workgroup][bucket_len], then the block's keys and values
  const int lane = threadIdx.x & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave_id & 3, qsel = wave_id >> 2;
  const int col = lane & 15, grp = lane >> 4;
  const int group = n_heads / n_kv_heads;
  const int chunks = (group + waves_per_group - 1) / waves_per_group;
  int b = blockIdx.x;
  const int cut = b % cuts;
  b /= cuts;
  const int chunk = b % chunks;
  b /= chunks;
  const int kvh = b % n_kv_heads;
  const int tile = b / n_kv_heads;
  const int in_group = chunk * waves_per_group + wave;
  const bool idle = in_group >= group;  // a wave beyond the group's heads helps to fetch and stores nothing
  const int head = kvh * group + (idle ? group - 1 : in_group);
  // without a table of tiles every token is a tile of its own and row t of the block table is token t's
  const int tok0 = tiles ? tiles[4 * tile] : tile, count = tiles ? tiles[4 * tile + 1] : 1;
  const int row = tiles ? tiles[4 * tile + 2] : tile, pos0 = tiles ? tiles[4 * tile + 3] : positions[tile];
  const int kv_last = pos0 + count - 1;
  const bool works = !idle && (qsel == 0 || count > 16);  // other waves only help to fetch
  const int* table = block_table + static_cast<size_t>(row) * table_width;

  const int tstride = (bucket_len + 3) & ~3;  // keeps what follows the tables 16-byte aligned
  float* tbl = bias_lds + wave * tstride;
  const int kstr = dim + 8, vstr = AS_BLOCK + 8;  // LDS rows, padded against bank conflicts
  // two buffers of a block's keys and values, used in turns
  bf16_t* kv_lds = reinterpret_cast<bf16_t*>(bias_lds + waves_per_group * tstride);
  const int buf_elems = AS_BLOCK * kstr + ((vdim + 15) & ~15) * vstr;
  constexpr int threads = 2 * waves_per_group * 64;
  const float* bias_row = bias ? bias + static_cast<size_t>(head) * bucket_len : nullptr;
  if (bias != nullptr) {
#pragma unroll 8
    for (int d = lane; d < bucket_len; d += 64) tbl[d] = bias_row[d];
  }
  const float far_bias = bias != nullptr ? bias_row[bucket_len - 1] : 0.f;
  const float left = softcap > 0.f ? 1.f : scale;  // a capped score has its scale

  // Q^T operands: column = query, eight key elements per lane and step
  bf16x8 qf[KS];
  const int qi = qsel * 16 + col;
  const int qpos = pos0 + qi, qfirst = first_visible(qpos, window);  // the query's position and the first key it sees
  {
    const int t = tok0 + (qi < count ? qi : count - 1);
    const bf16_t* qr = q + static_cast<size_t>(t) * q_stride + static_cast<size_t>(head) * dim;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d = ks * 32 + grp * 8;
      u32x4 raw = {0u, 0u, 0u, 0u};
      if (FULL || d < dim) raw = *reinterpret_cast<const u32x4*>(qr + d);
      qf[ks] = __builtin_bit_cast(bf16x8, raw);
    }
  }

  floatx4 o[NV];
  // the sink: a key without a value (one lane of a query's four carries its one) whose score is 0,
  // or the head's learned number
  float m_run = (sink && cut == 0) ? (sink_logit != nullptr ? sink_logit[head] : 0.f) : -INFINITY;
  float l_run = (sink && cut == 0 && grp == 0) ? 1.f : 0.f;
#pragma unroll
  for (int dt = 0; dt < NV; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};

  // the walk starts at the block of the first key that the tile's first query sees
  const int kb_first = first_visible(pos0, window) / AS_BLOCK * AS_BLOCK;
  const int n_blocks = (kv_last - kb_first) / AS_BLOCK + 1;
  const int per_cut = (n_blocks + cuts - 1) / cuts;
  const int kb_begin = kb_first + cut * per_cut * AS_BLOCK;
  const int kb_end = kb_first + ((cut + 1) * per_cut < n_blocks ? (cut + 1) * per_cut : n_blocks) * AS_BLOCK;
  const int wave_first = pos0 + qsel * 16, last_first = first_visible(wave_first + 15, window);
  // A block's keys and values travel global -> registers -> LDS; the registers of block b + 1
  // are filled while block b is computed.
  u32x4 kreg[KL], vreg[VL];
  const int kchunks = dim >> 3;  // 16-byte pieces of a key row
  // where this thread's pieces lie, in the caches behind a block's first key and in LDS
  int k_from[KL], k_to[KL], v_to[VL];
  long long v_from[VL];
#pragma unroll
  for (int n = 0; n < KL; ++n) {
    const int c = threadIdx.x + n * threads, r = c / kchunks, e = (c - r * kchunks) * 8;
    k_from[n] = r * n_kv_heads * dim + e, k_to[n] = ((r & 4) * 4 + (r >> 3) * 4 + (r & 3)) * kstr + e;
  }
#pragma unroll
  for (int n = 0; n < VL; ++n) {
    const int c = threadIdx.x + n * threads, r = c / (AS_BLOCK / 8), e = (c - r * (AS_BLOCK / 8)) * 8;
    v_from[n] = static_cast<long long>(r) * page_size + e, v_to[n] = AS_BLOCK * kstr + r * vstr + e;
  }
  int page_at = kb_begin / page_size, in_page = kb_begin - page_at * page_size;  // of the block that is fetched next
  int kb_next = kb_begin, page = kb_begin < kb_end ? table[page_at] : 0;
  auto fetch = [&]() {
    const bf16_t* kbase = k_cache + ((static_cast<size_t>(page) * page_size + in_page) * n_kv_heads + kvh) * dim;
#pragma unroll
    for (int n = 0; n < KL; ++n) {
      const int c = threadIdx.x + n * threads;
      if (KEYS_FIT || c < AS_BLOCK * kchunks) kreg[n] = *reinterpret_cast<const u32x4*>(kbase + k_from[n]);
    }
    const bf16_t* vbase = v_cache + (static_cast<size_t>(page) * n_kv_heads + kvh) * vdim * page_size + in_page;
#pragma unroll
    for (int n = 0; n < VL; ++n) {
      const int c = threadIdx.x + n * threads;
      if (VALUES_FIT || c < vdim * (AS_BLOCK / 8)) vreg[n] = *reinterpret_cast<const u32x4_at8*>(vbase + v_from[n]);
    }
    in_page += AS_BLOCK, kb_next += AS_BLOCK;
    if (in_page == page_size && kb_next < kb_end) in_page = 0, page = table[++page_at];
  };
  auto stage = [&](int turn, int kb) {
    bf16_t* const block = kv_lds + turn * buf_elems;
    if (kb + AS_BLOCK - 1 > kv_last) {  // slots past the request's end hold anything; their weights are 0, and so are they
#pragma unroll
      for (int n = 0; n < VL; ++n) {
        const int first = kb + (threadIdx.x + n * threads) % (AS_BLOCK / 8) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (first + e > kv_last) vreg[n][e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
      }
    }
#pragma unroll
    for (int n = 0; n < KL; ++n) {
      const int c = threadIdx.x + n * threads;
      if (KEYS_FIT || c < AS_BLOCK * kchunks) *reinterpret_cast<u32x4*>(block + k_to[n]) = kreg[n];
    }
#pragma unroll
    for (int n = 0; n < VL; ++n) {
      const int c = threadIdx.x + n * threads;
      if (VALUES_FIT || c < vdim * (AS_BLOCK / 8)) *reinterpret_cast<u32x4*>(block + v_to[n]) = vreg[n];
    }
  };
  // Block b is computed from one buffer while block b + 1, fetched during block b - 1's math, is
  // written to the other and block b + 2 is sent for: one barrier a block.
  if (kb_begin < kb_end) fetch();
  __builtin_amdgcn_s_waitcnt(0x0f70);  // of all loads: a wait for the queries inside the walk would be one for the next block
  if (kb_begin < kb_end) {
    stage(0, kb_begin);
    if (kb_begin + AS_BLOCK < kb_end) fetch();
  }
  __syncthreads();
  int turn = 0;
  for (int kb = kb_begin; kb < kb_end; kb += AS_BLOCK, turn ^= 1) {
    const bf16_t* k_lds = kv_lds + turn * buf_elems;
    const bf16_t* v_lds = k_lds + AS_BLOCK * kstr;
    if (works) {
      // K operands: row 16 t + 4 g + i of the block in LDS = key 8 g + 4 t + i, eight elements per lane and step: a lane's
      // eight scores are of eight keys side by side, whose values it then reads as one piece
      floatx4 s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16_t* kr = k_lds + (t * 16 + col) * kstr;
        s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int d = ks * 32 + grp * 8;
          u32x4 raw = {0u, 0u, 0u, 0u};
          if (FULL || d < dim) raw = *reinterpret_cast<const u32x4*>(kr + d);
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, raw), qf[ks], s[t], 0, 0, 0);
        }
      }
      // Scores of this lane: keys kb + 8 grp + e for query qpos.  Three ways, one question a block for the whole
      // wave: every query sees every key and all are far (or there is no bias), or all near, or anything.
      float sc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = s[e >> 2][e & 3];
      if (softcap > 0.f) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sc[e] = capped_score(sc[e], scale, softcap);
      }
      const bool seen = kb + AS_BLOCK - 1 <= wave_first && kb >= last_first;
      if (seen && (bias == nullptr || wave_first - (kb + AS_BLOCK - 1) >= bucket_len - 1)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sc[e] = fmaf(sc[e], left, far_bias);
      } else if (seen && wave_first + 15 - kb < bucket_len) {
        const float* const near = tbl + (qpos - kb - 8 * grp - 7);
#pragma unroll
        for (int e = 0; e < 8; ++e) sc[e] = fmaf(sc[e], left, near[7 - e]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = kb + 8 * grp + e, dist = qpos - key;
          const int idx = dist < 0 ? 0 : dist < bucket_len - 1 ? dist : bucket_len - 1;
          const float v = fmaf(sc[e], left, bias == nullptr ? 0.f : tbl[idx]);
          sc[e] = (dist >= 0 && key >= qfirst) ? v : -INFINITY;
        }
      }
      float top = m_run;
#pragma unroll
      for (int e = 0; e < 8; ++e) top = fmaxf(top, sc[e]);
      top = as_column_max(top);
      // a query past the tile's end, or one whose every key so far is hidden, keeps -inf: no NaN from inf - inf
      const float base = (top == -INFINITY) ? 0.f : top;
      const float corr = (top == -INFINITY) ? 1.f : as_exp(m_run - top);
      float p[8], sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = as_exp(sc[e] - base);
        sum += p[e];
      }
      l_run = l_run * corr + sum;
      m_run = top;
      u32x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        // hi: the upper sixteen bits of p as they are; lo: those of the rest (p - hi is exact)
        const uint32_t a = __float_as_uint(p[e]), c = __float_as_uint(p[e + 1]);
        hi[e >> 1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
        const float ra = p[e] - __uint_as_float(a & 0xffff0000u), rc = p[e + 1] - __uint_as_float(c & 0xffff0000u);
        lo[e >> 1] = __builtin_amdgcn_perm(__float_as_uint(rc), __float_as_uint(ra), 0x07060302u);
      }
      const bf16x8 p_hi = __builtin_bit_cast(bf16x8, hi), p_lo = __builtin_bit_cast(bf16x8, lo);
      if (__any(corr != 1.f)) {  // else no query of the wave raised its maximum: nothing to scale
#pragma unroll
        for (int dt = 0; dt < NV; ++dt) o[dt][0] *= corr, o[dt][1] *= corr, o[dt][2] *= corr, o[dt][3] *= corr;
      }
      // V^T operands: row = value element, keys kb + 8 grp + {0..7}
#pragma unroll
      for (int dt = 0; dt < NV; ++dt) {
        const int d = dt * 16 + col;
        u32x4 raw = {0u, 0u, 0u, 0u};
        if (FULL || d < vdim) raw = *reinterpret_cast<const u32x4*>(v_lds + d * vstr + 8 * grp);
        const bf16x8 vf = __builtin_bit_cast(bf16x8, raw);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_hi, o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_lo, o[dt], 0, 0, 0);
      }
    }
    if (kb + AS_BLOCK < kb_end) {
      stage(turn ^ 1, kb + AS_BLOCK);  // nobody reads that buffer: the block before this one is done everywhere
      if (kb + 2 * AS_BLOCK < kb_end) fetch();
    }
    __syncthreads();
  }

  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (qi >= count || idle) return;
  if (cuts > 1) {
    // [token, head, cut, 2 + vdim]: maximum, sum, unnormalised output
    float* dst = partial + ((static_cast<size_t>(tok0 + qi) * n_heads + head) * cuts + cut) * (2 + vdim);
    if (grp == 0) {
      dst[0] = m_run;
      dst[1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < NV; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (dt * 16 + 4 * grp + i < vdim) dst[2 + dt * 16 + 4 * grp + i] = o[dt][i];
    return;
  }
  const float inv = 1.0f / l;
  bf16_t* orow = out + (static_cast<size_t>(tok0 + qi) * n_heads + head) * vdim;
#pragma unroll
  for (int dt = 0; dt < NV; ++dt) {
    const int d = dt * 16 + 4 * grp;
    if (d + 3 < vdim) {
      u32x2 packed = {as_pack(o[dt][0] * inv, o[dt][1] * inv), as_pack(o[dt][2] * inv, o[dt][3] * inv)};
      *reinterpret_cast<u32x2*>(orow + d) = packed;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (d + i < vdim) orow[d + i].bits = float_to_bf16_bits(o[dt][i] * inv);
    }
  }
}

// A step of single tokens: one workgroup per (token, key/value head, cut of the keys).  The heads of
// the group (at most 16) sit side by side in the query columns of one tile, all at the token's
// position, so a block's scores for the whole group cost what one head's cost; the four waves take
// every fourth block of the cut and fetch their operands themselves (no wave reads what another
// fetched, so nothing is staged and nothing waits at a barrier); at the end the four waves' partial
// results (maximum, sum, unnormalised output, all float) meet in LDS and are merged in the order of
// the waves: into the output if the keys are not cut, else into the cut's partial result for the
// merge kernel.
//
// What bounds it is the chain of loads of a wave's few blocks, not the bytes: position, page, then the
// block's keys, biases and values, which all go out before the first is used; the registers of each are
// filled for the next block as soon as this block is done with them.  The biases are gathered by distance
// straight from the table: a workgroup needs a few hundred entries of it, and copying all of a group's
// tables to LDS first (32 KB at 2,048 distances and four heads) took longer than the walk itself.
// The last block is a step of its own and nothing in a step is asked per operand, so that a wait is one for what
// it is about (the first matrix instruction had waited for every load, the values' too); a lane's eight keys are
// neighbours, their values one piece of 16 bytes; two waves a SIMD are asked for, which keeps the sums out of the
// accumulation registers (each block had moved them there and back).
// 32 heads of 128 over 8 and 2,048 distances, with the merge: 4 requests of 1,524 keys in 16 cuts 12.8 -> 10.0 us,
// 4 of 700 in 8 9.7 -> 7.7, 1 of 8,000 in 64 16.9 -> 13.6, 16 of 1,524 in 4 26.6 -> 20.2, 64 of 1,000, uncut, 48.5
// -> 36.3, 4 of 40 6.4 -> 4.7; without a bias, 2 of 2,524 in a window of 1,024 and 8 cuts 11.7 -> 8.3.
template <int KS, int NV, bool FULL>
__global__ __launch_bounds__(256, AS_SINGLE_WAVES(KS, NV)) void attention_sink_decode_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, long long q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ positions, int n_heads, int n_kv_heads, int dim_arg, int vdim_arg, int page_size, float scale,
    const float* __restrict__ bias, int bucket_len, int sink, int cuts, float* __restrict__ partial, int window,
    float softcap, const float* __restrict__ sink_logit) {
  extern __shared__ float mrg[];  // [4 waves][group][2 + vdim]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int dim = FULL ? 32 * KS : dim_arg, vdim = FULL ? 16 * NV : vdim_arg;
  const int group = n_heads / n_kv_heads;
  int b = blockIdx.x;
  const int cut = b % cuts;
  b /= cuts;
  const int kvh = b % n_kv_heads;
  const int tok = b / n_kv_heads;
  const int pos = positions[tok];
  const int* table = block_table + static_cast<size_t>(tok) * table_width;
  const int my_head = kvh * group + (col < group ? col : group - 1);  // columns past the group repeat its last head
  const float* bias_row = bias + static_cast<size_t>(my_head) * bucket_len;  // read only if there is a bias

  const int first_key = first_visible(pos, window);  // a window, a chunk: the walk starts at its block
  const int kb_first = first_key / AS_BLOCK * AS_BLOCK;
  const int n_blocks = (pos - kb_first) / AS_BLOCK + 1;
  const int per_cut = (n_blocks + cuts - 1) / cuts;
  const int kb_begin = kb_first + cut * per_cut * AS_BLOCK;
  const int kb_end = kb_first + ((cut + 1) * per_cut < n_blocks ? (cut + 1) * per_cut : n_blocks) * AS_BLOCK;

  u32x4 kraw[2][KS];
  u32x4 vraw[NV];
  float add[8];
  // row 4 g + i of tile t is key 8 g + 4 t + i of the block: a lane's eight scores are of eight neighbours
  const int key_row = (col >> 2) * 8 + (col & 3);
  auto load_keys = [&](int kb, int page) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const size_t slot = static_cast<size_t>(page) * page_size + kb % page_size + key_row + 4 * t;
      const bf16_t* kr = k_cache + (slot * n_kv_heads + kvh) * dim;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d = ks * 32 + grp * 8;
        kraw[t][ks] = u32x4{0u, 0u, 0u, 0u};
        if (FULL || d < dim) kraw[t][ks] = *reinterpret_cast<const u32x4*>(kr + d);
      }
    }
  };
  auto load_bias = [&](int kb) {
    if (bias == nullptr) {
#pragma unroll
      for (int e = 0; e < 8; ++e) add[e] = 0.f;
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int idx = pos - (kb + 8 * grp + e);
      idx = idx < 0 ? 0 : (idx < bucket_len - 1 ? idx : bucket_len - 1);
      add[e] = bias_row[idx];
    }
  };
  auto load_values = [&](int kb, int page) {
    const bf16_t* block = v_cache + (static_cast<size_t>(page) * n_kv_heads + kvh) * vdim * page_size + kb % page_size + 8 * grp;
#pragma unroll
    for (int dt = 0; dt < NV; ++dt) {
      const int d = dt * 16 + col;
      vraw[dt] = u32x4{0u, 0u, 0u, 0u};
      if (FULL || d < vdim) vraw[dt] = *reinterpret_cast<const u32x4_at8*>(block + static_cast<size_t>(d) * page_size);
    }
  };

  int kb = kb_begin + wave * AS_BLOCK;
  floatx4 o[NV];
#pragma unroll
  for (int dt = 0; dt < NV; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  const float left = softcap > 0.f ? 1.f : scale;  // a capped score has its scale
  const bool first = sink && cut == 0 && wave == 0;  // the sink belongs to one partial result
  float m_run = first ? (sink_logit != nullptr ? sink_logit[my_head] : 0.f) : -INFINITY;
  float l_run = (first && grp == 0) ? 1.f : 0.f;
  bf16x8 qf[KS];

  // One block; with another behind it the registers are filled again as they come free (no branch in between, so that a
  // wait for the keys is one for the keys).
  auto step = [&](auto another) __attribute__((always_inline)) {
    constexpr bool more = decltype(another)::value;
    const int next = kb + 4 * AS_BLOCK, next_page = more ? table[next / page_size] : 0;
    floatx4 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kraw[t][ks]), qf[ks], s[t], 0, 0, 0);
    }
    if (more) load_keys(next, next_page);
    float sc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sc[e] = s[e >> 2][e & 3];
    if (softcap > 0.f) {  // asked once: inside the loop it is a branch and a wait for all loads a score
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = capped_score(sc[e], scale, softcap);
    }
    float top = m_run;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int key = kb + 8 * grp + e;
      const float v = fmaf(sc[e], left, add[e]);
      sc[e] = (key <= pos && key >= first_key) ? v : -INFINITY;
      top = fmaxf(top, sc[e]);
    }
    if (more) load_bias(next);
    top = as_column_max(top);
    const float base = (top == -INFINITY) ? 0.f : top;  // no key so far: no NaN from inf - inf
    const float corr = (top == -INFINITY) ? 1.f : as_exp(m_run - top);
    float p[8], sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = as_exp(sc[e] - base);
      sum += p[e];
    }
    l_run = l_run * corr + sum;
    m_run = top;
    u32x4 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const uint32_t a = __float_as_uint(p[e]), c = __float_as_uint(p[e + 1]);
      hi[e >> 1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
      const float ra = p[e] - __uint_as_float(a & 0xffff0000u), rc = p[e + 1] - __uint_as_float(c & 0xffff0000u);
      lo[e >> 1] = __builtin_amdgcn_perm(__float_as_uint(rc), __float_as_uint(ra), 0x07060302u);
    }
    const bf16x8 p_hi = __builtin_bit_cast(bf16x8, hi), p_lo = __builtin_bit_cast(bf16x8, lo);
    if (!more && kb + AS_BLOCK - 1 > pos) {  // slots behind the token may hold anything; they lie in the last block
#pragma unroll
      for (int dt = 0; dt < NV; ++dt)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (kb + 8 * grp + e > pos) vraw[dt][e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
    }
#pragma unroll
    for (int dt = 0; dt < NV; ++dt) {
      const bf16x8 vf = __builtin_bit_cast(bf16x8, vraw[dt]);
      floatx4 acc = o[dt];
      acc[0] *= corr; acc[1] *= corr; acc[2] *= corr; acc[3] *= corr;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_hi, acc, 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_lo, acc, 0, 0, 0);
    }
    if (more) load_values(next, next_page);
    kb = next;
  };
  if (kb < kb_end) {  // all its loads in here: a path without them would end the loop's waits early
    const bf16_t* qr = q + static_cast<size_t>(tok) * q_stride + static_cast<size_t>(my_head) * dim;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d = ks * 32 + grp * 8;
      u32x4 raw = {0u, 0u, 0u, 0u};
      if (FULL || d < dim) raw = *reinterpret_cast<const u32x4*>(qr + d);
      qf[ks] = __builtin_bit_cast(bf16x8, raw);
    }
    const int page = table[kb / page_size];
    load_keys(kb, page);
    load_bias(kb);
    load_values(kb, page);
    while (kb + 4 * AS_BLOCK < kb_end) step(as_flag<true>{});
    step(as_flag<false>{});
  }
  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (col < group) {
    float* mine = mrg + (wave * group + col) * (2 + vdim);
    if (grp == 0) {
      mine[0] = m_run;
      mine[1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < NV; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (dt * 16 + 4 * grp + i < vdim) mine[2 + dt * 16 + 4 * grp + i] = o[dt][i];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < group * vdim; idx += 256) {
    const int h = idx / vdim, d = idx - h * vdim;
    const float* src = mrg + h * (2 + vdim);
    const int stride = group * (2 + vdim);
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, src[w * stride]);
    float total = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = src[w * stride];
      const float f = (mw == -INFINITY) ? 0.f : as_exp(mw - m);
      total = fmaf(src[w * stride + 1], f, total);
      acc = fmaf(src[w * stride + 2 + d], f, acc);
    }
    const size_t item = static_cast<size_t>(tok) * n_heads + kvh * group + h;
    if (cuts == 1) {
      out[item * vdim + d].bits = float_to_bf16_bits(acc / total);
    } else {
      float* dst = partial + (item * cuts + cut) * (2 + vdim);
      if (d == 0) {
        dst[0] = m;
        dst[1] = total;
      }
      dst[2 + d] = acc;
    }
  }
}

// One wave per 64 values of a (token, head): out = sum_c o_c e^(m_c - m) / sum_c l_c e^(m_c - m), cuts in
// order.  All it does is wait for loads, so sixteen cuts' are sent for together with the maxima and sums.
__global__ void attention_sink_merge_kernel(bf16_t* __restrict__ out, const float* __restrict__ partial, int items,
                                            int cuts, int vdim) {
  const int chunks = (vdim + 63) / 64;
  const int unit = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int item = unit / chunks, d = (unit - item * chunks) * 64 + (threadIdx.x & 63);
  const int lane = threadIdx.x & 63;
  if (item >= items) return;
  const float* src = partial + static_cast<size_t>(item) * cuts * (2 + vdim);
  // lane c takes cut c's maximum and sum (at most 64 cuts)
  const float mc = lane < cuts ? src[lane * (2 + vdim)] : -INFINITY;
  const float lc = lane < cuts ? src[lane * (2 + vdim) + 1] : 0.f;
  const bool mine = d < vdim;  // every lane stays in the loop: its weight is read by the others
  constexpr int BATCH = 16;
  float part[BATCH];
  auto load = [&](int c0) {
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      part[j] = 0.f;
      if (mine && c0 + j < cuts) part[j] = src[(c0 + j) * (2 + vdim) + 2 + d];
    }
  };
  load(0);
  const float m = wave_max(mc);
  const float w = (mc == -INFINITY) ? 0.f : __expf(mc - m);
  const float inv = 1.0f / wave_sum(lc * w);
  float acc = 0.f;
  for (int c0 = 0; c0 < cuts; c0 += BATCH) {
#pragma unroll
    for (int j = 0; j < BATCH; ++j)  // beyond the last cut the weight and the value are zero
      acc = fmaf(part[j], __shfl(w, c0 + j, 64), acc);
    if (c0 + BATCH < cuts) load(c0 + BATCH);
  }
  if (mine) out[static_cast<size_t>(item) * vdim + d].bits = float_to_bf16_bits(acc * inv);
}

// The instances for heads of these sizes.
typedef decltype(&attention_sink_kernel<1, 2, false>) SinkPrompt;
typedef decltype(&attention_sink_decode_kernel<1, 2, false>) SinkSingle;
#define AS_OF_VALUES(KERNEL, KS) \
  (nv <= 2 ? &KERNEL<KS, 2, false> : nv <= 4 ? &KERNEL<KS, 4, false> : nv <= 8 ? &KERNEL<KS, 8, false> : &KERNEL<KS, 16, false>)
#define AS_OF_SIZES(KERNEL)                                                                       \
  (ks <= 1 ? AS_OF_VALUES(KERNEL, 1) : ks <= 2 ? AS_OF_VALUES(KERNEL, 2) : ks <= 4 ? AS_OF_VALUES(KERNEL, 4) \
                                                                                   : AS_OF_VALUES(KERNEL, 8))

static SinkPrompt prompt_kernel(int dim, int vdim) {
  const int ks = (dim + 31) / 32, nv = (vdim + 15) / 16;
  // the sizes of the usual heads with their strides as constants (128 and 128, 2,048 tokens: 115 -> 106 registers)
  if (dim == 64 && vdim == 64) return &attention_sink_kernel<2, 4, true>;
  if (dim == 128 && vdim == 128) return &attention_sink_kernel<4, 8, true>;
  if (dim == 192 && vdim == 128) return &attention_sink_kernel<6, 8, true>;
  return AS_OF_SIZES(attention_sink_kernel);
}

static SinkSingle single_kernel(int dim, int vdim) {
  const int ks = (dim + 31) / 32, nv = (vdim + 15) / 16;
  if (dim == 64 && vdim == 64) return &attention_sink_decode_kernel<2, 4, true>;
  if (dim == 128 && vdim == 128) return &attention_sink_decode_kernel<4, 8, true>;
  return AS_OF_SIZES(attention_sink_decode_kernel);
}
#undef AS_OF_SIZES
#undef AS_OF_VALUES

static size_t prompt_lds(int dim, int vdim, int table_len) {  // four heads' biases, two buffers of bfloat16
  return sizeof(float) * 4 * ((table_len + 3) & ~3) +
         2 * 2 * (static_cast<size_t>(AS_BLOCK) * (dim + 8) + static_cast<size_t>((vdim + 15) / 16 * 16) * (AS_BLOCK + 8));
}

// What a compute unit makes of the kernels for heads of these sizes: the workgroups of the prompt kernel that it holds at
// once beside tables of `bucket_len` distances (0: no bias), and the scratch memory of a lane, of the prompt kernel and of
// the one of single tokens (the registers that did not fit).
extern "C" int pylon_attention_sink_resources(int dim, int vdim, int bucket_len, int* workgroups, int* prompt_scratch,
                                              int* single_scratch) {
  PYLON_REQUIRE(dim >= 8 && dim % 8 == 0 && dim <= 256 && vdim >= 4 && vdim % 4 == 0 && vdim <= 256 && bucket_len >= 0 &&
                    bucket_len <= AS_MAX_BIAS && workgroups && prompt_scratch && single_scratch,
                "attention_sink_resources: sizes that the kernels do not take");
  const void* prompt = reinterpret_cast<const void*>(prompt_kernel(dim, vdim));
  const size_t lds = prompt_lds(dim, vdim, bucket_len > 0 ? bucket_len : 1);
  hipFuncAttributes of_prompt, of_single;
  PYLON_REQUIRE(hipFuncGetAttributes(&of_prompt, prompt) == hipSuccess &&
                    hipFuncGetAttributes(&of_single, reinterpret_cast<const void*>(single_kernel(dim, vdim))) == hipSuccess &&
                    hipOccupancyMaxActiveBlocksPerMultiprocessor(workgroups, prompt, 512, lds) == hipSuccess,
                "attention_sink_resources: the device does not say");
  *prompt_scratch = static_cast<int>(of_prompt.localSizeBytes);
  *single_scratch = static_cast<int>(of_single.localSizeBytes);
  return 0;
}

// q: bf16 [tokens, n_heads, dim], rows q_stride elements apart; out: bf16 [tokens, n_heads, vdim].
// k_cache: bf16 [pages * page_size, n_kv_heads, dim]; v_cache: bf16 [pages, n_kv_heads, vdim, page_size].
// tiles: int [n_tiles, 4] = (first token, count <= 32, block-table row, first position) of runs of
// consecutive tokens of one request; or null, and then positions: int [n_tiles], one token per tile,
// token t on row t of the block table (a step of single tokens).  bias: null or float [n_heads, bucket_len
// <= 4096], a head's bias by distance, the last entry for every distance from bucket_len - 1 on.  dim a multiple of 8 up to 256, vdim a multiple of 4
// up to 256, page_size a multiple of 32.  window: the mask as one integer (first_visible in common.h).
// The host guarantees that the tiles lie inside q and the table.
extern "C" int pylon_attention_sink(void* out, const void* q, long long q_stride, const void* k_cache,
                                    const void* v_cache, const int* block_table, int table_width, const int* tiles,
                                    const int* positions, int n_tiles, int n_heads, int n_kv_heads, int dim, int vdim, int page_size,
                                    float scale, const float* bias, int bucket_len, int sink,
                                    int cuts, float* partial, long long partial_floats, int tokens, int window,
                                    float softcap, const float* sink_logit, hipStream_t stream) {
  PYLON_REQUIRE(sink_logit == nullptr || sink, "attention_sink: a learned sink is a sink");
  PYLON_REQUIRE(n_tiles >= 0 && n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0,
                "attention_sink: %d query heads cannot be grouped over %d key/value heads", n_heads, n_kv_heads);
  PYLON_REQUIRE(dim >= 8 && dim % 8 == 0 && dim <= 256, "attention_sink: keys of a multiple of 8 up to 256 elements, got %d", dim);
  PYLON_REQUIRE(vdim >= 4 && vdim % 4 == 0 && vdim <= 256, "attention_sink: values of a multiple of 4 up to 256 elements, got %d", vdim);
  PYLON_REQUIRE(page_size > 0 && page_size % AS_BLOCK == 0, "attention_sink: pages of a multiple of %d tokens, got %d", AS_BLOCK, page_size);
  PYLON_REQUIRE(table_width > 0 && q_stride >= static_cast<long long>(n_heads) * dim && q_stride % 8 == 0,
                "attention_sink: bad table width or q stride");
  PYLON_REQUIRE((reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(k_cache) & 15) == 0 &&
                (reinterpret_cast<uintptr_t>(v_cache) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
                "attention_sink: q and keys must be 16-byte aligned, values and results 8-byte");
  PYLON_REQUIRE(tiles != nullptr || positions != nullptr, "attention_sink: tiles or positions are required");
  PYLON_REQUIRE(bias == nullptr || (bucket_len >= 1 && bucket_len <= AS_MAX_BIAS),
                "attention_sink: a bias by distance is a table of 1 to %d entries a head", AS_MAX_BIAS);
  PYLON_REQUIRE(cuts >= 1 && cuts <= 64, "attention_sink: 1 to 64 cuts, got %d", cuts);
  const int group = n_heads / n_kv_heads;
  // single tokens whose group of heads fits a tile's columns: the kernel with the heads side by side
  const bool side_by_side = tiles == nullptr && group <= 16 &&
                            (cuts == 1 || (partial != nullptr &&
                                           partial_floats >= static_cast<long long>(tokens) * n_heads * cuts * (2 + vdim)));
  PYLON_REQUIRE(side_by_side || cuts == 1 ||
                    (partial != nullptr && partial_floats >= static_cast<long long>(tokens) * n_heads * cuts * (2 + vdim)),
                "attention_sink: cut keys need room for their partial results");
  if (n_tiles == 0) return 0;
  if (side_by_side) {
    const long long wgs = static_cast<long long>(tokens) * n_kv_heads * cuts;
    PYLON_REQUIRE(wgs < (1ll << 31), "attention_sink: too many workgroups for one launch");
    const size_t lds_d = sizeof(float) * 4 * group * (2 + vdim);
    const SinkSingle kernel = single_kernel(dim, vdim);
    if (lds_d > 48 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(lds_d));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(wgs)), dim3(256), lds_d, stream, (bf16_t*)out, (const bf16_t*)q,
                       q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_table, table_width, positions,
                       n_heads, n_kv_heads, dim, vdim, page_size, scale, bias, bias != nullptr ? bucket_len : 1, sink, cuts,
                       partial, window, softcap, sink_logit);
    if (cuts > 1) {
      const int items = tokens * n_heads, units = items * ((vdim + 63) / 64);
      hipLaunchKernelGGL(attention_sink_merge_kernel, dim3((units + 3) / 4), dim3(256), 0, stream, (bf16_t*)out,
                         partial, items, cuts, vdim);
    }
    PYLON_LAUNCHED("attention_sink");
  }
  const int waves = 4;
  const int chunks = (group + waves - 1) / waves;
  const long long blocks = static_cast<long long>(n_tiles) * n_kv_heads * chunks * cuts;
  PYLON_REQUIRE(blocks < (1ll << 31), "attention_sink: too many tiles for one launch");
  dim3 grid(static_cast<unsigned>(blocks)), block(2 * 64 * waves);
  const int table_len = bias != nullptr ? bucket_len : 1;
  const size_t lds = prompt_lds(dim, vdim, table_len);
  PYLON_REQUIRE(lds <= 160 * 1024, "attention_sink: the bias table and a block do not fit LDS");
  const SinkPrompt kernel = prompt_kernel(dim, vdim);
  if (lds > 48 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(lds));
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, (bf16_t*)out, (const bf16_t*)q, q_stride, (const bf16_t*)k_cache,
                     (const bf16_t*)v_cache, block_table, table_width, tiles, positions, n_heads, n_kv_heads, dim, vdim,
                     page_size, scale, bias, table_len, sink, cuts, partial, window, softcap, sink_logit);
  if (cuts > 1) {
    const int items = tokens * n_heads, units = items * ((vdim + 63) / 64);
    hipLaunchKernelGGL(attention_sink_merge_kernel, dim3((units + 3) / 4), dim3(256), 0, stream, (bf16_t*)out, partial,
                       items, cuts, vdim);
  }
  PYLON_LAUNCHED("attention_sink");
}
