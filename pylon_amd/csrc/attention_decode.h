// Paged attention for steps with few query tokens (decode): bfloat16, head sizes 64, 128
// and 256, any grouping of up to 16 query heads per key/value head.
//
// A decode step waits on memory latency and, with one wavefront on a SIMD, on the four clocks that every
// instruction takes, more than on bandwidth: the kernel makes few trips to memory and gives the arithmetic
// of a batch of keys to the matrix cores.  One workgroup takes one (token, key/value head) and handles
// all query heads of the group together.  Its wavefronts cut the token's keys into equal
// ranges; a wave issues the loads of up to 64 keys and of their values all at once, then
// computes.  The waves' partial results (running maximum, sum, weighted values, in float)
// meet in LDS and are merged in the order of the ranges, so no partial result ever goes
// through global memory and there is no second kernel.
//
// Few tokens with long contexts would leave most of the chip idle that way.  Then the keys
// of a (token, head) are first cut over several workgroups (gridDim.z); each leaves its
// merged partial result (maximum, sum, unnormalised values, float) in a scratch buffer,
// and a second small kernel merges those in the order of the cuts.
//
// Scores come from the 16x16x32 bf16 matrix instruction with 16 keys as rows and the group's query heads, as often
// as they fit, as columns; every copy then takes the softmax of other tiles.  The weighted sum of values takes
// the probabilities as three bfloat16 parts each (exact for finite values; others are seen in the result).
// Softmax statistics are float throughout.
//
// The kernel can also take over the step that precedes attention: given the raw q/k/v
// projection instead of prepared queries, each workgroup first norms and rotates its
// group's query heads (kept in LDS) and its key head, and stores that key and its value
// head at the token's cache slot.  The loads of older keys do not wait for that: waves without keys of
// their own prepare, and the token's own key is a range of its own.  One launch and one pass over the projection
// less per layer.
//
// Clocks of a workgroup of a 4B layer (8 key/value heads of 128, 4 queries each; 8 tokens of 170 keys), from the
// position's arrival at 1,100 on: loads sent 4,200 (before: 6,450), queries there 4,800 (7,000), scores and
// softmax 6,900 (12,000), weighted values 7,400 (15,200), end 9,200 (19,800).  The launch in a step, us:
// batch 8 of 128 to 192 keys 12.1 -> 6.2, batch 48 of 75 to 175 keys 16.3 -> 10.2, and, without the merge, one request
// of 8,000 keys 13.9 -> 9.2, four of 1,500 to 3,000 15.6 -> 10.8.  Float results against 64 bits are as far off as
// with the values' sum on the vector units (5e-8 to 1e-6, by the scores' size).
#pragma once
#include "common.h"
#include "head_prepare.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

#define AD_MAX_GROUP 16
#define AD_TILE 16   // keys per score tile
#define AD_MAX_WAVES 8
#define AD_LDS_BYTES (160 * 1024)  // of a compute unit

// What the kernel needs to prepare q, k and v itself (PREP): the raw projection
// [tokens, row_stride] with q heads first, then k heads, then v heads.
// With n_parts > 0 the projection comes as that many float partial sums (a product whose K
// was cut over workgroups), part_stride elements apart; the kernel adds them in order and
// rounds the sum to bfloat16 once, which is what a projection stored as bfloat16 holds.
struct DecodePrep {
  const void* qkv;
  long long row_stride;
  int n_parts;
  long long part_stride;
  const float* q_weight;  // per-head RMSNorm weights, or null
  const float* k_weight;
  float eps;
  const float* inv_freq;  // head_dim/2 rotation frequencies, or null
  const int* slot_map;    // cache slot of each token's key and value; null: store nothing
};

// from[i] as a scalar load, whatever else the kernel has read or stored before it: nobody writes it meanwhile.
__device__ __forceinline__ int scalar_int(const int* from, int i) {
  return reinterpret_cast<const __attribute__((address_space(4))) int*>(reinterpret_cast<uintptr_t>(from))[i];
}

// Keys whose loads are in flight together in one wave: 64, or 32 where their values and the accumulators
// would not fit the registers.
static constexpr int decode_super(int head_dim, int gp) {
  return head_dim == 256 || (head_dim == 128 && gp >= 8) ? 32 : 64;
}

// The probabilities of a wave's keys in flight, in three bfloat16 parts (rows part * gp + head), and a row of zeros.
static constexpr int decode_p_row(int head_dim, int gp) { return 2 * decode_super(head_dim, gp) + 16; }  // bytes
static constexpr int decode_p_bytes(int head_dim, int gp) { return (3 * gp + 1) * decode_p_row(head_dim, gp); }

// A wave's part of LDS: its keys, and behind the last of them its partial result; its probabilities.
static constexpr int decode_wave_bytes(int head_dim, int gp) {
  const int keys = decode_super(head_dim, gp) * head_dim * 2, result = gp * head_dim * 4;
  return (keys > result ? keys : result) + decode_p_bytes(head_dim, gp);
}

// Maximum and sum of every range and head; what follows stays 16-byte aligned.
static constexpr int decode_ml_floats(int gp) { return (2 * (AD_MAX_WAVES + 1) * gp + 3) & ~3; }

// The LDS of a workgroup: the waves' parts; every range's maximum and sum per head (one more range: the
// token's own key); with PREP the queries and a rotation table per wave; the own key and value.
static size_t decode_lds_bytes(int key_waves, int n_waves, int gp, int head_dim, bool prep) {
  return static_cast<size_t>(key_waves) * decode_wave_bytes(head_dim, gp) + sizeof(float) * decode_ml_floats(gp) +
         (prep ? 2 * static_cast<size_t>(gp) * head_dim + 4 * static_cast<size_t>(n_waves) * head_dim : 0) + 4 * head_dim;
}

struct DecodeLaunch {
  int group, n_waves, key_shift;  // 1 << key_shift waves share the keys; the others only prepare
  int n_cuts, cut_shift, page_shift;  // the shifts: -1 where the number is no power of two
  int near;  // a cache is at most 4 GB
};

#define AD_LDS(T) __attribute__((address_space(3))) T

// The halves of two registers, or the odd and even rows of 16 lanes, change places: one sum over lanes
// (xor 32, xor 16) of two values in two instructions, each result in half of the lanes.
__device__ __forceinline__ float fold_halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold_rows(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v of the lane BY further on (cyclic) in the same row of 16.
template <int BY>
__device__ __forceinline__ float row_turn(float v) {
  return lanes_turned<0x120 + BY>(v);
}
// Over the 16 lanes of a row, in every lane, by a butterfly (the same bits in all): neighbours, pairs, quads and
// halves change places.
template <typename OP>
__device__ __forceinline__ float over_row(float v, OP op) {
  v = op(v, lanes_turned<0xB1>(v));
  v = op(v, lanes_turned<0x4E>(v));
  v = op(v, lanes_turned<0x141>(v));
  return op(v, lanes_turned<0x140>(v));
}
// Over the lanes of a wave with the same lane % STEP (STEP a power of two of at most 16), in every lane.
template <int STEP, typename OP>
__device__ __forceinline__ float over_columns(float v, OP op) {
  if constexpr (STEP <= 1) v = op(v, row_turn<1>(v));
  if constexpr (STEP <= 2) v = op(v, row_turn<2>(v));
  if constexpr (STEP <= 4) v = op(v, row_turn<4>(v));
  if constexpr (STEP <= 8) v = op(v, row_turn<8>(v));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// EPL = head_dim / 64, GP = heads per group rounded up to 1, 2, 4, 8, 16
// PARTS (with PREP): the projection comes as float partial sums (an instance of its own, so
// that the others keep their registers).
template <int EPL, int GP, bool PREP, bool PARTS = false>
__global__ __launch_bounds__(AD_MAX_WAVES* PYLON_WAVE) void attention_decode_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, uint16_t* k_cache,
    uint16_t* v_cache, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ tok_row, const int* __restrict__ positions, int n_heads, int n_kv_heads,
    int page_size, int window, float scale, DecodeLaunch shape, DecodePrep prep, float* __restrict__ partial) {
  constexpr int HD = EPL * 64, KSTEPS = HD / 32;
  constexpr int SUPER = decode_super(HD, GP), TILES = SUPER / AD_TILE;
  constexpr int LPK = HD / 8;            // lanes that share one key's row, 8 elements each
  constexpr int KPI = PYLON_WAVE / LPK;  // rows a load instruction brings
  constexpr int LOADS = SUPER / KPI;     // of keys, and of values
  static_assert(LOADS % 8 == 0, "eight keys of every lane make an operand");
  constexpr int WAVE_BYTES = decode_wave_bytes(HD, GP), P_ROW = decode_p_row(HD, GP);
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int n_waves = shape.n_waves, group = shape.group, key_waves = 1 << shape.key_shift;
  unsigned char* const own = lds + wave * WAVE_BYTES;  // (of a wave with keys)
  unsigned char* const p_tile = own + WAVE_BYTES - decode_p_bytes(HD, GP);  // [3 GP + 1][P_ROW]
  float* const part_ml = reinterpret_cast<float*>(lds + key_waves * WAVE_BYTES);      // [range][GP][2]
  uint16_t* const kv_new = reinterpret_cast<uint16_t*>(part_ml + decode_ml_floats(GP));  // [2][HD]
  uint16_t* const q_lds = kv_new + 2 * HD;                                                       // [GP][HD], PREP only
  const int col = lane & 15, grp = lane >> 4;
  const int kvh = blockIdx.x, t = blockIdx.y, cut = blockIdx.z;
  // When tok_row is null, token t uses row t of the block table.  Its first 64 entries are
  // then fetched together with the position (one trip to memory instead of two); lane i
  // keeps entry i.
  const int* table = block_table + static_cast<size_t>(tok_row ? tok_row[t] : t) * table_width;
  const int table_entry = table[lane < table_width ? lane : 0];

  // PREP: 512/head_dim heads per wave at a time, the group's query heads into LDS, then this key head and
  // this value head into the token's cache slot.  The last waves take them: those have no keys of
  // their own where a token has few.  Job -> where its head lies in the projection's row (lanes past the
  // last job repeat it).
  constexpr int HPW = KPI, FREQS = (HD / 2 + PYLON_WAVE - 1) / PYLON_WAVE;
  typedef const __attribute__((address_space(1))) float* global_floats;
  const int first_job = (n_waves - 1 - wave) * HPW, j = lane % LPK;
  const int jobs = group + (PREP && prep.slot_map != nullptr ? 2 : 0);
  uintptr_t weights_q = reinterpret_cast<uintptr_t>(prep.q_weight != nullptr ? prep.q_weight : prep.qkv);
  uintptr_t weights_k = reinterpret_cast<uintptr_t>(prep.k_weight != nullptr ? prep.k_weight : prep.qkv);
  // (kept in registers: told where they come from, the compiler fetches them again, by lane)
  if constexpr (PREP) asm volatile("" : "+s"(weights_q), "+s"(weights_k));
  RawHead<PARTS> raw;
  float weight[8], freq[FREQS];
  auto job_of = [&](int h0) __attribute__((always_inline)) { return h0 + lane / LPK < jobs ? h0 + lane / LPK : jobs - 1; };
  auto job_at = [&](int job) __attribute__((always_inline)) {
    const int head = job < group ? kvh * group + job : n_heads + (job == group ? 0 : n_kv_heads) + kvh;
    return static_cast<size_t>(t) * prep.row_stride + static_cast<size_t>(head) * HD + 8 * j;
  };
  // A head's elements and weights are sent for together, without a branch in between (behind one the
  // compiler waits for every load): what is not there is read from the projection instead.
  auto send = [&](int h0) __attribute__((always_inline)) {
    const int job = job_of(h0);
    raw.load(prep.qkv, job_at(job), prep.n_parts, prep.part_stride);
    const bool is_q = job < group, there = (is_q ? prep.q_weight : prep.k_weight) != nullptr;
    const global_floats from = reinterpret_cast<global_floats>(is_q ? weights_q : weights_k) + (there ? 8 * j : 0);
#pragma unroll
    for (int e = 0; e < 8; ++e) weight[e] = from[e];
  };
  if constexpr (PREP) {
    if (first_job < jobs) {  // before anything is known of the position
      const global_floats freqs = reinterpret_cast<global_floats>(
          prep.inv_freq != nullptr ? reinterpret_cast<uintptr_t>(prep.inv_freq) : reinterpret_cast<uintptr_t>(prep.qkv));
#pragma unroll
      for (int i = 0; i < FREQS; ++i)
        freq[i] = freqs[prep.inv_freq != nullptr && lane + i * PYLON_WAVE < HD / 2 ? lane + i * PYLON_WAVE : 0];
      send(first_job);
    }
  }
  const int pos = scalar_int(positions, t);
  // (without a condition, so that it is not waited for before the position is there, too)
  const int slot_there = scalar_int(PREP && prep.slot_map != nullptr ? prep.slot_map : positions, t);
  const int slot = PREP && prep.slot_map != nullptr ? slot_there : -1;

  // The keys of this workgroup (all of them unless they are cut), then of this wave.  The token's own key, the
  // last one, is no part of a wave's range: the cache may not hold it yet.  It is a range of its own.
  const int first = first_visible(pos, window);  // a window, a chunk, or everything
  int per_cut = pos + 1 - first;
  if (shape.n_cuts > 1)
    per_cut = shape.cut_shift >= 0 ? (per_cut + shape.n_cuts - 1) >> shape.cut_shift : (per_cut + shape.n_cuts - 1) / shape.n_cuts;
  per_cut = (per_cut + AD_TILE - 1) / AD_TILE * AD_TILE;
  const int c_begin = first + cut * per_cut;
  const int c_end = c_begin + per_cut < pos ? c_begin + per_cut : pos;
  const bool holds_last = pos >= c_begin && pos < c_begin + per_cut;  // true for exactly one cut
  const int n_keys = c_end > c_begin ? c_end - c_begin : 0;
  // A wave's range is a whole number of the batches it loads at once: with few keys, fewer
  // waves take part, rather than all of them loading a mostly empty batch each.
  int per_wave = (n_keys + key_waves - 1) >> shape.key_shift;
  per_wave = (per_wave + SUPER - 1) / SUPER * SUPER;
  const int k_begin = c_begin + wave * per_wave;
  const int k_end = k_begin + per_wave < c_end ? k_begin + per_wave : c_end;
  const bool has_keys = wave < key_waves && k_begin < k_end;
  // the new key and value are stored by the one workgroup whose keys include them
  const bool stored_new = PREP && slot >= 0 && holds_last;

  auto page_of = [&](int key) __attribute__((always_inline)) { return shape.page_shift >= 0 ? key >> shape.page_shift : key / page_size; };
  auto in_page = [&](int key, int page) __attribute__((always_inline)) { return key - page * page_size; };

  if constexpr (PREP) {
    float* const cs = reinterpret_cast<float*>(q_lds + GP * HD) + wave * HD;
    auto finish = [&](int h0) __attribute__((always_inline)) {
      const int job = job_of(h0);
      float v[8];
      raw.sum(prep.qkv, job_at(job), prep.n_parts, prep.part_stride, v);
      const bool is_q = job < group, is_key = job == group;
      norm_rotate8_with<HD>(v, j, (is_q && prep.q_weight != nullptr) || (is_key && prep.k_weight != nullptr), weight,
                            prep.eps, is_q || is_key, prep.inv_freq != nullptr ? cs : nullptr);
      if (h0 + lane / LPK >= jobs || (!is_q && !stored_new)) return;
      store8_bf16(is_q ? q_lds + job * HD + 8 * j : kv_new + (is_key ? 0 : HD) + 8 * j, v);
      if (!is_q) store8_bf16((is_key ? k_cache : v_cache) + (static_cast<size_t>(slot) * n_kv_heads + kvh) * HD + 8 * j, v);
    };
    if (first_job < jobs) {
      if (prep.inv_freq != nullptr) {
        const float fpos = static_cast<float>(pos);
#pragma unroll
        for (int i = 0; i < FREQS; ++i) {
          const int pair = lane + i * PYLON_WAVE;
          float c, sn;
          sincosf(fpos * freq[i], &sn, &c);
          if (pair < HD / 2) cs[pair] = c, cs[HD / 2 + pair] = sn;
        }
        __builtin_amdgcn_wave_barrier();  // a table of the wave's own: program order suffices
      }
      finish(first_job);
      for (int h0 = first_job + n_waves * HPW; h0 < jobs; h0 += n_waves * HPW) {
        send(h0);
        finish(h0);
      }
    }
  }
  if (holds_last && !stored_new && wave == n_waves - 1) {  // the own key and value from the cache
    const int page = page_of(pos);
    const size_t at = (static_cast<size_t>(table[page]) * page_size + in_page(pos, page)) * n_kv_heads + kvh;
    if (lane < 2 * LPK) {
      const uint16_t* from = (lane < LPK ? k_cache : v_cache) + at * HD + 8 * j;
      *reinterpret_cast<uint4*>(kv_new + 8 * lane) = *reinterpret_cast<const uint4*>(from);
    }
  }

  // A batch of SUPER keys: load i brings, by its lane group g = lane / LPK, the row of key g * LOADS + i (past the
  // end: the last key again), whole rows a load.  (A load in the shape of a matrix operand, 64 bytes of each of 16
  // rows, takes the memory path four times as long.)  Keys go straight into LDS, row i * KPI + g, piece c of 16
  // bytes at place c ^ (i & 7), so that operand reads are free of bank conflicts; values stay in registers.
  const int vkey = lane / LPK;
  uint32_t row_at[LOADS];  // the rows' numbers in the cache
  uint4 vv[LOADS];
  auto own_row = [&](int base, int end) __attribute__((always_inline)) {  // of key base + lane (past the end: of the last)
    const int key = base + lane < end ? base + lane : end - 1, page = page_of(key);
    int page_id = __shfl(table_entry, page & (PYLON_WAVE - 1), PYLON_WAVE);
    if (page_of(end - 1) >= PYLON_WAVE && page >= PYLON_WAVE) page_id = table[page];
    return static_cast<uint32_t>(page_id * page_size + in_page(key, page)) * n_kv_heads + kvh;
  };
  auto find_rows = [&](int base) __attribute__((always_inline)) {
    const uint32_t at = own_row(base, k_end);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) row_at[i] = __shfl(at, vkey * LOADS + i, PYLON_WAVE);
  };
  // The keys' loads go out ahead of the values', and nothing moves across this line or out of this function: the
  // wait for the keys counts on it.  (The caches are no restrict pointers, so that the clobber holds for them.)
  auto send_batch = [&]() __attribute__((always_inline)) {
    auto go = [&](auto&& row) __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)row(k_cache, i, 16 * (j ^ (i & 7))),
                                         (AD_LDS(void)*)(own + i * 1024), 16, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < LOADS; ++i) vv[i] = *reinterpret_cast<const uint4*>(row(v_cache, i, 16 * j));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    if (shape.near)  // 32-bit offsets from one base: an instruction an address instead of four
      go([&](const uint16_t* cache, int i, uint32_t piece) __attribute__((always_inline)) {
        return reinterpret_cast<const unsigned char*>(cache) + static_cast<uint32_t>(row_at[i] * (2u * HD) + piece);
      });
    else
      go([&](const uint16_t* cache, int i, uint32_t piece) __attribute__((always_inline)) {
        return reinterpret_cast<const unsigned char*>(cache) + piece + static_cast<size_t>(row_at[i]) * (2 * HD);
      });
  };

  if (has_keys) {  // on their way while the queries settle in LDS
    find_rows(k_begin);
    send_batch();
  }
  if constexpr (PREP) {
    // Only LDS has to be in order across this barrier (the queries, the new key and value):
    // the loads above and the stores into the cache stay in flight.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  // the token's own key: a range of one key, whose score is its maximum and whose sum is one
  if (holds_last && wave == n_waves - 1) {
    for (int h0 = 0; h0 < group; h0 += HPW) {
      const int h = h0 + lane / LPK < group ? h0 + lane / LPK : group - 1;
      float a[8], b[8], dot = 0.f;
      load8_bf16(PREP ? q_lds + h * HD + 8 * j : q + (static_cast<size_t>(t) * n_heads + kvh * group + h) * HD + 8 * j, a);
      load8_bf16(kv_new + 8 * j, b);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(a[e], b[e], dot);
      dot = head_sum<LPK>(dot);
      if (j == 0) {
        part_ml[2 * (AD_MAX_WAVES * GP + h)] = dot * scale;
        part_ml[2 * (AD_MAX_WAVES * GP + h) + 1] = 1.0f;
      }
    }
  }

  if (has_keys) {
    // query fragments: column `col` is head kvh*group + col % GP of the token (past the group: its first)
    const int head = col % GP;
    bf16x8 qf[KSTEPS];
    {
      const uint16_t* qrow = PREP ? q_lds + (head < group ? head : 0) * HD
                                  : q + (static_cast<size_t>(t) * n_heads + kvh * group + (head < group ? head : 0)) * HD;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(qrow + ks * 32 + grp * 8);
    }
    // Every column of scores is there 16 / GP times: its copies share the tiles, TPL of them each.
    constexpr int TPL = TILES * GP >= 16 ? TILES * GP / 16 : 1, SHARES = TILES / TPL, COPIES = 16 / GP / SHARES;
    const int share = (col / GP) % SHARES;
    float m_run = -INFINITY, l_run = 0.f;  // for head `head`, in every lane of it
    // The weighted values run on the matrix cores, too: a probability is the sum of three bfloat16 numbers to its
    // last bit (24 = 3 x 8), the values are bfloat16, and the products of such numbers are exact in the float sums
    // (of finite values: for others see below).
    // The three parts are rows of one operand: part 4 * (lane group) with up to four heads, which would be alone in
    // 16 rows otherwise; two and three instructions with 8 and 16.  Column n, element 8 g + i of the other operand
    // is a value that lane 16 g + n has loaded itself.  What the lanes of a group hold: with 128 elements one key
    // each; with 256 half of a key (two products, each with zeros for the other half's groups); with 64 two
    // keys (two products, in each of which half of the columns count).
    constexpr int SETS = GP <= 4 ? 1 : 3 * GP <= 32 ? 2 : 3, VARIANTS = HD == 128 ? 1 : 2;
    const unsigned char* p_at[SETS][VARIANTS];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int v = 0; v < VARIANTS; ++v) {
        const int at = 16 * s + col, part = GP <= 4 ? at / 4 : at / GP, h = (GP <= 4 ? at % 4 : at) % GP;
        const bool zeros = part > 2 || (HD == 256 && (grp & 1) != v);
        const int keys = HD == 128 ? grp : HD == 256 ? grp >> 1 : 2 * grp + v;  // the lane group in find_rows' sense
        p_at[s][v] = p_tile + (zeros ? 3 * GP : part * GP + h) * P_ROW + (zeros ? 0 : 2 * LOADS * keys);
      }
    if (lane < P_ROW / 4) reinterpret_cast<uint32_t*>(p_tile + 3 * GP * P_ROW)[lane] = 0;
    floatx4 acc[VARIANTS][8];  // rows 4 grp + r, column col: element 8 n + e (see above)
#pragma unroll
    for (int v = 0; v < VARIANTS; ++v)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int k_row = (col % LOADS) * KPI + col / LOADS;  // of key 16 kt + col: (kt * 16 / LOADS) rows further

    auto batch = [&](int base, auto first_batch) __attribute__((always_inline)) {
      // all loads but the LOADS sent last (the values', or later ones) are through
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
      floatx4 sc[TILES];
#pragma unroll
      for (int kt = 0; kt < TILES; ++kt) sc[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(own + (k_row + kt * (16 / LOADS)) * (HD * 2) +
                                                             ((4 * ks + grp) ^ (col & 7)) * 16);
          sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], sc[kt], 0, 0, 0);
        }
      const bool more = base + SUPER < k_end;
      // lane holds, for its head, the scores of keys base + 16*kt + 4*grp + r
      float x[TPL][4];
#pragma unroll
      for (int u = 0; u < TPL; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = sc[u][r];
#pragma unroll
          for (int w = 1; w < SHARES; ++w) v = share == w ? sc[w * TPL + u][r] : v;
          x[u][r] = v * scale;
        }
      const int key0 = base + 16 * TPL * share + 4 * grp;
      if (!more) {
#pragma unroll
        for (int u = 0; u < TPL; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) x[u][r] = key0 + 16 * u + r < k_end ? x[u][r] : -INFINITY;
      }
      float tile_max = x[0][0];
#pragma unroll
      for (int u = 0; u < TPL; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) tile_max = fmaxf(tile_max, x[u][r]);
      tile_max = over_columns<GP>(tile_max, [](float a, float b) { return fmaxf(a, b); });
      const float m_new = fmaxf(m_run, tile_max);  // finite: key `base` is always live
      float tile_sum = 0.f;
      __builtin_amdgcn_wave_barrier();  // the previous round's reads of p_tile come first
#pragma unroll
      for (int u = 0; u < TPL; ++u) {
        float p[4];
        bf16x4 parts[3];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = expf(x[u][r] - m_new);  // exp(-inf) = 0 for keys past the end
          tile_sum += p[r];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            parts[k][r] = static_cast<__bf16>(p[r]);
            p[r] -= static_cast<float>(parts[k][r]);
          }
          *reinterpret_cast<bf16x4*>(p_tile + (k * GP + head) * P_ROW + 2 * (16 * (TPL * share + u) + 4 * grp)) = parts[k];
        }
      }
      tile_sum = over_columns<GP>(tile_sum, [](float a, float b) { return a + b; }) * (1.0f / COPIES);
      if (!first_batch) {  // rescale what has been accumulated: the factor of head h sits in lane h
        const float corr = expf(m_run - m_new);
        l_run *= corr;
        // (row 4 grp + r is of head r, of head 4 (grp & 1) + r, of head 4 grp + r)
#pragma unroll
        for (int r = 0; r < (GP < 4 ? GP : 4); ++r) {
          const float c = GP <= 4 ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(corr), r))
                                  : __shfl(corr, 4 * (GP == 8 ? grp & 1 : grp) + r, PYLON_WAVE);
#pragma unroll
          for (int v = 0; v < VARIANTS; ++v)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[v][e][r] *= c;
        }
      }
      l_run += tile_sum;
      m_run = m_new;
      __builtin_amdgcn_wave_barrier();  // p_tile is private to the wave: program order suffices
      // keys past the end weigh 0 and their value row is the last key's
#pragma unroll
      for (int a = 0; a < LOADS; a += 8) {
        bf16x8 p[SETS][VARIANTS];
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
          for (int v = 0; v < VARIANTS; ++v) p[s][v] = *reinterpret_cast<const bf16x8*>(p_at[s][v] + 2 * a);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          uint32_t w[4];  // element e of keys a .. a + 7 of the lane's
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t lo[4] = {vv[a + 2 * i].x, vv[a + 2 * i].y, vv[a + 2 * i].z, vv[a + 2 * i].w};
            const uint32_t hi[4] = {vv[a + 2 * i + 1].x, vv[a + 2 * i + 1].y, vv[a + 2 * i + 1].z, vv[a + 2 * i + 1].w};
            w[i] = __builtin_amdgcn_perm(hi[e / 2], lo[e / 2], e % 2 ? 0x07060302u : 0x05040100u);
          }
          const uintx4 packed{w[0], w[1], w[2], w[3]};
          const bf16x8 values = __builtin_bit_cast(bf16x8, packed);
#pragma unroll
          for (int v = 0; v < VARIANTS; ++v)
#pragma unroll
            for (int s = 0; s < SETS; ++s)
              acc[v][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[s][v], values, acc[v][e], 0, 0, 0);
        }
      }
      if (more) {
        find_rows(base + SUPER);
        send_batch();
      }
    };
    // The first batch is code of its own where that is faster: with 128 elements (8 tokens of 170 keys 4.6 us, else
    // 5.0) and where a batch takes few matrix instructions; with 256 elements two copies are up to 7 % slower than one.
    if constexpr (HD == 128 || (HD == 64 ? GP < 16 : GP == 1)) {
      batch(k_begin, std::true_type{});
      for (int base = k_begin + SUPER; base < k_end; base += SUPER) batch(base, std::false_type{});
    } else {
      for (int base = k_begin; base < k_end; base += SUPER) batch(base, base == k_begin);
    }

    // The parts of a row are added over the lane groups that hold them, and what is left is spread over all lanes.
    float* const part_acc = reinterpret_cast<float*>(own);  // [GP][HD]
    __builtin_amdgcn_wave_barrier();  // the last keys have been read
    if constexpr (HD == 64) {  // columns 0 .. 7 of the first product, 8 .. 15 of the second: other keys, the same elements
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float one = col & 8 ? acc[1][e][r] : acc[0][e][r];
          acc[0][e][r] = one + row_turn<8>(one);
        }
    }
#pragma unroll
    for (int v = 0; v < (HD == 256 ? 2 : 1); ++v)
#pragma unroll
      for (int r = 0; r < (GP < 4 ? GP : 4); ++r) {
        float* const row = part_acc + (GP <= 4 ? r : 4 * (GP == 8 ? grp & 1 : grp) + r) * HD + 128 * v + 8 * (HD == 64 ? col & 7 : col);
        float sums[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) sums[e] = acc[v][e][r];
        if constexpr (GP <= 8) {
#pragma unroll
          for (int e = 0; e < 4; ++e) sums[e] = fold_halves(sums[e], sums[e + 4]);  // upper half of the lanes: the upper four
        }
        if constexpr (GP <= 4) {
#pragma unroll
          for (int e = 0; e < 2; ++e) sums[e] = fold_rows(sums[e], sums[e + 2]);  // odd rows of lanes: the upper two of those
          *reinterpret_cast<float2*>(row + 4 * (grp >> 1) + 2 * (grp & 1)) = float2{sums[0], sums[1]};
        } else {
#pragma unroll
          for (int e = 0; e < (GP == 8 ? 4 : 8); e += 4)
            *reinterpret_cast<float4*>(row + e + (GP == 8 ? 4 * (grp >> 1) : 0)) = float4{sums[e], sums[e + 1], sums[e + 2], sums[e + 3]};
        }
      }
    if (lane < GP) *reinterpret_cast<float2*>(part_ml + 2 * (wave * GP + lane)) = float2{m_run, l_run};
  }
  __syncthreads();
  // Wave h merges head h over all ranges, in their order, the own key last.  Lane w (of every row of 16) takes
  // the maximum and the sum of range w, so that all come at once.
  const int ranges = n_keys > 0 ? (n_keys + per_wave - 1) / per_wave : 0;
  const int mine = (lane & 15) < ranges ? lane & 15 : holds_last && (lane & 15) == AD_MAX_WAVES ? AD_MAX_WAVES : -1;
  float beyond = 0.f;  // NaN where a result is no finite number
  auto merge = [&](int h, auto whole) __attribute__((always_inline)) {
    const float2 ml = *reinterpret_cast<const float2*>(part_ml + 2 * ((mine >= 0 ? mine : 0) * GP + h));
    const float m = over_row(mine >= 0 ? ml.x : -INFINITY, [](float a, float b) { return fmaxf(a, b); });
    const float f = mine >= 0 ? expf(ml.x - m) : 0.f;
    const float l = over_row(mine >= 0 ? ml.y * f : 0.f, [](float a, float b) { return a + b; });
    float o[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) o[i] = 0.f;
    if constexpr (decltype(whole)::value) {  // a key a lane for the probabilities, then EPL elements a lane
      const uint16_t* const qrow = PREP ? q_lds + h * HD : q + (static_cast<size_t>(t) * n_heads + kvh * group + h) * HD;
#pragma unroll 1
      for (int base = c_begin; base < c_end; base += PYLON_WAVE) {
        const uint32_t at = own_row(base, c_end);
        float dot = 0.f;
#pragma unroll 1
        for (int c = 0; c < HD; c += 8) {
          float a[8], b[8];
          load8_bf16(qrow + c, a);
          load8_bf16(k_cache + static_cast<size_t>(at) * HD + c, b);
#pragma unroll
          for (int e = 0; e < 8; ++e) dot = fmaf(a[e], b[e], dot);
        }
        const float p = expf(dot * scale - m);
        const int keys = c_end - base < PYLON_WAVE ? c_end - base : PYLON_WAVE;
#pragma unroll 1
        for (int i0 = 0; i0 < keys; i0 += 4) {
          float v[4][EPL];
#pragma unroll
          for (int u = 0; u < 4; ++u) {  // past the last: the last again, unused
            const uint32_t row = __builtin_amdgcn_readlane(at, i0 + u < keys ? i0 + u : keys - 1);
#pragma unroll
            for (int i = 0; i < EPL; ++i) v[u][i] = bf16_bits_to_float(v_cache[static_cast<size_t>(row) * HD + lane * EPL + i]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (i0 + u >= keys) break;
            const float pu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), i0 + u));
#pragma unroll
            for (int i = 0; i < EPL; ++i) o[i] = fmaf(v[u][i], pu, o[i]);
          }
        }
      }
    } else {
      for (int w0 = 0; w0 < ranges; w0 += 4) {
        float a[4][EPL];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float* arow = reinterpret_cast<const float*>(lds + (w0 + w < ranges ? w0 + w : ranges - 1) * WAVE_BYTES) + h * HD;
#pragma unroll
          for (int i = 0; i < EPL; ++i) a[w][i] = arow[lane * EPL + i];
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float fw = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), w0 + w));  // 0 past the last
#pragma unroll
          for (int i = 0; i < EPL; ++i) o[i] = fmaf(a[w][i], fw, o[i]);
        }
      }
    }
    if (holds_last) {
      const float fw = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), AD_MAX_WAVES));
#pragma unroll
      for (int i = 0; i < EPL; ++i) o[i] = fmaf(bf16_bits_to_float(kv_new[HD + lane * EPL + i]), fw, o[i]);
    }
#pragma unroll
    for (int i = 0; i < EPL; ++i) beyond = fmaf(o[i], 0.f, beyond);
    if (shape.n_cuts > 1) {
      // [token][head][cut][HD values, maximum, sum]
      float* prow = partial + ((static_cast<size_t>(t) * n_heads + kvh * group + h) * shape.n_cuts + cut) * (HD + 2);
#pragma unroll
      for (int i = 0; i < EPL; ++i) prow[lane * EPL + i] = o[i];
      if (lane == 0) {
        prow[HD] = m;
        prow[HD + 1] = l;
      }
    } else {
      const float inv = 1.0f / l;
      uint16_t* orow = out + (static_cast<size_t>(t) * n_heads + kvh * group + h) * HD + lane * EPL;
#pragma unroll
      for (int i = 0; i < EPL; ++i) reinterpret_cast<__bf16*>(orow)[i] = static_cast<__bf16>(o[i] * inv);
    }
  };
  for (int h = wave; h < group; h += n_waves) merge(h, std::false_type{});
  // An infinite or NaN value, or a sum beyond float32's range, leaves no finite number above, in other elements, too: a
  // part of its probability may be 0 or negative, and rows of zeros and ranges past the last meet it.  The wave's
  // heads are then merged once more from the keys themselves, with whole probabilities.  (Asked once, behind the
  // stores, it costs nothing: 419 launches of one to 1,024 tokens within 0.1 % on average; asked a head 1.2 %.)
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(beyond != 0.f) != 0, 0)) {
#pragma unroll 1
    for (int h = wave; h < group; h += n_waves) merge(h, std::true_type{});
  }
}

// One wave per (token, query head) merges the partial results of the cuts (at most 64), in
// their order.  Lane c takes the maximum and the sum of cut c, so that all of them come in one
// trip to memory, and so do the weighted values of 32 cuts (eight at a time they were four trips: an 8,000-token
// document and its answer, 12 layers, 56.5 -> 55.6 ms).
template <int EPL>
__global__ __launch_bounds__(PYLON_WAVE) void attention_decode_merge_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ partial, int n_heads, int n_cuts) {
  constexpr int HD = EPL * 64;
  constexpr int BATCH = 8, BATCHES = 32 / BATCH;  // on their way together
  const int lane = threadIdx.x;
  const size_t row = static_cast<size_t>(blockIdx.y) * n_heads + blockIdx.x;
  const float* prow = partial + row * n_cuts * (HD + 2);
  float mc = -INFINITY, lc = 0.f;
  if (lane < n_cuts) {
    mc = prow[lane * (HD + 2) + HD];
    lc = prow[lane * (HD + 2) + HD + 1];
  }
  typedef float lane_part __attribute__((ext_vector_type(EPL < 2 ? 1 : EPL), aligned(4 * (EPL < 2 ? 1 : 2))));
  lane_part v[BATCHES][BATCH];
  auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BATCHES; ++b)
      if (c0 + b * BATCH < n_cuts) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
          const int c = c0 + b * BATCH + u;  // past the end: the last cut again, unused
          v[b][u] = *reinterpret_cast<const lane_part*>(prow + (c < n_cuts ? c : n_cuts - 1) * (HD + 2) + lane * EPL);
        }
      }
  };
  load(0);
  const float m = wave_max(mc);
  const float fc = (lc == 0.f) ? 0.f : expf(mc - m);  // a cut without keys
  const float wc = lc * fc;
  auto of = [](float x, int c) __attribute__((always_inline)) {  // lane c's
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), c & (PYLON_WAVE - 1)));
  };
  float l = 0.f;
  lane_part o = {};
  for (int c0 = 0; c0 < n_cuts; c0 += BATCHES * BATCH) {
#pragma unroll
    for (int b = 0; b < BATCHES; ++b)
      if (c0 + b * BATCH < n_cuts) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
          const int c = c0 + b * BATCH + u;
          const float f = of(fc, c), w = of(wc, c);
          if (c < n_cuts) {
            l += w;
#pragma unroll
            for (int i = 0; i < EPL; ++i) o[i] = fmaf(v[b][u][i], f, o[i]);
          }
        }
      }
    if (c0 + BATCHES * BATCH < n_cuts) load(c0 + BATCHES * BATCH);
  }
  const float inv = 1.0f / l;
  uint16_t* orow = out + row * HD + lane * EPL;
#pragma unroll
  for (int i = 0; i < EPL; ++i) orow[i] = float_to_bf16_bits(o[i] * inv);
}

template <int EPL, bool PREP, bool PARTS = false>
static int launch_decode(void* out, const void* q, void* k_cache, void* v_cache,
                         const int* block_table, int table_width, const int* tok_row,
                         const int* positions, int tokens, int n_heads, int n_kv_heads, int page_size,
                         int window, float scale, int n_waves, DecodePrep prep, int n_cuts, float* partial,
                         long long cache_slots, hipStream_t stream) {
  const int group = n_heads / n_kv_heads;
  const int gp = group <= 1 ? 1 : group <= 2 ? 2 : group <= 4 ? 4 : group <= 8 ? 8 : 16;
  while (n_waves > 1 && decode_lds_bytes(n_waves, AD_MAX_WAVES, gp, EPL * 64, true) > AD_LDS_BYTES) n_waves /= 2;
  DecodeLaunch shape{group, n_waves, 0, n_cuts, -1, -1, cache_slots > 0 && cache_slots * n_kv_heads <= (1ll << 32) / (EPL * 128)};
  while (2 << shape.key_shift <= n_waves) ++shape.key_shift;
  for (int s = 0; s < 31; ++s) {
    if (n_cuts == 1 << s) shape.cut_shift = s;
    if (page_size == 1 << s) shape.page_shift = s;
  }
  if (PREP) {
    // waves of their own for the preparation, where every workgroup has a compute unit to itself
    const int heads = group + (prep.slot_map != nullptr ? 2 : 0), per_wave = 512 / (EPL * 64);
    const int spare = (heads + per_wave - 1) / per_wave;
    if (static_cast<long long>(n_kv_heads) * tokens * n_cuts <= pylon_compute_units())
      shape.n_waves = n_waves + spare < AD_MAX_WAVES ? n_waves + spare : AD_MAX_WAVES;
  }
  const size_t lds = decode_lds_bytes(n_waves, shape.n_waves, gp, EPL * 64, PREP);
  dim3 grid(n_kv_heads, tokens, n_cuts), block(shape.n_waves * PYLON_WAVE);
#define LAUNCH(GP)                                                                                             \
  do {                                                                                                         \
    /* (one value for every launch: a thread must not lower what another has just set) */                      \
    if (lds > 65536)                                                                                           \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_decode_kernel<EPL, GP, PREP, PARTS>), \
                                hipFuncAttributeMaxDynamicSharedMemorySize, AD_LDS_BYTES);                       \
    hipLaunchKernelGGL((attention_decode_kernel<EPL, GP, PREP, PARTS>), grid, block, lds, stream, (uint16_t*)out, \
                       (const uint16_t*)q, (uint16_t*)k_cache, (uint16_t*)v_cache, block_table, table_width, tok_row, \
                       positions, n_heads, n_kv_heads, page_size, window, scale, shape, prep, partial);        \
  } while (0)
  switch (gp) {
    case 1: LAUNCH(1); break;
    case 2: LAUNCH(2); break;
    case 4: LAUNCH(4); break;
    case 8: LAUNCH(8); break;
    default: LAUNCH(16); break;
  }
#undef LAUNCH
  if (n_cuts > 1)
    hipLaunchKernelGGL((attention_decode_merge_kernel<EPL>), dim3(n_heads, tokens), dim3(PYLON_WAVE), 0, stream,
                       (uint16_t*)out, partial, n_heads, n_cuts);
  return 0;
}

// The launches of one head size, by what the kernel starts from (mode 0: prepared queries; 1: the
// raw projection in bfloat16; 2: float partial sums of it).  Each head size is a translation unit
// of its own, so that the many instances compile side by side.
#define AD_MODE_QUERIES 0
#define AD_MODE_PROJECTION 1
#define AD_MODE_PARTIAL_SUMS 2
#define AD_RUN_ARGS                                                                                     \
  int mode, void *out, const void *q, void *k_cache, void *v_cache, const int *block_table, int table_width, \
      const int *tok_row, const int *positions, int tokens, int n_heads, int n_kv_heads, int page_size,    \
      int window, float scale, int n_waves, DecodePrep prep, int n_cuts, float *partial, long long cache_slots, \
      hipStream_t stream
int pylon_decode_run_64(AD_RUN_ARGS);
int pylon_decode_run_128(AD_RUN_ARGS);
int pylon_decode_run_256(AD_RUN_ARGS);

template <int EPL>
static int decode_run(AD_RUN_ARGS) {
  if (mode == AD_MODE_QUERIES)
    return launch_decode<EPL, false>(out, q, k_cache, v_cache, block_table, table_width, tok_row, positions, tokens,
                                     n_heads, n_kv_heads, page_size, window, scale, n_waves, prep, n_cuts, partial,
                                     cache_slots, stream);
  if (mode == AD_MODE_PROJECTION)
    return launch_decode<EPL, true>(out, nullptr, k_cache, v_cache, block_table, table_width, tok_row, positions,
                                    tokens, n_heads, n_kv_heads, page_size, window, scale, n_waves, prep, n_cuts,
                                    partial, cache_slots, stream);
  return launch_decode<EPL, true, true>(out, nullptr, k_cache, v_cache, block_table, table_width, tok_row, positions,
                                        tokens, n_heads, n_kv_heads, page_size, window, scale, n_waves, prep, n_cuts,
                                        partial, cache_slots, stream);
}
