// out[M, N] = x[M, K] * w[N, K]^T in bfloat16 for the many rows of prompt portions, on the matrix
// cores, with the activation of a feed-forward on the float sums before they are rounded: the products
// of a prompt step, bound by the matrix cores where the rows are many and by moving w where they are few.
//
// Four wavefronts a workgroup, two by two, each a quarter of a tile of 64 to 256 rows by 64 to 256
// columns in accumulators.  K is walked in chunks of 64 elements; both operands of a chunk go from
// memory straight into LDS (buffer_load_dwordx4 ... lds: eight whole 128-byte row segments a load;
// segments of 64 bytes, chunks of 32, were a quarter slower).  In LDS piece q of row R (16 bytes)
// lies at place q ^ (R & 7) of its row, so that operand reads are free of bank conflicts.
//
// A chunk is two turns of matrix instructions.  While a turn multiplies, the operands of the next one
// leave LDS and a part of a later chunk's loads is sent, one read or load every few matrix instructions
// (the order is fixed with sched_barrier; with all loads of a chunk sent at once a wave stands for the
// 700 clocks that the loads of four waves take to be accepted).  One barrier a chunk, between its turns,
// behind a counted wait: the next chunk has landed, and nobody reads this one's place any more.
//
// Two ways to lay chunks out in LDS.  STAGES > 0: that many stages of x and w, as many as fit.
// STAGES = 0: three places for x and two for w, two and a half chunks; those of a 256 x 256 tile fill the 160 KB,
// where two stages keep too few bytes in flight for the latency of memory (2048 rows, gate/up 2 x 12288 x 4096:
// 346 -> 307 us).
//
// What bounds it.  A 256 x 256 tile is bound by the matrix cores (2048 x 2 x 12288 x 4096 in 279 us with its activation,
// 1.48 PFLOP/s; with loads and LDS reads left out the loop reaches 1.7).  Smaller tiles are bound by the way from the
// second-level cache into the unit: its first-level cache has some 115 lines of 128 bytes on their way at any time, whatever
// is sent, 200 clocks a line that the second level holds, 1,100 to 1,600 one that it does not (2048 x 2560 x 9728 in 128 x 160
// tiles: 105 us, its loads alone 102, its matrix instructions alone 63, its LDS reads alone 34, its loads from the second
// level 57).  Pulling lines there ahead of their use, by scalar loads or by other waves' loads, does not help; what does is
// a large tile (fewer lines a product), and that the tiles a die has at one time share rows (gw_deep: the same product
// in 111 us with 16 x 2 tiles a die, 101 with 8 x 4).  Hence for a matrix with too few large tiles for the units
// K cut into ranges (pylon_gemm_wide_parts): that product in two ranges of 256 x 160 tiles 82 us.
//
// Which tile: gw_choose, by a model of the launch's rounds over the compute units; a last round that would leave most
// of them idle is a launch of its own (gw_launches).  Gate/up with its activation here, one tile for all (before the
// tiles of 160 and 192 columns and that) -> now, and the library's product alone, us: 2 x 9728 x 2560 at 520, 1000,
// 2048 rows 67, 107, 168 -> 56, 90, 157 (61, 104, 189); 2 x 12288 x 4096 at 1000, 2048, 2096 165, 290, 364 -> 149, 279, 322
// (165, 269, 334); 2 x 25600 x 5120 at 1000, 2048 446, 796 -> 387, 739 (475, 772).  The products without an activation:
// plan.wide_beats_library, plan.portion_beats_library, and pylon_gemm_wide_parts_plan for those into the residual stream.
//
// A kernel's code has to stay small: two compute units share 64 KB of instruction cache.  Results stored with
// an unrolled fallback for odd widths, software rounding and a peeled first chunk (55 to 87 KB of code instead
// of 14 to 37) cost 15 % of a step's launches, though nothing of launches back to back.
#include "common.h"

#include <type_traits>
#include <utility>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

#define GW_LDS(T) __attribute__((address_space(3))) T
#define GW_CHUNK 64
#define GW_ROW_BYTES 128
#define GW_X_PLACES 3  // of tiles that keep two and a half chunks
#define GW_W_PLACES 2

// What happens to the sums: nothing; act(gate) * up of a fused gate/up matrix; max(v, 0)^2.
// The last one is a part's float sums, unrounded.
enum GwEpilogue { GW_PLAIN = 0, GW_SILU = 1, GW_RELU2 = 2, GW_GELU = 3, GW_CAPPED = 4, GW_SUMS = 5 };

// A gate of up to GW_EXACT_ROWS rows is expf and a true division, as in the kernels for fewer rows: up to there
// the activation of a request's tokens has one precision whatever shares its step.  Beyond, where the other
// route (the library's product rounded to bfloat16, then the activation) rounds gate and up by 2^-9 first, it is
// the hardware's exponential and reciprocal, about 2^-22 off: the exact forms make the code of a 128 x 256 tile 46
// KB instead of 19.  (Gate/up of 100 rows, silu, with them and with the hardware's: 4B 46.6 and 45.6 us, 8B 88.7 and
// 87.3, 32B 153.0 and 149.9.)
#define GW_EXACT_ROWS 128
enum GwGate { GW_NO_GATE = 0, GW_FAST_GATE = 1, GW_EXACT_GATE = 2 };

template <int V>
using Int = std::integral_constant<int, V>;
template <typename F, int... I>
__device__ __forceinline__ void gw_for_(F&& f, std::integer_sequence<int, I...>) {
  (f(Int<I>{}), ...);
}
// f(0), f(1), ... f(N - 1) with the number a constant each time.
template <int N, typename F>
__device__ __forceinline__ void gw_for(F&& f) {
  gw_for_(f, std::make_integer_sequence<int, N>{});
}

// All but the N loads sent last have landed, this wave's LDS reads have returned, and every wave is here.
// (A fence would wait for every load, because the loads write LDS.)
template <int N>
__device__ __forceinline__ void gw_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

struct GwShape {
  int M, N, K;
  int m_tiles, n_tiles, deep;  // deep: tile rows that are walked together
  long long ldx, ldw, ldo;
  int up_rows;                 // from a gate row of w to its up row
  int parts;                   // ranges K is cut into, each with float sums of its own, part_apart elements apart
  long long part_apart;
  float alpha, offset, limit;  // of the capped gate
  int epilogue;
};

// z / (1 + exp(-y)); the fast form about one part in 2^22 off.
template <bool EXACT>
__device__ __forceinline__ float gw_gate(float z, float y) {
  if constexpr (EXACT) return z / (1.0f + expf(-y));
  return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * y));
}
template <bool EXACT>
__device__ __forceinline__ float gw_gelu(float z) {  // pylon_gelu_tanh
  return gw_gate<EXACT>(z, 1.5957691216057308f * fmaf(0.044715f * z * z, z, z));
}
template <bool EXACT>
__device__ __forceinline__ float gw_capped(float g, float u, const GwShape& p) {
  if (p.limit > 0.f) {
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
  }
  return gw_gate<EXACT>(g, p.alpha * g) * (u + p.offset);
}

typedef unsigned int gw_u32x4 __attribute__((ext_vector_type(4), aligned(8)));

// Four columns of two tiles in lanes g = lane / 16, columns 4 g of either -> eight columns: of the first tile 0 and 8 in
// the lanes of g = 0 and 2, of the second in those of 1 and 3.
__device__ __forceinline__ gw_u32x4 gw_pair(uint2 lo, uint2 hi) {
  const auto x = __builtin_amdgcn_permlane16_swap(lo.x, hi.x, false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(lo.y, hi.y, false, false);
  return gw_u32x4{x[0], y[0], x[1], y[1]};
}

// MT, NT: tiles of 16 rows and of 16 columns per wave.  With a gate w is a fused matrix of 2 N rows, gate rows
// first; a pair of a wave's column tiles is 16 gate rows and their 16 up rows, N rows further down.
// (The body is a device function: the host pass does not know the descriptor type and would drop a kernel
// that names it, launch stub and all.)
template <int MT, int NT, int STAGES, int GATE>
__device__ __forceinline__ void gemm_wide_body(uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                                               const uint16_t* __restrict__ w, const GwShape p) {
  constexpr bool HALVES = STAGES == 0, GATED = GATE != GW_NO_GATE, EXACT = GATE == GW_EXACT_GATE;
  static_assert(!GATED || NT % 2 == 0, "a gate tile and its up tile belong to one wave");
  constexpr int TM = 32 * MT, TN = 32 * NT;
  constexpr int XL = TM / 32, WL = TN / 32, LOADS = XL + WL;  // loads a wave sends per chunk
  constexpr int STAGE_BYTES = (TM + TN) * GW_ROW_BYTES, X_BYTES = TM * GW_ROW_BYTES, W_BYTES = TN * GW_ROW_BYTES;
  __shared__ __attribute__((aligned(1024))) unsigned char
      lds[HALVES ? GW_X_PLACES * X_BYTES + GW_W_PLACES * W_BYTES : STAGES * STAGE_BYTES];

  // Every eighth workgroup runs on one die: a die gets consecutive tiles of one part, `deep` rows of tiles walked
  // together (gw_deep), so that its cache serves most of what its workgroups read.
  const int tiles = p.m_tiles * p.n_tiles, all = tiles * p.parts, per_die = (all + 7) >> 3;
  int id = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_die || id >= all) return;
  int part = 0;
  if (p.parts > 1) {
    part = id / tiles;
    id -= part * tiles;
  }
  const int deep_tiles = p.deep * p.n_tiles, stripe = id / deep_tiles, within = id - stripe * deep_tiles;
  const int deep = p.m_tiles - stripe * p.deep < p.deep ? p.m_tiles - stripe * p.deep : p.deep;
  const int m0 = (stripe * p.deep + within % deep) * TM, n0 = within / deep * (GATED ? TN / 2 : TN);

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int r = lane & 15, g = lane >> 4, wm = wave & 1, wn = wave >> 1;
  int chunks = p.K / GW_CHUNK, first = 0;
  if (p.parts > 1) {
    first = chunks * part / p.parts;
    chunks = chunks * (part + 1) / p.parts - first;
  }
  const uint16_t* xt = x + static_cast<size_t>(m0) * p.ldx + first * GW_CHUNK;
  const uint16_t* wt = w + static_cast<size_t>(n0) * p.ldw + first * GW_CHUNK;

  // Load i of wave v brings rows 8 (v XL + i) .. + 7 of the tile.  Rows beyond M or N are read as the last
  // one (their results go nowhere).
  unsigned x_at[XL], w_at[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = 8 * (wave * XL + i) + (lane >> 3);
    const int at = m0 + row < p.M ? row : p.M - 1 - m0;
    x_at[i] = static_cast<unsigned>(at) * static_cast<unsigned>(p.ldx) * 2u + ((lane & 7) ^ (row & 7)) * 16;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int row = 8 * (wave * WL + i) + (lane >> 3);
    int at = GATED ? (row >> 5) * 16 + (row & 15) : row;
    at = n0 + at < p.N ? at : p.N - 1 - n0;
    if (GATED && (row & 16)) at += p.up_rows;
    w_at[i] = static_cast<unsigned>(at) * static_cast<unsigned>(p.ldw) * 2u + ((lane & 7) ^ (row & 7)) * 16;
  }
  // Beyond K the descriptor spans nothing and the chunk's offset is zero: the load fetches nothing, whether or
  // not the range check counts the scalar offset, and every count of loads stays exact.
  auto rows_of = [&](bool is_x, int chunk) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(is_x ? xt : wt), 0, chunk < chunks ? 0x7fffffff : 0,
                                             0x00020000);
  };
  auto load = [&](__amdgpu_buffer_rsrc_t rows, bool is_x, int chunk, int base, int i) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (GW_LDS(void)*)(lds + base + (wave * (is_x ? XL : WL) + i) * 1024), 16, is_x ? x_at[i] : w_at[i],
        chunk < chunks ? chunk * GW_ROW_BYTES : 0, 0, 0);
  };

  // Operands: lane (r, g) takes piece 4 s + g of row r of a tile for turn s.
  unsigned piece_at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) piece_at[s] = r * GW_ROW_BYTES + ((4 * s + g) ^ (r & 7)) * 16;
  bf16x8 xf[2][MT], wf[2][NT];
  constexpr int READS = MT + NT;
  auto read = [&](int s, int x_base, int w_base, int q) __attribute__((always_inline)) {
    if (q < NT)
      wf[s][q] = *reinterpret_cast<const GW_LDS(bf16x8)*>((const GW_LDS(unsigned char)*)lds + w_base +
                                                          (wn * NT + q) * 2048 + piece_at[s]);
    else
      xf[s][q - NT] = *reinterpret_cast<const GW_LDS(bf16x8)*>((const GW_LDS(unsigned char)*)lds + x_base +
                                                               (wm * MT + q - NT) * 2048 + piece_at[s]);
  };

  constexpr int PRODUCTS = MT * NT;  // of a turn
  floatx4 acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      // zeros of its own: told that all accumulators start as one value, the compiler moves them about in the loop
      if constexpr (PRODUCTS >= 64)
        asm volatile("" : "+a"(acc[j][t]));
      else
        asm volatile("" : "+v"(acc[j][t]));
    }

  // Turn S: its products; between them the reads of the other turn's operands and `send(Int<i>)` for
  // i = 0 .. SENDS - 1, spread over the first SPREAD products.
  auto turn = [&](auto S, int x_base, int w_base, auto SENDS, auto SPREAD, auto send) __attribute__((always_inline)) {
    constexpr int s = decltype(S)::value, sends = decltype(SENDS)::value, spread = decltype(SPREAD)::value;
    static_assert(sends <= spread, "at most one load a product");
    __builtin_amdgcn_sched_barrier(0);
    gw_for<PRODUCTS>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      constexpr int q = (i * READS + PRODUCTS - 1) / PRODUCTS;  // the read that falls due here, if one does
      if constexpr (q < READS && q * PRODUCTS / READS == i) read(s ^ 1, x_base, w_base, q);
      if constexpr (sends > 0) {
        constexpr int l = (i * sends + spread - 1) / spread;
        if constexpr (l < sends && l * spread / sends == i) send(Int<l>{});
      }
      acc[i / MT][i % MT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s][i / MT], xf[s][i % MT], acc[i / MT][i % MT], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  if constexpr (HALVES) {
    // x has three places, w two.  In flight besides the chunk in use: the next one and x of the one after it.
    constexpr int W_AT = GW_X_PLACES * X_BYTES;
    auto whole = [&](bool is_x, int chunk, int at) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rows = rows_of(is_x, chunk);
#pragma unroll
      for (int i = 0; i < (is_x ? XL : WL); ++i) load(rows, is_x, chunk, at, i);
    };
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      whole(true, c, c * X_BYTES);
      whole(false, c, W_AT + c * W_BYTES);
    }
    gw_sync<LOADS>();
#pragma unroll
    for (int q = 0; q < READS; ++q) read(0, 0, W_AT, q);
    int x_now = 0, w_now = W_AT;  // of the chunk in use
    for (int c = 0; c < chunks; ++c) {
      const int x_next = x_now == 2 * X_BYTES ? 0 : x_now + X_BYTES, x_then = x_next == 2 * X_BYTES ? 0 : x_next + X_BYTES;
      const int w_next = 2 * W_AT + W_BYTES - w_now;
      const __amdgpu_buffer_rsrc_t xr = rows_of(true, c + 2), wr = rows_of(false, c + 2);
      turn(Int<0>{}, x_now, w_now, Int<XL>{}, Int<PRODUCTS>{},
           [&](auto I) __attribute__((always_inline)) { load(xr, true, c + 2, x_then, decltype(I)::value); });
      gw_sync<XL>();  // all of the next chunk; x of the one after it is on its way
      turn(Int<1>{}, x_next, w_next, Int<WL>{}, Int<PRODUCTS / 2>{},
           [&](auto I) __attribute__((always_inline)) { load(wr, false, c + 2, w_now, decltype(I)::value); });
      x_now = x_next, w_now = w_next;
    }
  } else {
    constexpr int HALF = (LOADS + 1) / 2;  // of a chunk's loads, sent per turn
    auto load_one = [&](__amdgpu_buffer_rsrc_t xr, __amdgpu_buffer_rsrc_t wr, int chunk, int stage, int i)
                        __attribute__((always_inline)) {
      if (i < XL)
        load(xr, true, chunk, stage * STAGE_BYTES, i);
      else
        load(wr, false, chunk, stage * STAGE_BYTES + TM * GW_ROW_BYTES, i - XL);
    };
#pragma unroll
    for (int c = 0; c < STAGES; ++c) {
      const __amdgpu_buffer_rsrc_t xr = rows_of(true, c), wr = rows_of(false, c);
#pragma unroll
      for (int i = 0; i < (c + 1 < STAGES ? LOADS : HALF); ++i) load_one(xr, wr, c, c, i);
    }
    gw_sync<(STAGES - 2) * LOADS + HALF>();
#pragma unroll
    for (int q = 0; q < READS; ++q) read(0, 0, TM * GW_ROW_BYTES, q);
    int stage = 0;
    // Chunk c + STAGES goes to the place of chunk c: half of its loads in c's second turn, the others in the
    // first turn of c + 1.
    for (int c = 0; c < chunks; ++c) {
      const int next = stage + 1 == STAGES ? 0 : stage + 1, before = stage == 0 ? STAGES - 1 : stage - 1;
      const int base = stage * STAGE_BYTES, next_base = next * STAGE_BYTES;
      {
        const __amdgpu_buffer_rsrc_t xr = rows_of(true, c - 1 + STAGES), wr = rows_of(false, c - 1 + STAGES);
        turn(Int<0>{}, base, base + TM * GW_ROW_BYTES, Int<LOADS - HALF>{}, Int<PRODUCTS>{},
             [&](auto I) __attribute__((always_inline)) { load_one(xr, wr, c - 1 + STAGES, before, HALF + decltype(I)::value); });
      }
      gw_sync<(STAGES - 2) * LOADS>();
      const __amdgpu_buffer_rsrc_t xr = rows_of(true, c + STAGES), wr = rows_of(false, c + STAGES);
      turn(Int<1>{}, next_base, next_base + TM * GW_ROW_BYTES, Int<HALF>{}, Int<PRODUCTS>{},
           [&](auto I) __attribute__((always_inline)) { load_one(xr, wr, c + STAGES, stage, decltype(I)::value); });
      stage = next;
    }
  }
  // Loads beyond K fetch nothing but do write (zeros) into LDS: the wave sees them through before it leaves.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");

  if constexpr (!GATED) {
    if (p.epilogue == GW_SUMS) {
      float* const base = reinterpret_cast<float*>(out) + part * p.part_apart +
                          static_cast<size_t>(m0 + wm * MT * 16 + r) * p.ldo + n0 + wn * NT * 16 + 4 * g;
      const int rows = p.M - (m0 + wm * MT * 16 + r), cols = p.N - (n0 + wn * NT * 16 + 4 * g);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if (16 * t >= rows) break;
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (16 * j < cols) *reinterpret_cast<floatx4*>(base + static_cast<size_t>(16 * t) * p.ldo + 16 * j) = acc[j][t];
      }
      return;
    }
  }
  // acc[j][t][i] is out[16 t + r][16 j + 4 g + i] of the wave's quarter (a pair of column tiles with GATED).  Of two
  // neighbouring tiles the lanes of g = 0 and 1, and of 2 and 3, swap halves: a lane then has eight columns of one of
  // them, and a store 64 bytes of each of 16 rows instead of 32 (gw_pair; 2048 x 16384 x 4096 205 -> 196 us, 2048 x 6144 x
  // 2560 53 -> 50, 2048 x 2 x 12288 x 4096 with its gate 290 -> 279; nothing stored at all 182, 45, 273).
  // N is a multiple of four: of a lane's eight values all, the first four or none lie within.
  auto store = [&](auto value) __attribute__((always_inline)) {
    constexpr int OT = GATED ? NT / 2 : NT, PAIRS = OT / 2;  // tiles of the result
    const int row0 = m0 + wm * MT * 16 + r, col0 = n0 + wn * OT * 16;
    uint16_t* const base = out + static_cast<size_t>(row0) * p.ldo + col0;
    const int rows = p.M - row0, cols = p.N - col0, eight = (g & 1) * 16 + (g >> 1) * 8;
    auto four = [&](int j, int t) __attribute__((always_inline)) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = static_cast<__bf16>(GATED ? value(acc[2 * j % NT][t][i], acc[(2 * j + 1) % NT][t][i]) : value(acc[j][t][i], 0.f));
      return __builtin_bit_cast(uint2, v);
    };
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if (16 * t >= rows) break;
      uint16_t* const row = base + static_cast<size_t>(16 * t) * p.ldo;
#pragma unroll
      for (int j = 0; j < PAIRS; ++j) {
        const uint2 lo = four(2 * j, t), hi = four(2 * j + 1, t);
        const gw_u32x4 v = gw_pair(lo, hi);
        const int at = 32 * j + eight;
        if (at + 8 <= cols)
          *reinterpret_cast<gw_u32x4*>(row + at) = v;
        else if (at < cols)
          *reinterpret_cast<uint2*>(row + at) = uint2{v[0], v[1]};
      }
      if constexpr (OT % 2 == 1) {
        const int at = 16 * (OT - 1) + 4 * g;
        if (at < cols) *reinterpret_cast<uint2*>(row + at) = four(OT - 1, t);
      }
    }
  };
  if constexpr (GATED) {
    if (p.epilogue == GW_SILU)
      store([&](float gate, float up) __attribute__((always_inline)) { return gw_gate<EXACT>(gate, gate) * up; });
    else if (p.epilogue == GW_GELU)
      store([&](float gate, float up) __attribute__((always_inline)) { return gw_gelu<EXACT>(gate) * up; });
    else
      store([&](float gate, float up) __attribute__((always_inline)) { return gw_capped<EXACT>(gate, up, p); });
  } else if (p.epilogue == GW_RELU2) {
    store([](float v, float) __attribute__((always_inline)) {
      const float pos = fmaxf(v, 0.f);
      return pos * pos;
    });
  } else {
    store([](float v, float) __attribute__((always_inline)) { return v; });
  }
}

// Two workgroups to a compute unit where their LDS fits.
template <int MT, int NT, int STAGES>
constexpr int gw_per_unit() {
  const int bytes = 32 * (STAGES == 0 ? GW_X_PLACES * MT + GW_W_PLACES * NT : STAGES * (MT + NT)) * GW_ROW_BYTES;
  return 2 * bytes <= 160 * 1024 ? 2 : 1;
}

template <int MT, int NT, int STAGES, int GATE>
__global__ __launch_bounds__(256, (gw_per_unit<MT, NT, STAGES>())) void gemm_wide_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const GwShape p) {
  gemm_wide_body<MT, NT, STAGES, GATE>(out, x, w, p);
}

// The tiles (the sums depend on none): rows, columns, workgroups per compute unit, and what a chunk of 64 of K costs a workgroup in
// nanoseconds where the launch's last round leaves it alone on its unit (for one workgroup a unit: leaves
// units idle) and in full rounds (measured over the layer sizes of 4B to 32B, each launch behind 256 MB of
// other traffic, as in a step: launched back to back the small tiles look a third faster than they are).
struct GwTile {
  int rows, cols, per_unit, alone_ns, full_ns;
};
static const GwTile kTiles[] = {
    {64, 64, 2, 230, 450},      // 2 x 2, five stages
    {128, 128, 1, 560, 575},    // 4 x 4, four stages
    {128, 128, 2, 700, 930},    // 4 x 4, two and a half chunks
    {128, 192, 1, 660, 670},    // 4 x 6, three stages
    {128, 192, 2, 850, 1330},   // 4 x 6, two stages
    {96, 256, 1, 740, 750},     // 3 x 8, three stages
    {256, 128, 1, 855, 855},    // 8 x 4, three stages
    {128, 256, 1, 860, 870},    // 4 x 8, three stages
    {160, 256, 1, 940, 990},    // 5 x 8, three stages
    {256, 256, 1, 1300, 1380},  // 8 x 8, two and a half chunks
    {128, 160, 1, 600, 615},    // 4 x 5, four stages; none of the next two with a gate, whose halves share a wave
    {256, 160, 1, 940, 950},    // 8 x 5, three stages
    {256, 192, 1, 1055, 1075},  // 8 x 6, two and a half chunks
    {192, 256, 1, 1080, 1100},  // 6 x 8, two and a half chunks
};
#define GW_ROUND_US 3.5  // of a round: the first chunks' way to LDS, and the results' way out
static const int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);

// What a full round costs the smallest tile, which asks most of the way to the second-level caches, where these hold
// w (nanoseconds a chunk, and the most bytes): 1,024 to 4,096 x 1,024 to 3,072 210 to 320 at 300 to 2,000 rows, 4,096 x 2,048 270 to 430,
// from 2,560 x 4,096 on 400 to 490.
#define GW_NEAR_NS 380
#define GW_NEAR_BYTES 18000000

// A float result of a part leaves late: its bytes, in us a MB.
#define GW_STORE_US_MB 0.27

static double gw_time_us(const GwTile& t, int M, int N, int K, bool gated, int units, int parts = 1) {
  const int cols = gated ? t.cols / 2 : t.cols;
  const long long tiles = static_cast<long long>((M + t.rows - 1) / t.rows) * ((N + cols - 1) / cols) * parts;
  const long long slots = static_cast<long long>(units) * t.per_unit;
  const long long rounds = tiles / slots, left = tiles - rounds * slots;
  const double chunks = 1e-3 * (K / GW_CHUNK) / parts;
  const bool near = t.rows == 64 && (gated ? 4ll : 2ll) * N * K <= GW_NEAR_BYTES;
  const int full_ns = near ? GW_NEAR_NS : t.full_ns;
  const double last = left == 0 ? 0.0 : chunks * (left <= units ? t.alone_ns : full_ns) + GW_ROUND_US;
  const double stored = parts == 1 ? 0.0 : GW_STORE_US_MB * 4e-6 * parts * M * N / (rounds + (left > 0));
  return rounds * (chunks * full_ns + GW_ROUND_US) + last + stored;
}

static bool gw_takes(const GwTile& t, int M, bool gated) {
  return !gated || (t.cols % 64 == 0 && (M > GW_EXACT_ROWS || t.rows <= GW_EXACT_ROWS));
}

static int gw_choose(int M, int N, int K, bool gated, int units, double* us = nullptr) {
  int best = 0;
  double least = 1e30;
  for (int i = 0; i < kTileCount; ++i) {
    if (!gw_takes(kTiles[i], M, gated)) continue;
    const double now = gw_time_us(kTiles[i], M, N, K, gated, units);
    if (now < least) least = now, best = i;
  }
  if (us) *us = least;
  return best;
}

// How a product is launched: the first `ahead` columns in a launch of tile `first` (0: no such launch), the others in one of
// tile `rest`; us: by the model.
struct GwLaunches {
  int ahead, first, rest;
  double us;
};

// One launch, or, where a last round would leave most units idle, the whole rounds of one tile in a launch of their own
// and the columns that are left in a launch of the tile that suits them, where both take 2 % less than one.  (Measured, 183 products
// that the model would split: where it gives less than 2 %, two launches take 1.006 of the time of one, where it gives 2 to 10 %
// 0.98, beyond 0.91.)
#define GW_SECOND_US 2.5
#define GW_SECOND_SHARE 0.98
static GwLaunches gw_launches(int M, int N, int K, bool gated, int units) {
  GwLaunches best{0, -1, 0, 0.0};
  best.rest = gw_choose(M, N, K, gated, units, &best.us);
  if (M <= 4 * GW_EXACT_ROWS) return best;
  double least = GW_SECOND_SHARE * best.us;
  for (int i = 0; i < kTileCount; ++i) {
    const GwTile& t = kTiles[i];
    if (!gw_takes(t, M, gated)) continue;
    const int cols = gated ? t.cols / 2 : t.cols, m_tiles = (M + t.rows - 1) / t.rows;
    const long long slots = static_cast<long long>(units) * t.per_unit;
    const long long rounds = static_cast<long long>(m_tiles) * (N / cols) / slots;
    const long long n = rounds * slots / m_tiles * cols;
    if (rounds == 0 || n >= N) continue;
    const double whole = gw_time_us(t, M, static_cast<int>(n), K, gated, units) + GW_SECOND_US;
    if (whole >= least) continue;  // what is left takes some time too
    double left;
    const int rest = gw_choose(M, N - static_cast<int>(n), K, gated, units, &left);
    if (whole + left < least) least = whole + left, best = GwLaunches{static_cast<int>(n), i, rest, least};
  }
  return best;
}

// The tile that suits a product of these sizes best in one launch (units 0: the current device's), and in *us the time that
// the model gives it; pylon_gemm_wide_launches says whether there are two.  Touches no device memory.
extern "C" int pylon_gemm_wide_plan(int M, int N, int K, int gated, int units, int* tile, float* us) {
  PYLON_REQUIRE(tile != nullptr && us != nullptr && M >= 1 && N >= 1 && K >= GW_CHUNK, "gemm_wide_plan: bad arguments");
  if (units <= 0) units = pylon_compute_units();
  PYLON_REQUIRE(units > 0, "gemm_wide_plan: no device to take the number of compute units from");
  double least;
  *tile = gw_choose(M, N, K, gated != 0, units, &least);
  *us = static_cast<float>(least);
  return 0;
}

// The launches of pylon_gemm_wide for a product of these sizes: columns of the first of two (0: there is one), its tile, the
// tile of the other columns, and the time that the model gives them.  Touches no device memory.
extern "C" int pylon_gemm_wide_launches(int M, int N, int K, int gated, int units, int* ahead, int* first, int* rest, float* us) {
  PYLON_REQUIRE(ahead && first && rest && us && M >= 1 && N >= 1 && K >= GW_CHUNK, "gemm_wide_launches: bad arguments");
  if (units <= 0) units = pylon_compute_units();
  PYLON_REQUIRE(units > 0, "gemm_wide_launches: no device to take the number of compute units from");
  const GwLaunches found = gw_launches(M, N, K, gated != 0, units);
  *ahead = found.ahead, *first = found.first, *rest = found.rest, *us = static_cast<float>(found.us);
  return 0;
}

// Ranges of K for a product into the residual stream, with the tile, or one range and tile -1 (pylon_gemm_wide): the
// quickest with what the residual norm pays for reading float sums of every range instead of one bfloat16 result, by
// their size.  Product and norm over 1,096 sizes of 1,024 to 5,120 columns, K of 1,024 to 25,600 and 129 to 2,111 rows take 0.81 of the
// time of the uncut kernel or the library, whichever it was before (1.03 to 1.06 in ten of them); with 380 ns for
// every full round of the smallest tile 4096 x 4096 at 435 and 512 rows and 2560 x 4096 at 768 took 39, 40 and 37 us against
// 34, 37 and 35, where two ranges take 29, 32 and 30.
#define GW_ADD_US_MB 0.2
#define GW_MOST_PARTS 4
#define GW_LEAST_CHUNKS 8  // of a range
extern "C" int pylon_gemm_wide_parts_plan(int M, int N, int K, int units, int* parts, int* tile, float* us) {
  PYLON_REQUIRE(parts && tile && us && M >= 1 && N >= 1 && K >= GW_CHUNK, "gemm_wide_parts_plan: bad arguments");
  if (units <= 0) units = pylon_compute_units();
  PYLON_REQUIRE(units > 0, "gemm_wide_parts_plan: no device to take the number of compute units from");
  double least = gw_launches(M, N, K, false, units).us;
  *parts = 1, *tile = -1;
  for (int n = 2; n <= GW_MOST_PARTS && n * GW_LEAST_CHUNKS <= K / GW_CHUNK; ++n)
    for (int i = 0; i < kTileCount; ++i) {
      const double now = gw_time_us(kTiles[i], M, N, K, false, units, n) + GW_ADD_US_MB * 1e-6 * (4 * n - 2) * M * N;
      if (now < least) least = now, *parts = n, *tile = i;
    }
  *us = static_cast<float>(least);
  return 0;
}

// Rows of tiles that a die walks together, of stripes of one depth: those with which the tiles that its units hold at
// one time need the fewest rows of x and w.
static int gw_deep(int m_tiles, int n_tiles, int rows, int cols, int held) {
  int best = 1;
  long long least = -1;
  for (int stripes = 1; stripes <= m_tiles; ++stripes) {
    const int deep = (m_tiles + stripes - 1) / stripes, down = deep < held ? deep : held;
    const long long across = held <= deep ? 16 : 16ll * held / deep;  // sixteenths of a tile
    const long long need = 16ll * down * rows + (across < 16ll * n_tiles ? across : 16ll * n_tiles) * cols;
    if (least < 0 || need < least) least = need, best = deep;
  }
  return best;
}

template <int MT, int NT, int STAGES>
static void launch_wide(void* out, const void* x, const void* w, GwShape p, hipStream_t stream) {
  const bool gated = p.epilogue != GW_PLAIN && p.epilogue != GW_RELU2 && p.epilogue != GW_SUMS;
  const int cols = gated ? 16 * NT : 32 * NT;
  p.m_tiles = (p.M + 32 * MT - 1) / (32 * MT), p.n_tiles = (p.N + cols - 1) / cols;
  p.deep = gw_deep(p.m_tiles, p.n_tiles, 32 * MT, 32 * NT, 32 * gw_per_unit<MT, NT, STAGES>());
  const dim3 grid((static_cast<unsigned>(p.m_tiles) * p.n_tiles * p.parts + 7) / 8 * 8), block(256);
#define GO(GATE)                                                                                                     \
  hipLaunchKernelGGL((gemm_wide_kernel<MT, NT, STAGES, GATE>), grid, block, 0, stream, (uint16_t*)out, (const uint16_t*)x, \
                     (const uint16_t*)w, p)
  if (!gated) {
    GO(GW_NO_GATE);
    return;
  }
  if constexpr (NT % 2 == 0) {
    if constexpr (32 * MT <= GW_EXACT_ROWS) {
      if (p.M <= GW_EXACT_ROWS) {
        GO(GW_EXACT_GATE);
        return;
      }
    }
    GO(GW_FAST_GATE);
  }
#undef GO
}

static void gw_launch(int tile, void* out, const void* x, const void* w, const GwShape& p, hipStream_t stream) {
  switch (tile) {
    case 0: launch_wide<2, 2, 5>(out, x, w, p, stream); break;
    case 1: launch_wide<4, 4, 4>(out, x, w, p, stream); break;
    case 2: launch_wide<4, 4, 0>(out, x, w, p, stream); break;
    case 3: launch_wide<4, 6, 3>(out, x, w, p, stream); break;
    case 4: launch_wide<4, 6, 2>(out, x, w, p, stream); break;
    case 5: launch_wide<3, 8, 3>(out, x, w, p, stream); break;
    case 6: launch_wide<8, 4, 3>(out, x, w, p, stream); break;
    case 7: launch_wide<4, 8, 3>(out, x, w, p, stream); break;
    case 8: launch_wide<5, 8, 3>(out, x, w, p, stream); break;
    case 9: launch_wide<8, 8, 0>(out, x, w, p, stream); break;
    case 10: launch_wide<4, 5, 4>(out, x, w, p, stream); break;
    case 11: launch_wide<8, 5, 3>(out, x, w, p, stream); break;
    case 12: launch_wide<8, 6, 0>(out, x, w, p, stream); break;
    default: launch_wide<6, 8, 0>(out, x, w, p, stream); break;
  }
}

// x: [M, ldx] bf16; w: [N, ldw] bf16, or with a gate [2 N, ldw], gate rows first; out: [M, ldo] bf16, rounded
// once.  epilogue: GwEpilogue; alpha, offset, limit: of the capped gate, min(g, limit) sigmoid(alpha g) times
// clamp(u, -limit, limit) + offset (limit <= 0: no caps).  tile: an index of kTiles, or -1 for the rule; the
// sums do not depend on it.
extern "C" int pylon_gemm_wide(void* out, const void* x, const void* w, int M, int N, int K, long long ldx, long long ldw,
                               long long ldo, int epilogue, float alpha, float offset, float limit, int tile,
                               hipStream_t stream) {
  PYLON_REQUIRE(epilogue >= GW_PLAIN && epilogue <= GW_CAPPED, "gemm_wide: unknown epilogue %d", epilogue);
  PYLON_REQUIRE(M >= 0 && N > 0 && K > 0 && K % GW_CHUNK == 0, "gemm_wide: bad sizes M=%d N=%d K=%d (K a multiple of %d)",
                M, N, K, GW_CHUNK);
  PYLON_REQUIRE(ldx >= K && ldw >= K && ldo >= N && ldx % 8 == 0 && ldw % 8 == 0, "gemm_wide: bad row strides");
  PYLON_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                "gemm_wide: operands must be 16-byte aligned");
  const bool gated = epilogue != GW_PLAIN && epilogue != GW_RELU2;
  PYLON_REQUIRE(ldx * 512 < (1ll << 31) && (static_cast<long long>(gated ? N : 0) + 256) * ldw * 2 < (1ll << 31),
                "gemm_wide: the rows of a tile are beyond the 2 GB that one view of them may span");
  PYLON_REQUIRE(N % 4 == 0 && ldo % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
                "gemm_wide: rows of the result are multiples of 4 elements at 8-byte aligned addresses");
  PYLON_REQUIRE(tile >= -1 && tile < kTileCount, "gemm_wide: there is no tile %d", tile);
  PYLON_REQUIRE(tile < 0 || gw_takes(kTiles[tile], M, gated),
                "gemm_wide: a gate takes no tile of %d columns, and up to %d rows one of up to as many rows", kTiles[tile].cols,
                GW_EXACT_ROWS);
  PYLON_REQUIRE(static_cast<long long>((M + 63) / 64) * ((N + 31) / 32) < (1ll << 30), "gemm_wide: too many tiles for one launch");
  if (M == 0) return 0;
  int ahead = 0;
  if (tile < 0) {
    const int units = pylon_compute_units();
    PYLON_REQUIRE(units > 0, "gemm_wide: the device's number of compute units is unknown");
    const GwLaunches found = gw_launches(M, N, K, gated, units);
    ahead = found.ahead, tile = found.rest;
    if (ahead > 0)
      gw_launch(found.first, out, x, w, GwShape{M, ahead, K, 0, 0, 0, ldx, ldw, ldo, N, 1, 0, alpha, offset, limit, epilogue}, stream);
  }
  gw_launch(tile, static_cast<uint16_t*>(out) + ahead, x, static_cast<const uint16_t*>(w) + ahead * ldw,
            GwShape{M, N - ahead, K, 0, 0, 0, ldx, ldw, ldo, N, 1, 0, alpha, offset, limit, epilogue}, stream);
  PYLON_LAUNCHED("gemm_wide");
}

// Float sums of `parts` ranges of K, each of them unrounded, for a consumer to add in order: out [parts][M][N] float.
// tile: as pylon_gemm_wide_parts_plan says; -1 with one part for the rule of pylon_gemm_wide.
extern "C" int pylon_gemm_wide_parts(float* out, const void* x, const void* w, int M, int N, int K, long long ldx,
                                     long long ldw, int parts, int tile, hipStream_t stream) {
  PYLON_REQUIRE(M >= 0 && N > 0 && K > 0 && K % GW_CHUNK == 0 && N % 4 == 0, "gemm_wide_parts: bad sizes M=%d N=%d K=%d", M, N, K);
  PYLON_REQUIRE(parts >= 1 && parts <= 8 && parts <= K / GW_CHUNK, "gemm_wide_parts: cannot cut %d into %d parts", K, parts);
  PYLON_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0, "gemm_wide_parts: bad row strides");
  PYLON_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 15) == 0, "gemm_wide_parts: operands must be 16-byte aligned");
  PYLON_REQUIRE(ldx * 512 < (1ll << 31) && 256 * ldw * 2 < (1ll << 31),
                "gemm_wide_parts: the rows of a tile are beyond the 2 GB that one view of them may span");
  PYLON_REQUIRE(tile >= (parts == 1 ? -1 : 0) && tile < kTileCount, "gemm_wide_parts: there is no tile %d", tile);
  PYLON_REQUIRE(static_cast<long long>((M + 63) / 64) * ((N + 31) / 32) < (1ll << 27), "gemm_wide_parts: too many tiles for one launch");
  if (M == 0) return 0;
  if (tile < 0) {
    const int units = pylon_compute_units();
    PYLON_REQUIRE(units > 0, "gemm_wide_parts: the device's number of compute units is unknown");
    tile = gw_choose(M, N, K, false, units);
  }
  gw_launch(tile, out, x, w,
            GwShape{M, N, K, 0, 0, 0, ldx, ldw, N, N, parts, static_cast<long long>(M) * N, 0.f, 0.f, 0.f, GW_SUMS}, stream);
  PYLON_LAUNCHED("gemm_wide_parts");
}
