// out[M, N] = x[M, K] * w[N, K]^T in bfloat16 for up to 64 rows of x a workgroup (up to 128 a
// launch, as two halves with workgroups of their own): the matrix products of a decode step,
// bound by reading w once, with x from 17 rows on no longer small beside a workgroup's share
// of w.
//
// A workgroup of four wavefronts owns 64 or 128 columns of the output (each wave one or two
// tiles of 16 rows of w) over a range of K; K is cut over blockIdx.y and every cut writes
// its own float partial result, which the consumer adds (the fused residual norm does), or,
// with one cut, the result itself.  The workgroup walks its range in chunks of 128 elements.
//
// Both operands travel from memory straight into LDS (buffer_load_dwordx4 ... lds: a wave
// fills 1 KB of consecutive LDS from 64 places of its choice) in whole row segments: one
// load takes the 256 contiguous bytes that a chunk is of each of four rows.  (A load that
// takes 64 bytes of each of 16 rows, the shape of a matrix-instruction operand, moves less
// than half as much per compute unit: measured 21 us against 8 us for the rows of x of a
// 19456 x 2560 product.)  The rows of x of a chunk are shared by the four waves; each wave
// brings its own tiles of w.  In LDS a tile is 16 rows of 256 bytes, and the 16-byte piece q
// of row R lies at position q ^ R of that row, so that the operand reads (lane r takes piece
// 4 s + g of row r) of 16 lanes fall into 16 different groups of banks.  Several chunks are in
// flight: while chunk c is multiplied, the next two or three travel.  There is one barrier
// per chunk, preceded by a counted wait for this wave's loads of chunk c only, so the later
// loads stay in flight across it.  No sums cross waves: a wave owns its columns.
//
// A workgroup takes `wg_cols` columns, at most what its waves' tiles hold and not necessarily
// that many: the host gives every workgroup of a launch the same share of the columns, chosen
// so that the workgroups are a whole number of rounds over the compute units.  Its waves take
// full tiles in turn; the rows of a tile beyond the workgroup's columns are out of range and
// fetch nothing, and a wave left without columns only helps to bring the rows of x.  (The
// gate/up product of 2 x 9728 columns: 38 per workgroup, one workgroup per unit, 20.0 us
// against 21.0 for 64 or 48 columns per workgroup where some units stream half as much again
// as others.)
//
// All loads go through buffer descriptors (of the workgroup's rows of w; of x): rows beyond
// N or M are read as zeros without a memory access and without a branch, so every wave
// issues the same number of loads per chunk and the counted waits are exact.
//
// A launch of a few microseconds is mostly its start and its end, and with one wavefront on a
// SIMD every instruction takes four clocks or more: a load is two instructions (its offset
// within the chunk is computed once, the chunk's is scalar), what is asked before the first
// load comes with the launch, and nothing is sent beyond the range.  With a check a load and
// loads beyond the range 6144 x 2560, 2560 x 4096, 2560 x 9728 and 2 x 9728 x 2560 took 8.3,
// 6.3, 11.8 and 20.9 us at 8 rows, then 7.6, 5.6, 11.0 and 20.0; at 48 rows 10.5, 9.3, 14.3
// and 25.2, then 9.3, 8.3, 12.9 and 23.4 (under a graph, matrices that no cache holds).
//
// The lines of w are marked as read once (PYLON_STREAMED): the same products then 6.8, 5.3, 10.1 and 18.1 us at 8 rows
// and 8.6, 7.2, 11.5 and 21.4 at 48 (heads of 151,936 rows 12 % less at 8, 4 to 10 at 64).
#include "common.h"

#include <type_traits>
#include <utility>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

#define GR_CHUNK 128
#define GR_TILE_BYTES 4096  // 16 rows of one chunk
#define GR_LDS(T) __attribute__((address_space(3))) T

// A barrier behind a wait for this wave's reads of LDS only.  The invariant it keeps: when a
// wave passes it, every wave's operand reads of the chunk before have returned, so the loads
// issued next may overwrite that chunk's stage.  The loads from memory that must have landed
// are counted by hand below and are not waited for here.  (A release fence on LDS would wait
// for every outstanding load, because the loads that write LDS are among them, and the
// chunks in flight would drain at every barrier.)
__device__ __forceinline__ void gr_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// vmcnt <= N (N < 64); the other counters are left alone.
template <int N>
__device__ __forceinline__ void gr_wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

template <typename F, int... I>
__device__ __forceinline__ void gr_for_(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), ... f(N - 1) with the number a constant each time.
template <int N, typename F>
__device__ __forceinline__ void gr_for(F&& f) {
  gr_for_(f, std::make_integer_sequence<int, N>{});
}

// Stages of LDS for MT tiles of x and WAVES * CT tiles of w per chunk.
template <int MT, int CT, int WAVES>
struct GrShape {
  static constexpr int TILES = MT + WAVES * CT;
  static constexpr int STAGE_BYTES = TILES * GR_TILE_BYTES;
  // Four stages where they fit and a wave brings one tile of w per chunk, else three: 2560 x 9728 at
  // 8 rows takes 11.9, 11.0, 11.2 and 11.6 us with three, four, six and eight, 2560 x 4096 6.2, 5.6, 5.8
  // and 6.1; with two tiles a wave (36 KB a stage and more) three and four are within 1 %.
  static constexpr int STAGES = (4 * STAGE_BYTES <= 144 * 1024 && CT == 1) ? 4 : 3;
};

// What happens to the sums.  Gated: `variant` picks the gate's activation (pylon_gate_act), or gate and up are
// capped, as pylon_gated_act does it; not gated: nothing, or (variant 1) the squared relu.
struct GrAct {
  int variant;
  float alpha, offset, limit;
};
enum GrGate { GR_NO_GATE = 0, GR_GATE = 1, GR_CAPPED_GATE = 2 };

// MT: tiles of 16 rows of x (1..4); CT: tiles of 16 rows of w per wave (1 or 2).
// GLU (CT = 2): w is a fused gate/up matrix of 2 N rows; a wave's first tile is 16 gate rows,
// its second the 16 up rows that lie N rows further down, and it writes the activated gate times up.
// (The capped gate has a kernel of its own: with alpha, offset and limit among the arguments of all, every
// decode step lost 0.4 %.  In the epilogue it saves a layer the activation's launch, 4.8 us, and the float32
// round trip of gate and up: a run of eight layers, 4 requests, 33.5 -> 33.2 ms.)
// (The body is a device function: the host pass does not know the descriptor type and would
// drop a kernel that names it, launch stub and all.)
template <int MT, int CT, int GLU, int WAVES, typename TO>
__device__ __forceinline__ void gemm_rows_body(
    TO* __restrict__ out, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int N,
    int K, int ldx, int ldw, long long ldo, long long part_stride, int chunks_per_part,
    int wg_cols, int group, bool wide, GrAct act) {
  typedef GrShape<MT, CT, WAVES> Shape;
  constexpr int QW = 4 / WAVES;  // quarters of every tile of x that a wave fills
  constexpr int STAGES = Shape::STAGES;
  constexpr int LOADS = QW * MT + 4 * CT;  // loads a wave issues per chunk
  __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * Shape::STAGE_BYTES];

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int r = lane & 15, g = lane >> 4;
  constexpr int WAVE_COLS = (GLU ? 1 : CT) * 16;  // columns of the output per wave
  const int wg_row0 = group * wg_cols;  // the workgroup's first row of w
  const int wg_rows = N - wg_row0 < wg_cols ? N - wg_row0 : wg_cols;
  const int first = wave * WAVE_COLS;  // the wave's first column, of the workgroup's
  const int part = blockIdx.y;
  const int chunks = (K + GR_CHUNK - 1) / GR_CHUNK;
  const int c_begin = part * chunks_per_part;
  const int c_end = (c_begin + chunks_per_part < chunks) ? c_begin + chunks_per_part : chunks;

  // Every view ends with its last row: a tile's rows beyond the workgroup's columns, or beyond M, lie outside it
  // and fetch nothing.  With GLU the up rows have a view of their own, N rows further.
  const uint16_t* const wg_w = w + static_cast<size_t>(wg_row0) * ldw;
  const unsigned w_bytes = (static_cast<unsigned>(wg_rows - 1) * ldw + K) * 2u;
  const unsigned x_bytes = (static_cast<unsigned>(M - 1) * ldx + K) * 2u;

  // A load fills rows 4 q .. 4 q + 3 of a tile (q: the quarter): lane l brings, for row
  // R = 4 q + l / 16, the piece (l % 16) ^ R.  Byte offsets in chunk 0: of at most 128 rows of 8 MB, which the host sees
  // to, so that none of them, nor with a chunk's added, passes 2^31.
  // x: this wave fills quarters QW * wave .. of every tile of x; w: all four of its own CT tiles.
  const int lrow = lane >> 4, piece = (lane & 15) ^ lrow;
  unsigned x_at[QW][MT], w_at[GLU ? 1 : CT][4];
#pragma unroll
  for (int u = 0; u < QW; ++u) {
    const int q = QW * wave + u;
#pragma unroll
    for (int t = 0; t < MT; ++t)
      x_at[u][t] = static_cast<unsigned>(16 * t + 4 * q + lrow) * (2u * ldx) + ((piece ^ (4 * q)) * 16);
  }
#pragma unroll
  for (int j = 0; j < (GLU ? 1 : CT); ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      w_at[j][q] = static_cast<unsigned>(first + 16 * j + 4 * q + lrow) * (2u * ldw) + ((piece ^ (4 * q)) * 16);
  // Operand reads: lane (r, g) takes piece 4 s + g of row r of a tile.
  unsigned piece_at[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) piece_at[s] = (r >> 2) * 1024 + (r & 3) * 256 + (((4 * s + g) ^ r) * 16);

  floatx4 acc[CT][MT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  // The loads of chunk c into a stage, its offset their scalar one.  Pieces beyond K (of a chunk that K ends
  // within) bring what follows in the view, or zeros behind its last row; their products are left out.
  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wg_w), 0, w_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ures = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(wg_w + (GLU ? static_cast<size_t>(N) * ldw : 0)), 0, w_bytes, 0x00020000);
  auto issue = [&](int c, int stage) __attribute__((always_inline)) {
    int at = c * (GR_CHUNK * 2);
    if ((c + 1) * GR_CHUNK > K) {
      // The range check does not count the scalar offset: in this chunk, which is the last that is sent, the lanes'
      // offsets carry it, so that the last rows' pieces beyond K are beyond their views too.
#pragma unroll
      for (int u = 0; u < QW; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t) x_at[u][t] += at;
#pragma unroll
      for (int j = 0; j < (GLU ? 1 : CT); ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) w_at[j][q] += at;
      at = 0;
    }
    unsigned char* const base = lds + stage * Shape::STAGE_BYTES;
#pragma unroll
    for (int u = 0; u < QW; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (GR_LDS(void)*)(base + t * GR_TILE_BYTES + (QW * wave + u) * 1024), 16,
                                                 x_at[u][t], at, 0, 0);
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            GLU && j == 1 ? ures : wres, (GR_LDS(void)*)(base + (MT + wave * CT + j) * GR_TILE_BYTES + q * 1024), 16,
            w_at[GLU ? 0 : j][q], at, 0, PYLON_STREAMED);
  };
  auto compute = [&](int stage, int left) __attribute__((always_inline)) {  // left: elements from the chunk's first to K
    const GR_LDS(unsigned char)* base = (const GR_LDS(unsigned char)*)(lds + stage * Shape::STAGE_BYTES);
    auto product = [&](auto there) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        bf16x8 xf[MT], wf[CT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
          xf[t] = there(*reinterpret_cast<const GR_LDS(bf16x8)*>(base + t * GR_TILE_BYTES + piece_at[s]), s);
#pragma unroll
        for (int j = 0; j < CT; ++j)
          wf[j] = there(*reinterpret_cast<const GR_LDS(bf16x8)*>(base + (MT + wave * CT + j) * GR_TILE_BYTES + piece_at[s]), s);
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[t], acc[j][t], 0, 0, 0);
      }
    };
    if (left >= GR_CHUNK)
      product([](bf16x8 v, int) __attribute__((always_inline)) { return v; });
    else
      product([&](bf16x8 v, int s) __attribute__((always_inline)) { return (4 * s + g) * 8 < left ? v : bf16x8{}; });
  };

  // Chunk c lives in stage (c - c_begin) % STAGES.  At the top of turn c the loads of chunks
  // c .. c + STAGES - 2 are outstanding; chunk c has landed once at most those of the later
  // ones are.  After the barrier every wave is past the products of chunk c - 1, whose stage
  // chunk c + STAGES - 1 takes.  The last turns have nothing left to send and wait for fewer loads each (loads
  // beyond the range, sent to keep one count, cost a launch 0.14 us a chunk).
  int stage = 0;
  auto turn = [&](int c) __attribute__((always_inline)) {
    if (first < wg_rows) compute(stage, K - c * GR_CHUNK);
    stage = (stage + 1 == STAGES) ? 0 : stage + 1;
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (c_begin + i < c_end) issue(c_begin + i, i);
  int c = c_begin;
  for (; c + STAGES - 1 < c_end; ++c) {
    gr_wait_loads<LOADS*(STAGES - 2)>();
    gr_barrier();
    issue(c + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
    turn(c);
  }
  gr_for<STAGES - 1>([&](auto I) __attribute__((always_inline)) {
    constexpr int later = STAGES - 2 - decltype(I)::value;  // chunks behind this turn's
    if (c + later < c_end) {
      gr_wait_loads<LOADS * later>();
      gr_barrier();
      turn(c++);
    }
  });

  // acc[j][t][i] is out[16 t + r][first + 16 j + 4 g + i] of the workgroup's columns (with GLU: gate and up of
  // column first + 4 g + i).  Four values of a lane go out as one store where every row of every part is
  // aligned for it.
  TO* dst = out + static_cast<size_t>(part) * part_stride + wg_row0;
  wide = wide && (wg_row0 & 3) == 0;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < (GLU ? 1 : CT); ++j) {
      const int n = first + 16 * j + 4 * g;
      floatx4 v = acc[j][t];
      if constexpr (GLU == GR_GATE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = pylon_gate_act(acc[0][t][i], act.variant) * acc[1][t][i];
      } else if constexpr (GLU == GR_CAPPED_GATE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float gate = acc[0][t][i], up = acc[1][t][i];
          if (act.limit > 0.f) {
            gate = fminf(gate, act.limit);
            up = fminf(fmaxf(up, -act.limit), act.limit);
          }
          v[i] = (gate / (1.0f + expf(-act.alpha * gate))) * (up + act.offset);
        }
      } else if (act.variant) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pos = fmaxf(v[i], 0.f);
          v[i] = pos * pos;
        }
      }
      TO* p = dst + static_cast<size_t>(m) * ldo + n;
      if (wide && n + 3 < wg_rows) {
        if constexpr (sizeof(TO) == 4) {
          *reinterpret_cast<floatx4*>(p) = v;
        } else {
          uint2 packed;
          packed.x = floats_to_bf16_pair(v[0], v[1]);
          packed.y = floats_to_bf16_pair(v[2], v[3]);
          *reinterpret_cast<uint2*>(p) = packed;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < wg_rows) p[i] = from_float<TO>(v[i]);
      }
    }
  }
}

// The arguments that the first loads need are the first 14 words, which come with the launch.
template <int MT, int CT, int GLU, int WAVES, typename TO>
__global__ __launch_bounds__(WAVES* PYLON_WAVE) void gemm_rows_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int N, int K, int ldx, int ldw,
    int chunks_per_part, int wg_cols, int row_split, int groups, int flags, TO* __restrict__ out, long long ldo,
    long long part_stride) {
  // More than 64 rows of x go as two halves of `row_split` rows, each to workgroups of its
  // own that take the same columns: blockIdx.x counts eight groups of columns for the first
  // half, the same eight for the second, then the next eight, so that the two workgroups that
  // stream the same rows of w start together and on the same die (a die takes every eighth
  // workgroup), where the second finds in the cache what the first brought.
  int group = blockIdx.x;
  if (row_split > 0) {
    const int half = (blockIdx.x >> 3) & 1;
    group = ((blockIdx.x >> 4) << 3) | (blockIdx.x & 7);
    if (group >= groups) return;  // the grid is padded to whole sixteens
    x += static_cast<size_t>(half) * row_split * ldx;
    out += static_cast<size_t>(half) * row_split * ldo;
    M = (M - half * row_split < row_split) ? M - half * row_split : row_split;
  }
  gemm_rows_body<MT, CT, GLU, WAVES, TO>(out, x, w, M, N, K, ldx, ldw, ldo, part_stride, chunks_per_part, wg_cols,
                                         group, (flags & 2) != 0, GrAct{flags & 1, 0.f, 0.f, 0.f});
}

// The same with a capped gate; up to 64 rows, whole K.
template <int MT, int WAVES>
__global__ __launch_bounds__(WAVES* PYLON_WAVE) void gemm_rows_capped_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int N, int K, int ldx, int ldw, int wg_cols,
    int wide, bf16_t* __restrict__ out, long long ldo, GrAct act) {
  gemm_rows_body<MT, 2, GR_CAPPED_GATE, WAVES, bf16_t>(out, x, w, M, N, K, ldx, ldw, ldo, 0, (K + GR_CHUNK - 1) / GR_CHUNK,
                                                       wg_cols, blockIdx.x, wide != 0, act);
}

// How a product is laid over the chip: wavefronts per workgroup, workgroups along the columns,
// and the columns each of them takes.
struct GrLaunch {
  int waves, groups, wg_cols;
};

// units: compute units of the device.  waves: 4, 2, or 0 for two where four would give fewer
// workgroups than half the units.  cols: columns per workgroup, or 0 for the rule: an equal
// share for every workgroup of as many whole rounds over the units as workgroups of full
// width would need (at least 16 columns), unless that makes the workgroups re-read more rows
// of x than they stream rows of w; then, and beyond 16 rows of x in launches of several rounds
// whose last is not mostly empty, the full width.  Measured at 2560 x 9728, K cut in eight, 32 rows: 11.2 us with 80
// columns (256 workgroups) against 12.9 with 128 (160); 2560 x 4096 cut in four, 48 rows: 8.1 with
// 40 columns against 8.4 with 64; the head of 151936 rows at 8 rows of x: 137.6 with 119
// columns against 138.4; at 64 rows of x (4.6 rounds): 179.6 against 169.1; a gate/up matrix of
// 2 x 17408 rows at 17 rows of x (1.06 rounds of 64 columns): 65 with 34 columns in 512 workgroups against 86.
static GrLaunch gr_launch_shape(int M, int N, int parts, int col_tiles, int glu, int waves, int units, int cols) {
  const int wave_cols = (glu ? 1 : col_tiles) * 16;
  if (waves == 0)
    waves = (static_cast<long long>((N + 4 * wave_cols - 1) / (4 * wave_cols)) * parts < units / 2) ? 2 : 4;
  const int full = waves * wave_cols;
  if (cols <= 0) {
    const long long least = static_cast<long long>((N + full - 1) / full) * parts;  // workgroups of full width
    const long long rounds = (least + units - 1) / units;
    const long long groups = rounds * units / parts;
    int even = groups > 0 ? static_cast<int>((N + groups - 1) / groups) : full;
    even = even < 16 ? 16 : (even > full ? full : even);
    // several rounds of full width are left alone unless the last is mostly empty
    const bool uneven = rounds == 1 || least * 100 < rounds * units * 85;
    const bool pays = M <= 16 || (uneven && even * (glu ? 2 : 1) >= M);
    cols = pays ? even : full;
  }
  return GrLaunch{waves, (N + cols - 1) / cols, cols};
}

template <int MT, int CT, int GLU, int WAVES>
static void launch_rows_waves(void* out, int out_dtype, const void* x, const void* w, int M, int N, int K,
                              long long ldx, long long ldw, long long ldo, int parts, long long part_stride,
                              const GrLaunch& shape, int row_split, GrAct act, hipStream_t stream) {
  const int chunks = (K + GR_CHUNK - 1) / GR_CHUNK;
  const int per_part = (chunks + parts - 1) / parts;
  dim3 grid(row_split > 0 ? 2 * ((shape.groups + 7) / 8 * 8) : shape.groups, parts), block(WAVES * PYLON_WAVE);
  // columns at multiples of four are aligned for a store of four in every row of every part
  const int size = out_dtype == PYLON_F32 ? 4 : 2;
  const int wide = (ldo & 3) == 0 && (part_stride & 3) == 0 &&
                   (reinterpret_cast<uintptr_t>(out) & (4 * size - 1)) == 0;
  if constexpr (GLU == GR_CAPPED_GATE)
    hipLaunchKernelGGL((gemm_rows_capped_kernel<MT, WAVES>), grid, block, 0, stream, (const uint16_t*)x, (const uint16_t*)w,
                       M, N, K, (int)ldx, (int)ldw, shape.wg_cols, wide, (bf16_t*)out, ldo, act);
  else if (out_dtype == PYLON_F32)
    hipLaunchKernelGGL((gemm_rows_kernel<MT, CT, GLU, WAVES, float>), grid, block, 0, stream, (const uint16_t*)x,
                       (const uint16_t*)w, M, N, K, (int)ldx, (int)ldw, per_part, shape.wg_cols, row_split, shape.groups,
                       act.variant | wide << 1, (float*)out, ldo, part_stride);
  else
    hipLaunchKernelGGL((gemm_rows_kernel<MT, CT, GLU, WAVES, bf16_t>), grid, block, 0, stream, (const uint16_t*)x,
                       (const uint16_t*)w, M, N, K, (int)ldx, (int)ldw, per_part, shape.wg_cols, row_split, shape.groups,
                       act.variant | wide << 1, (bf16_t*)out, ldo, part_stride);
}

// Workgroups of four waves, or of two where four would leave compute units without one.
template <int MT, int CT, int GLU>
static void launch_rows(void* out, int out_dtype, const void* x, const void* w, int M, int N, int K,
                        long long ldx, long long ldw, long long ldo, int parts, long long part_stride,
                        const GrLaunch& shape, int row_split, GrAct act, hipStream_t stream) {
  if (shape.waves == 2)
    launch_rows_waves<MT, CT, GLU, 2>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape,
                                      row_split, act, stream);
  else
    launch_rows_waves<MT, CT, GLU, 4>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape,
                                      row_split, act, stream);
}

// What pylon_gemm_rows would launch for these arguments on a device of `units` compute units
// (0: the current device's): shape[0] wavefronts per workgroup, shape[1] workgroups along
// the columns (times `parts` along K), shape[2] the columns each of them takes.
// Touches no device memory; with units given it runs without a GPU.
extern "C" int pylon_gemm_rows_shape(int M, int N, int parts, int col_tiles, int glu, int waves, int units,
                                     int cols, int* shape) {
  PYLON_REQUIRE(shape != nullptr && M >= 1 && N > 0 && parts >= 1 && cols >= 0, "gemm_rows_shape: bad arguments");
  PYLON_REQUIRE(col_tiles == 1 || col_tiles == 2, "gemm_rows_shape: col_tiles is 1 or 2");
  PYLON_REQUIRE(waves == 0 || waves == 2 || waves == 4, "gemm_rows_shape: waves is 0, 2 or 4");
  if (units <= 0) units = pylon_compute_units();
  PYLON_REQUIRE(units > 0, "gemm_rows_shape: no device to take the number of compute units from");
  // beyond 64 rows each half of the rows has workgroups of its own: shape[1] of them per half
  const GrLaunch l = gr_launch_shape(M > 64 ? (M + 1) / 2 : M, N, parts, col_tiles, glu, waves, units, cols);
  shape[0] = l.waves, shape[1] = l.groups, shape[2] = l.wg_cols;
  return 0;
}

// x: [M, ldx] bf16, 1 <= M <= 128 (beyond 64 rows two halves of (M + 1) / 2 and the rest, each to
// workgroups of its own); w: [N, ldw] bf16 (with glu: [2N, ldw], gate rows first, then
// up rows); out: `parts` results [M, ldo] spaced part_stride elements apart (parts > 1 needs
// float out and no glu).  col_tiles: tiles of 16 columns per wave, 1 or 2; with glu a wave
// takes 16 gate rows and their 16 up rows, gated through silu (glu = 3: through gelu; glu = 5: capped as
// pylon_gated_act does it, by alpha, offset and limit, which the others do not read; up to 64 rows, bfloat16 result);
// glu = 2: no gate, the result is max(x w^T, 0)^2.  waves: wavefronts per workgroup, 4 or 2 (0: two if
// four would give fewer workgroups than half the device's compute units).  cols: columns per
// workgroup, at most what its waves' tiles hold (0: the rule of gr_launch_shape); the sums do
// not depend on it.
extern "C" int pylon_gemm_rows(void* out, int out_dtype, const void* x, const void* w, int M, int N, int K,
                               long long ldx, long long ldw, long long ldo, int parts, long long part_stride,
                               int col_tiles, int glu, int waves, int cols, float alpha, float offset,
                               float limit, hipStream_t stream) {
  PYLON_REQUIRE(pylon_valid_dtype(out_dtype), "gemm_rows: unknown output dtype");
  PYLON_REQUIRE((glu >= 0 && glu <= 3) || glu == 5, "gemm_rows: unknown epilogue %d", glu);
  const bool capped = glu == 5;
  PYLON_REQUIRE(!capped || (out_dtype == PYLON_BF16 && M <= 64), "gemm_rows: the capped gate takes up to 64 rows and "
                "a bfloat16 result");
  // 1: the squared relu of a product without a gate, or gelu instead of silu in one with
  const GrAct act{glu == 2 || glu == 3 ? 1 : 0, alpha, offset, limit};
  PYLON_REQUIRE(parts == 1 || glu != 2, "gemm_rows: the squared relu needs the whole of K");
  glu &= 1;
  PYLON_REQUIRE(M >= 0 && M <= 128, "gemm_rows: takes at most 128 rows, got %d", M);
  PYLON_REQUIRE(N > 0 && K > 0, "gemm_rows: bad sizes N=%d K=%d", N, K);
  PYLON_REQUIRE(K % 8 == 0, "gemm_rows: K=%d must be a multiple of 8", K);
  PYLON_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0, "gemm_rows: row strides must be multiples of 8 elements");
  PYLON_REQUIRE(ldw >= K && ldx >= K && ldo >= N, "gemm_rows: a row stride is too short");
  PYLON_REQUIRE(ldw <= (1ll << 22) && ldx <= (1ll << 22),
                "gemm_rows: row strides beyond 4M elements are not supported");
  PYLON_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                "gemm_rows: operands must be 16-byte aligned");
  PYLON_REQUIRE(col_tiles == 1 || col_tiles == 2, "gemm_rows: col_tiles is 1 or 2, got %d", col_tiles);
  PYLON_REQUIRE(parts >= 1 && parts <= 64, "gemm_rows: parts must be 1..64");
  PYLON_REQUIRE(parts == 1 || out_dtype == PYLON_F32, "gemm_rows: partial results must be float");
  PYLON_REQUIRE(parts == 1 || !glu, "gemm_rows: the gated epilogue needs the whole of K");
  PYLON_REQUIRE(parts == 1 || part_stride >= static_cast<long long>(M) * ldo,
                "gemm_rows: partial results overlap");
  // (one view once spanned gate and up rows; each has its own now, and larger matrices stay refused)
  PYLON_REQUIRE(!glu || (static_cast<long long>(N) + 64) * ldw * 2 < (1ll << 31),
                "gemm_rows: a fused gate/up matrix of %d rows of %lld elements is beyond the 2 GB a "
                "workgroup's view of it may span", 2 * N, ldw);
  PYLON_REQUIRE(waves == 0 || waves == 2 || waves == 4, "gemm_rows: waves is 0, 2 or 4, got %d", waves);
  if (M == 0) return 0;
  const int units = pylon_compute_units();
  PYLON_REQUIRE(units > 0, "gemm_rows: the device's number of compute units is unknown");
  // beyond 64 rows: two halves, each to workgroups of its own
  const int row_split = M > 64 ? (M + 1) / 2 : 0;
  const int rows_each = row_split > 0 ? row_split : M;
  const GrLaunch shape = gr_launch_shape(rows_each, N, parts, col_tiles, glu, waves, units, cols);
  PYLON_REQUIRE(cols >= 0 && cols <= shape.waves * (glu ? 1 : col_tiles) * 16,
                "gemm_rows: %d columns per workgroup are more than the tiles of its %d waves hold", cols, shape.waves);
#define GO(MT)                                                                                              \
  do {                                                                                                      \
    if (capped) launch_rows<MT, 2, GR_CAPPED_GATE>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape, row_split, act, stream); \
    else if (glu) launch_rows<MT, 2, GR_GATE>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape, row_split, act, stream); \
    else if (col_tiles == 2) launch_rows<MT, 2, GR_NO_GATE>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape, row_split, act, stream); \
    else launch_rows<MT, 1, GR_NO_GATE>(out, out_dtype, x, w, M, N, K, ldx, ldw, ldo, parts, part_stride, shape, row_split, act, stream); \
  } while (0)
  switch ((rows_each + 15) / 16) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 3: GO(3); break;
    default: GO(4); break;
  }
#undef GO
  PYLON_LAUNCHED("gemm_rows");
}
