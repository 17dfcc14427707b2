// out[M, N] = x[M, K] * w[N, K]^T, everything in float32, on the matrix cores' float32
// instruction (16x16x4: full 32-bit products and sums, no reduced-precision mode): the matrix
// products of the 32-bit path whose rows are 16-byte aligned.  gemm_tiled takes the rest.
//
// Every element is added up in one order that depends on K alone: K is cut into eight ranges of
// whole chunks of 64 elements, a range is one chain of fused multiply-adds, the sums of the first
// four ranges are added one after the other, those of the last four likewise, and then the two.
// The kernels below share that order, so an element's value does not depend on M, on the tile it
// falls in, or on what else is in the batch.  (A chain is an eighth as long as one over all of K,
// which gemm_tiled takes: logits of six layers are 2.6e-6 off 64 bits instead of 6.7e-6.)
//
// gemm_f32_rows_kernel, up to 32 rows: a step of a few tokens, bound by reading w once.  A
// workgroup owns a tile of up to 16 columns (gf_row_cols); its eight waves take one of the eight ranges
// each, so that even a matrix of 2560 rows has 1,280 waves that stream it, and the order of the
// sums falls out of the order in which the waves' results are added through LDS.  A wave's share
// of w goes from memory straight into LDS in whole 256-byte row segments (four rows a load;
// gemm_rows measures what that is worth), one chunk of 16 rows ahead of the one it multiplies; the
// few rows of x come in operand shape, a chunk ahead too.  No barrier until the end: a wave reads only
// what it brought.  Two workgroups fit a compute unit, and more tiles a workgroup never paid (3 rows, us behind
// 384 MB of other traffic, 1, 2, 3 and 4 tiles: 2560 x 9728 40, 51, 69, 83; 6144 x 2560 28, 28, 30, 32; 19456 x 2560
// 66, 70, 70, 81; 151936 x 2560 289, 298, 311, 312).
//
// gemm_f32_tiles_kernel, more rows: LDS tiles, a chunk ahead, a wave a quarter of the tile's.  One
// 16-byte read from LDS feeds four matrix instructions of 32 clocks and more, so the matrix cores (157 TFLOP/s
// in float32) are what bounds it, where a launch reaches all of them: seven tiles, from 32 x 32 to 96 x 64, some by two
// teams of four waves with half of K each, chosen by a model of the launch's rounds (gf_tiling).
//
// Measured, 4B layer sizes, weights from memory, gemm_tiled (one chain per element on the vector ALUs)
// before: of a step of 3 rows q/k/v 13 us, gate/up 34 (5.9 TB/s), out and down 10 and 22, the head 230 (6.8; the lines
// of w not marked as read once 14, 37, 11, 24, 255)
// where a launch took 615 on average; out, down, q/k/v and gate/up of 270 rows 61, 135, 93 and 266 (91 to 101 TFLOP/s; 600 rows
// 104 to 110).
#include "gemm_f32.h"
#include <type_traits>

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int intx4 __attribute__((ext_vector_type(4)));

#define GF_CHUNK 64           // elements of K: 256 bytes of a row
#define GF_RANGES 8
#define GF_TILE_BYTES 4096    // 16 rows of one chunk
#define GF_ROWS 32            // most rows of the streaming kernel
#define GF_LDS(T) __attribute__((address_space(3))) T
#define GF_OOB 0x80000000u

__device__ __forceinline__ int gf_range_begin(int range, int chunks) {
  return static_cast<int>(static_cast<long long>(range) * chunks / GF_RANGES);
}

// All but the N loads sent last have landed.  No load passes it: neither one that writes LDS nor one of a pointer
// that may be written to (x of the streaming kernel, which is not __restrict__ for that reason: loads of one that is
// are moved to where their values are used, past the wait that counts them).
template <int N>
__device__ __forceinline__ void gf_wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Every wave's reads of LDS have returned and its loads into LDS have landed.
__device__ __forceinline__ void gf_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The body is a device function: the host pass does not know the descriptor type and would drop a
// kernel that names it, launch stub and all.
template <int MT, bool W_FIRST>
__device__ __forceinline__ void gemm_f32_rows_body(float* __restrict__ out, const float* x,
                                                   const float* __restrict__ w, int M, int N, int K, int ldx, int ldw,
                                                   long long ldo, int cols) {
  // per wave two stages of the tile of w; then the ranges' sums, [range][row tile][64 lanes][4]
  __shared__ __attribute__((aligned(1024))) unsigned char lds[GF_RANGES * 2 * GF_TILE_BYTES + GF_RANGES * MT * 1024];
  float* sums = reinterpret_cast<float*>(lds + GF_RANGES * 2 * GF_TILE_BYTES);

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int range = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int r = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * cols;  // first row of w of this workgroup
  const int rows = (N - row0 < cols) ? N - row0 : cols;
  const int chunks = (K + GF_CHUNK - 1) / GF_CHUNK;
  const int c_begin = gf_range_begin(range, chunks), c_end = gf_range_begin(range + 1, chunks);

  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(w + static_cast<size_t>(row0) * ldw), 0,
      static_cast<int>((static_cast<long long>(rows - 1) * ldw + K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(x), 0, static_cast<int>((static_cast<long long>(M - 1) * ldx + K) * 4), 0x00020000);

  // A load brings rows 4 q .. 4 q + 3 of the tile: lane l, for row R = 4 q + l / 16, the 16-byte piece
  // (l % 16) ^ R, which lies at place l % 16 of that row in LDS: operand reads (lane r takes piece
  // 4 s + g of row r) then fall into different groups of banks.  The lanes' offsets are those of chunk 0, the chunk's is
  // scalar; only the chunk that K ends within asks for the lanes' places (the range check of a view does not count the
  // scalar offset).
  const int lrow = lane >> 4, lpos = lane & 15;
  unsigned char* stage_base = lds + range * 2 * GF_TILE_BYTES;
  unsigned w_at[4], x_at[MT], piece_at[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int R = 4 * q + lrow;
    w_at[q] = R < rows ? static_cast<unsigned>(R) * static_cast<unsigned>(ldw) * 4u + (lpos ^ R) * 16 : GF_OOB;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + r;
    x_at[t] = m < M ? static_cast<unsigned>(m) * static_cast<unsigned>(ldx) * 4u + g * 16 : GF_OOB;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) piece_at[s] = (r >> 2) * 1024 + (r & 3) * 256 + (((4 * s + g) ^ r) * 16);

  auto bring = [&](floatx4 (&xv)[MT][4], int chunk, int stage) __attribute__((always_inline)) {
    const int at = chunk * (GF_CHUNK * 4);
    auto send = [&](auto w_off, auto x_off, int offset) __attribute__((always_inline)) {
      auto send_w = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (GF_LDS(void)*)(stage_base + stage * GF_TILE_BYTES + q * 1024), 16,
                                                   w_off(q), offset, 0, PYLON_STREAMED);
      };
      if (W_FIRST) send_w();
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          xv[t][s] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xres, x_off(t, s), offset, 0));
      if (!W_FIRST) send_w();
    };
    if ((chunk + 1) * GF_CHUNK <= K) {
      send([&](int q) { return w_at[q]; }, [&](int t, int s) { return x_at[t] + 64 * s; }, at);
    } else {
      const int left = K - chunk * GF_CHUNK;
      send([&](int q) { return ((lpos ^ (4 * q + lrow)) * 4 < left) ? w_at[q] + at : GF_OOB; },
           [&](int t, int s) { return 16 * s + 4 * g < left ? x_at[t] + 64 * s + at : GF_OOB; }, 0);
    }
  };
  floatx4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const floatx4 (&xv)[MT][4], int stage) __attribute__((always_inline)) {
    const GF_LDS(unsigned char)* base = (const GF_LDS(unsigned char)*)(stage_base + stage * GF_TILE_BYTES);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const floatx4 wf = *reinterpret_cast<const GF_LDS(floatx4)*>(base + piece_at[s]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i], xv[t][s][i], acc[t], 0, 0, 0);
    }
    // this wave's reads of the stage are over before a later turn's loads overwrite it
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  floatx4 x_even[MT][4], x_odd[MT][4];
  auto turn = [&](int chunk, const floatx4 (&xv)[MT][4], floatx4 (&x_next)[MT][4], int stage) __attribute__((always_inline)) {
    if (chunk + 1 < c_end) {
      bring(x_next, chunk + 1, stage ^ 1);
      gf_wait_loads<4 * MT + 4>();  // all but the loads just sent
    } else {
      gf_wait_loads<0>();
    }
    multiply(xv, stage);
  };
  bring(x_even, c_begin, 0);
  for (int chunk = c_begin; chunk < c_end; chunk += 2) {
    turn(chunk, x_even, x_odd, 0);
    if (chunk + 1 < c_end) turn(chunk + 1, x_odd, x_even, 1);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
    *reinterpret_cast<floatx4*>(sums + ((range * MT + t) * PYLON_WAVE + lane) * 4) = acc[t];
  gf_barrier();

  // Wave t now adds row tile t: element (row 16 t + r, column row0 + 4 g + i).
  const bool wide = ((ldo | row0) & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  if (range < MT) {
    const int t = range;
    floatx4 half[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int p = 0; p < GF_RANGES; ++p)
      half[p / (GF_RANGES / 2)] +=
          *reinterpret_cast<const floatx4*>(sums + ((p * MT + t) * PYLON_WAVE + lane) * 4);
    const floatx4 v = half[0] + half[1];
    const int m = 16 * t + r, n = row0 + 4 * g;
    if (m >= M) return;
    float* p = out + static_cast<size_t>(m) * ldo + n;
    const int left = row0 + rows - n;  // columns from here on
    if (wide && left >= 4) {
      *reinterpret_cast<floatx4*>(p) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < left) p[i] = v[i];
    }
  }
}

// What the first loads need are the first 14 words of the arguments, which come with the launch.  W_FIRST: a chunk of w is
// sent for before that of x, for up to 16 deep rows.  It is what rows of 8,192 numbers want (us, x first and w first: 1 x 4096 x
// 8192 39.7, 37.4, 3 x 2560 x 8192 23.7, 23.3; of 9,216 to 25,600 numbers no difference beyond 3 %); shorter ones want x first
// (3 x 6144 x 2560 13.3, 13.7, 16 x 8192 x 512 5.1, 5.4).
template <int MT, bool W_FIRST>
__global__ __launch_bounds__(GF_RANGES* PYLON_WAVE) void gemm_f32_rows_kernel(
    const float* x, const float* __restrict__ w, int M, int N, int K, int cols, int ldx, int ldw,
    float* __restrict__ out, long long ldo) {
  gemm_f32_rows_body<MT, W_FIRST>(out, x, w, M, N, K, ldx, ldw, ldo, cols);
}

// TM, TN: tiles of 16 rows and of 16 columns per wave; WM, WN: waves of a team along them, four together.  TEAMS: 1, or
// 2 teams of four waves that take half of K each.
template <int TM, int TN, int WM, int WN, int TEAMS>
__device__ __forceinline__ void gemm_f32_tiles_body(float* __restrict__ out, const float* __restrict__ x,
                                                    const float* __restrict__ w, int M, int N, int K, long long ldx,
                                                    long long ldw, long long ldo, int m_tiles, int n_tiles) {
  static_assert(WM * WN == 4, "a team is four waves");
  constexpr int X_TILES = TM * WM, W_TILES = TN * WN;
  constexpr int STAGE_BYTES = (X_TILES + W_TILES) * GF_TILE_BYTES;  // the tiles of x, then those of w
  __shared__ __attribute__((aligned(1024))) unsigned char lds[TEAMS * 2 * STAGE_BYTES];

  // Workgroups that share columns of w run on one die (every eighth workgroup), one after the other,
  // so that its cache serves all but the first.
  const int die = blockIdx.x & 7, nth = blockIdx.x >> 3;
  const int mt = nth % m_tiles, nt = (nth / m_tiles) * 8 + die;
  if (nt >= n_tiles) return;
  const int m0 = mt * 16 * X_TILES, n0 = nt * 16 * W_TILES;
  const int m_rows = (M - m0 < 16 * X_TILES) ? M - m0 : 16 * X_TILES, n_rows = (N - n0 < 16 * W_TILES) ? N - n0 : 16 * W_TILES;

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE) & 3;
  const int team = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE) >> 2;
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  const int chunks = (K + GF_CHUNK - 1) / GF_CHUNK;
  const int middle = gf_range_begin(GF_RANGES / 2, chunks);
  const int c_begin = (TEAMS == 2 && team == 1) ? middle : 0, c_end = (TEAMS == 2 && team == 0) ? middle : chunks;
  // every wave of the workgroup takes the same number of turns (the second half is never the shorter one)
  const int turns = TEAMS == 2 ? chunks - middle : chunks;

  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(w + static_cast<size_t>(n0) * ldw), 0,
      static_cast<int>((static_cast<long long>(n_rows - 1) * ldw + K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(x + static_cast<size_t>(m0) * ldx), 0,
      static_cast<int>((static_cast<long long>(m_rows - 1) * ldx + K) * 4), 0x00020000);

  const int lrow = lane >> 4, lpos = lane & 15;
  // Wave v of a team brings quarter v of every tile of x and of w: rows 4 v .. 4 v + 3.
  const int R = 4 * wave + lrow;
  const int lk = (lpos ^ R) * 4;
  unsigned char* team_lds = lds + team * 2 * STAGE_BYTES;
  const unsigned x_step = static_cast<unsigned>(ldx) * 64u, w_step = static_cast<unsigned>(ldw) * 64u;  // a tile's rows
  const unsigned x_first = static_cast<unsigned>(R) * static_cast<unsigned>(ldx) * 4u + lk * 4u;
  const unsigned w_first = static_cast<unsigned>(R) * static_cast<unsigned>(ldw) * 4u + lk * 4u;
  auto issue = [&](int chunk, int stage) {
    // a chunk's first byte; the range check of a view does not count the scalar offset, which rows beyond it need not
    const int at = chunk * (GF_CHUNK * 4);
    unsigned char* base = team_lds + stage * STAGE_BYTES + wave * 1024;
    const bool live = chunk < c_end && chunk * GF_CHUNK + lk < K;
#pragma unroll
    for (int t = 0; t < X_TILES; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (GF_LDS(void)*)(base + t * GF_TILE_BYTES), 16,
                                               live && 16 * t + R < m_rows ? x_first + t * x_step : GF_OOB, at, 0, 0);
#pragma unroll
    for (int t = 0; t < W_TILES; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (GF_LDS(void)*)(base + (X_TILES + t) * GF_TILE_BYTES), 16,
                                               live && 16 * t + R < n_rows ? w_first + t * w_step : GF_OOB, at, 0, 0);
  };
  unsigned piece_at[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) piece_at[s] = (r >> 2) * 1024 + (r & 3) * 256 + (((4 * s + g) ^ r) * 16);

  // of the range under way, of the half under way, of the first half (one team): [column tile][row tile]
  floatx4 acc[TN][TM], half[TN][TM], first[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[j][t] = half[j][t] = first[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  issue(c_begin, 0);
  int range = team * (GF_RANGES / 2);
  for (int turn = 0; turn < turns; ++turn) {
    const int c = c_begin + turn, stage = turn & 1;
    // chunk c has landed for every wave, and every wave is past the products of the turn before
    gf_barrier();
    if (turn + 1 < turns) issue(c + 1, stage ^ 1);
    if (c >= c_end) continue;
    const GF_LDS(unsigned char)* xb =
        (const GF_LDS(unsigned char)*)(team_lds + stage * STAGE_BYTES + wm * TM * GF_TILE_BYTES);
    const GF_LDS(unsigned char)* wb =
        (const GF_LDS(unsigned char)*)(team_lds + stage * STAGE_BYTES + (X_TILES + wn * TN) * GF_TILE_BYTES);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      floatx4 xf[TM], wf[TN];
#pragma unroll
      for (int t = 0; t < TM; ++t) xf[t] = *reinterpret_cast<const GF_LDS(floatx4)*>(xb + t * GF_TILE_BYTES + piece_at[s]);
#pragma unroll
      for (int j = 0; j < TN; ++j) wf[j] = *reinterpret_cast<const GF_LDS(floatx4)*>(wb + j * GF_TILE_BYTES + piece_at[s]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int t = 0; t < TM; ++t)
            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][i], xf[t][i], acc[j][t], 0, 0, 0);
    }
    if (gf_range_begin(range + 1, chunks) == c + 1) {  // the range ends with this chunk
      ++range;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          half[j][t] += acc[j][t];
          acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (TEAMS == 1 && c + 1 == middle) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          first[j][t] = half[j][t];
          half[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if constexpr (TEAMS == 2) {
    // the second team's half goes to the first through LDS, which nobody reads any more
    static_assert(4 * TM * TN * PYLON_WAVE * 16 <= TEAMS * 2 * STAGE_BYTES, "room for a team's sums");
    gf_barrier();
    floatx4* meet = reinterpret_cast<floatx4*>(lds) + wave * TM * TN * PYLON_WAVE + lane;
    if (team == 1) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int t = 0; t < TM; ++t) meet[(j * TM + t) * PYLON_WAVE] = half[j][t];
    }
    gf_barrier();
    if (team == 1) return;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        first[j][t] = half[j][t];
        half[j][t] = meet[(j * TM + t) * PYLON_WAVE];
      }
  }

  const bool wide = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int m = m0 + (wm * TM + t) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + 4 * g;
      const floatx4 v = first[j][t] + half[j][t];
      float* p = out + static_cast<size_t>(m) * ldo + n;
      if (wide && n + 3 < N) {
        *reinterpret_cast<floatx4*>(p) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) p[i] = v[i];
      }
    }
  }
}

template <int TM, int TN, int WM, int WN, int TEAMS>
__global__ __launch_bounds__(TEAMS * 256) void gemm_f32_tiles_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                                     const float* __restrict__ w, int M, int N, int K,
                                                                     long long ldx, long long ldw, long long ldo,
                                                                     int m_tiles, int n_tiles) {
  gemm_f32_tiles_body<TM, TN, WM, WN, TEAMS>(out, x, w, M, N, K, ldx, ldw, ldo, m_tiles, n_tiles);
}

template <int TM, int TN, int WM, int WN, int TEAMS>
static void launch_tiles(float* out, const float* x, const float* w, int M, int N, int K, long long ldx, long long ldw,
                         long long ldo, hipStream_t stream) {
  const int m_side = 16 * TM * WM, n_side = 16 * TN * WN;
  const int m_tiles = (M + m_side - 1) / m_side, n_tiles = (N + n_side - 1) / n_side;
  const dim3 grid(static_cast<unsigned>((n_tiles + 7) / 8 * 8) * m_tiles), block(TEAMS * 256);
  hipLaunchKernelGGL((gemm_f32_tiles_kernel<TM, TN, WM, WN, TEAMS>), grid, block, 0, stream, out, x, w, M, N, K, ldx, ldw,
                     ldo, m_tiles, n_tiles);
}

// Columns a workgroup of the streaming kernel takes: 16, or an equal share where as many whole rounds of the units as
// 16 would need then each have less to stream: in launches of two rounds, in longer ones if K is not short, and in one if K is
// deep (us, 16 against the share.  3 and 24 rows: 2560 x 9728 in 10 25.1, 22.3 and 40.1, 39.2; 5120 x 8192 in 10 50.8, 42.5 and
// 71.7, 64.4; 6144 x 2560 in 12 14.6, 13.9 and 25.2, 23.9; 6144 x 4096 in 12 21.6, 20.3; but 2560 x 4096 10.5, 10.3 and 18.0, 18.2 and
// 3072 x 2560 in 12 8.6, 8.8.  In between, where there are none yet: 2560 x 5120 13.7, 12.8 and 23.9, 22.7; 3072 x 6144 in 12
// 16.3, 15.6 and 27.5, 26.7; 3584 x 7168 in 14 20.4, 20.3 and 31.5, 31.1.  Three rounds, 3 and 17 rows: 8448 x 2560 in 11 19.4,
// 17.6 and 29.4, 28.9, 10240 x 2560 in 14 21.1, 19.9 and 30.5, 30.8; but 8448 x 1536 13.0, 12.2 and 18.0, 22.3, 8448 x 768 8.0,
// 9.0 and 11.7, 13.8, 10240 x 1024 10.1, 9.9 and 14.4, 16.9.)
static int gf_row_cols(int N, int K, int units) {
  const long long rounds = ((N + 15) / 16 + units - 1) / units;
  if (rounds == 1 && (K < 8192 || N < 8 * units)) return 16;
  if (rounds > 2 && K < 2048) return 16;
  const int even = static_cast<int>((N + rounds * units - 1) / (rounds * units));
  return even < 8 ? 8 : even > 16 ? 16 : even;
}

// The tiles of a launch of more than 32 rows.  A workgroup's time for a chunk of K where one, two or three of its kind
// share a compute unit (us, measured over 33 to 900 rows of 2560 x 4096, 2560 x 9728, 6144 x 2560 and 19456 x 2560): from
// these and the number of rounds a launch is estimated, within 8 % of what it takes; the least is chosen.  Small tiles
// reach every unit in a launch of few rows, large ones read less from the second-level cache and from LDS for each
// product.  Two sizes alone, 32 x 32 and (from 512 rows on) 64 x 64, took, out, down, q/k/v and gate/up of 4B sizes at 270
// rows, 69, 156, 96 and 287 us where these take 61, 135, 93 and 266, at 600 135, 296, 189, 557 and 118, 274, 181, 546, at 900 212,
// 479, 282, 831 and 173, 397, 266, 786.
enum { GF_32_TEAMS, GF_32_WIDE, GF_48, GF_48_TEAMS, GF_64_TEAMS, GF_96, GF_64, GF_TILINGS };
struct GfTiling {
  int m, n, threads, resident;
  float chunk[3];  // with as many on a unit
};
static const GfTiling gf_tilings[GF_TILINGS] = {
    {32, 32, 512, 2, {0.46f, 0.64f, 0.f}}, {32, 64, 256, 3, {0.84f, 1.29f, 1.80f}}, {48, 64, 256, 2, {1.09f, 1.65f, 0.f}},
    {48, 64, 512, 1, {0.88f, 0.f, 0.f}},   {64, 64, 512, 1, {1.12f, 0.f, 0.f}},    {96, 64, 256, 2, {1.91f, 3.19f, 0.f}},
    {64, 64, 256, 2, {1.39f, 2.25f, 0.f}}};

static int gf_tiling(int M, int N, int units) {
  auto groups = [&](const GfTiling& t) {
    return static_cast<long long>((M + t.m - 1) / t.m) * (((N + t.n - 1) / t.n + 7) / 8 * 8);
  };
  // a launch holds less than 2^32 threads
  auto fits = [&](int tiling) { return groups(gf_tilings[tiling]) * gf_tilings[tiling].threads < (1ll << 32); };
  int best = GF_TILINGS;
  if (M <= (1 << 15) && N <= (1 << 20)) {  // (larger ones have not been measured)
    float least = 0.f;
    for (int i = 0; i < GF_TILINGS; ++i) {
      const GfTiling& t = gf_tilings[i];
      if (!fits(i)) continue;
      const long long round = static_cast<long long>(t.resident) * units;
      const long long count = static_cast<long long>((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
      const long long rest = count % round;
      float us = static_cast<float>(count / round) * t.chunk[t.resident - 1];
      if (rest > 0) us += t.chunk[(rest + units - 1) / units - 1];
      if (best == GF_TILINGS || us < least) best = i, least = us;
    }
    if (best != GF_TILINGS) return best;
  }
  const bool many = M >= 512 && static_cast<long long>((M + 63) / 64) * ((N + 63) / 64) >= 3ll * units;
  if (!many && fits(GF_32_TEAMS)) return GF_32_TEAMS;
  return fits(GF_64) ? GF_64 : GF_TILINGS;
}

// What computes a product of these sizes in float32 (units: compute units): 16 the streaming kernel, 32 tiles of fewer
// than 64 rows, 64 larger ones; 0 where gemm_tiled takes it.  Touches no device.
extern "C" int pylon_gemm_f32_plan(int M, int N, int units, int* side) {
  PYLON_REQUIRE(M >= 1 && N >= 1 && units >= 1 && side != nullptr, "gemm_f32_plan: bad arguments");
  const int tiling = gf_tiling(M, N, units);
  *side = M <= GF_ROWS ? 16 : tiling == GF_TILINGS ? 0 : gf_tilings[tiling].m < 64 ? 32 : 64;
  return 0;
}

// The columns that a workgroup of the streaming kernel takes of such a product.  Touches no device.
extern "C" int pylon_gemm_f32_columns(int N, int K, int units, int* columns) {
  PYLON_REQUIRE(N >= 1 && K >= 1 && units >= 1 && columns != nullptr, "gemm_f32_columns: bad arguments");
  *columns = gf_row_cols(N, K, units);
  return 0;
}

// Whether the kernels of this file take the operands: whole 16-byte pieces of rows, offsets within a
// workgroup's rows that a buffer descriptor spans, and a chunk of K for every range.  The last is not a
// matter of time (one row, 512 outputs: 44.0 us at K = 508 in gemm_tiled, 3.1 us at K = 512 here; 300 rows
// of 2048 outputs: 47.9 and 12.0): a shorter K would leave ranges empty, and models that small keep the
// one ascending chain that recorded runs of theirs hold, choices between near ties included.  Nothing here
// depends on M.
bool gemm_f32_takes(const void* x, const void* w, int K, long long ldx, long long ldw) {
  return K >= GF_RANGES * GF_CHUNK && K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && ldx <= (1ll << 21) &&
         ldw <= (1ll << 21) && (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
}

// M >= 1; false if the device is unknown or the launch would be too large (nothing launched then).
bool gemm_f32_launch(float* out, const float* x, const float* w, int M, int N, int K, long long ldx, long long ldw,
                     long long ldo, hipStream_t stream) {
  const int units = pylon_compute_units();
  if (units <= 0) return false;
  if (M <= GF_ROWS) {
    const int cols = gf_row_cols(N, K, units);
    const dim3 grid((N + cols - 1) / cols), block(GF_RANGES * PYLON_WAVE);
#define GO(MT, W_FIRST)                                                                                            \
  hipLaunchKernelGGL((gemm_f32_rows_kernel<MT, W_FIRST>), grid, block, 0, stream, x, w, M, N, K, cols, (int)ldx, (int)ldw, out, ldo)
    if (M > 16) GO(2, false);
    else if (K >= 8192) GO(1, true);
    else GO(1, false);
#undef GO
    return true;
  }
#define GO(TM, TN, WM, WN, TEAMS) launch_tiles<TM, TN, WM, WN, TEAMS>(out, x, w, M, N, K, ldx, ldw, ldo, stream)
  switch (gf_tiling(M, N, units)) {
    case GF_32_TEAMS: GO(1, 1, 2, 2, 2); break;
    case GF_32_WIDE: GO(2, 1, 1, 4, 1); break;
    case GF_48: GO(3, 1, 1, 4, 1); break;
    case GF_48_TEAMS: GO(3, 1, 1, 4, 2); break;
    case GF_64: GO(2, 2, 2, 2, 1); break;
    case GF_64_TEAMS: GO(2, 2, 2, 2, 2); break;
    case GF_96: GO(3, 2, 2, 2, 1); break;
    default: return false;
  }
#undef GO
  return true;
}
