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
// workgroup owns a tile of 16 columns; its eight waves take one of the eight ranges
// each, so that even a matrix of 2560 rows has 1,280 waves that stream it, and the order of the
// sums falls out of the order in which the waves' results are added through LDS.  A wave's share
// of w goes from memory straight into LDS in whole 256-byte row segments (four rows a load;
// gemm_rows measures what that is worth), one chunk of 16 rows ahead of the one it multiplies; the
// few rows of x come in operand shape, a chunk ahead too.  No barrier until the end: a wave reads only
// what it brought.  Two workgroups fit a compute unit, and more tiles a workgroup never paid (3 rows, us behind
// 384 MB of other traffic, 1, 2, 3 and 4 tiles: 2560 x 9728 40, 51, 69, 83; 6144 x 2560 28, 28, 30, 32; 19456 x 2560
// 66, 70, 70, 81; 151936 x 2560 289, 298, 311, 312).
//
// gemm_f32_tiles_kernel, more rows: LDS tiles, a chunk ahead, a wave a quarter of the tile.  One
// 16-byte read from LDS feeds four matrix instructions of 32 clocks, so the matrix cores (157 TFLOP/s
// in float32) are what bounds it: 64 x 64 for many rows; 32 x 32 otherwise, so that a launch of few
// rows still reaches every compute unit's matrix cores, by two teams of four waves with half of K each.
//
// Measured, 4B layer sizes, weights from memory, gemm_tiled (one chain per element on the vector ALUs)
// before: of a step of 3 rows q/k/v 14 us, gate/up 35 (5.7 TB/s), out and down 34 together, the head 247 (6.3)
// where a launch took 615 on average; 270 rows 106 + 79 + 299 + 177 (80 to 90 TFLOP/s); 2048 rows 112 TFLOP/s.
#include "gemm_f32.h"

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
template <int MT>
__device__ __forceinline__ void gemm_f32_rows_body(float* __restrict__ out, const float* x,
                                                   const float* __restrict__ w, int M, int N, int K, long long ldx,
                                                   long long ldw, long long ldo) {
  // per wave two stages of the tile of w; then the ranges' sums, [range][row tile][64 lanes][4]
  __shared__ __attribute__((aligned(1024))) unsigned char lds[GF_RANGES * 2 * GF_TILE_BYTES + GF_RANGES * MT * 1024];
  float* sums = reinterpret_cast<float*>(lds + GF_RANGES * 2 * GF_TILE_BYTES);

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int range = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE);
  const int r = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16;  // first row of w of this workgroup
  const int rows = (N - row0 < 16) ? N - row0 : 16;
  const int chunks = (K + GF_CHUNK - 1) / GF_CHUNK;
  const int c_begin = gf_range_begin(range, chunks), c_end = gf_range_begin(range + 1, chunks);

  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(w + static_cast<size_t>(row0) * ldw), 0,
      static_cast<int>((static_cast<long long>(rows - 1) * ldw + K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(x), 0, static_cast<int>((static_cast<long long>(M - 1) * ldx + K) * 4), 0x00020000);

  // A load brings rows 4 q .. 4 q + 3 of the tile: lane l, for row R = 4 q + l / 16, the 16-byte piece
  // (l % 16) ^ R, which lies at place l % 16 of that row in LDS: operand reads (lane r takes piece
  // 4 s + g of row r) then fall into different groups of banks.
  const int lrow = lane >> 4, lpos = lane & 15;
  unsigned char* stage_base = lds + range * 2 * GF_TILE_BYTES;
  auto issue = [&](int chunk, int stage) {
    const int k0 = chunk * GF_CHUNK;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int R = 4 * q + lrow;
      const int k = k0 + (lpos ^ R) * 4;
      const bool ok = chunk < c_end && R < rows && k < K;
      const unsigned at = static_cast<unsigned>(R) * static_cast<unsigned>(ldw) * 4u + static_cast<unsigned>(k) * 4u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          wres, (GF_LDS(void)*)(stage_base + stage * GF_TILE_BYTES + q * 1024), 16, ok ? at : GF_OOB, 0, 0, 0);
    }
  };
  unsigned piece_at[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) piece_at[s] = (r >> 2) * 1024 + (r & 3) * 256 + (((4 * s + g) ^ r) * 16);

  floatx4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto load_x = [&](floatx4 (&xv)[MT][4], int chunk) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = chunk * GF_CHUNK + 16 * s + 4 * g;
        const int m = 16 * t + r;
        const bool ok = chunk < c_end && m < M && k < K;
        const unsigned at = static_cast<unsigned>(m) * static_cast<unsigned>(ldx) * 4u + static_cast<unsigned>(k) * 4u;
        xv[t][s] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xres, ok ? at : GF_OOB, 0, 0));
      }
  };
  auto turn_of = [&](int chunk, floatx4 (&xv)[MT][4], floatx4 (&x_next)[MT][4], int stage) {
    load_x(x_next, chunk + 1);
    issue(chunk + 1, stage ^ 1);
    gf_wait_loads<4 * MT + 4>();  // all but the loads just sent
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
    // this wave's reads of the stage are over before the next turn's loads overwrite it
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  floatx4 x_even[MT][4], x_odd[MT][4];
  load_x(x_even, c_begin);
  issue(c_begin, 0);
  for (int chunk = c_begin; chunk < c_end; chunk += 2) {
    turn_of(chunk, x_even, x_odd, 0);
    if (chunk + 1 < c_end) turn_of(chunk + 1, x_odd, x_even, 1);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
    *reinterpret_cast<floatx4*>(sums + ((range * MT + t) * PYLON_WAVE + lane) * 4) = acc[t];
  gf_barrier();

  // Wave t now adds row tile t: element (row 16 t + r, column row0 + 4 g + i).
  const bool wide = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
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
    if (wide && n + 3 < N) {
      *reinterpret_cast<floatx4*>(p) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N) p[i] = v[i];
    }
  }
}

template <int MT>
__global__ __launch_bounds__(GF_RANGES* PYLON_WAVE) void gemm_f32_rows_kernel(
    float* __restrict__ out, const float* x, const float* __restrict__ w, int M, int N, int K,
    long long ldx, long long ldw, long long ldo) {
  gemm_f32_rows_body<MT>(out, x, w, M, N, K, ldx, ldw, ldo);
}

// T: tiles of 16 rows and of 16 columns per wave; a workgroup's tile is 32 T by 32 T.  TEAMS: 1, or
// 2 teams of four waves that take half of K each.
template <int T, int TEAMS>
__device__ __forceinline__ void gemm_f32_tiles_body(float* __restrict__ out, const float* __restrict__ x,
                                                    const float* __restrict__ w, int M, int N, int K, long long ldx,
                                                    long long ldw, long long ldo, int m_tiles, int n_tiles) {
  constexpr int SIDE = 32 * T;
  constexpr int STAGE_BYTES = 4 * T * GF_TILE_BYTES;  // 2 T tiles of x, then 2 T of w
  __shared__ __attribute__((aligned(1024))) unsigned char lds[TEAMS * 2 * STAGE_BYTES];

  // Workgroups that share columns of w run on one die (every eighth workgroup), one after the other,
  // so that its cache serves all but the first.
  const int die = blockIdx.x & 7, nth = blockIdx.x >> 3;
  const int mt = nth % m_tiles, nt = (nth / m_tiles) * 8 + die;
  if (nt >= n_tiles) return;
  const int m0 = mt * SIDE, n0 = nt * SIDE;
  const int m_rows = (M - m0 < SIDE) ? M - m0 : SIDE, n_rows = (N - n0 < SIDE) ? N - n0 : SIDE;

  const int lane = threadIdx.x & (PYLON_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE) & 3;
  const int team = __builtin_amdgcn_readfirstlane(threadIdx.x / PYLON_WAVE) >> 2;
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
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
  auto issue = [&](int chunk, int stage) {
    const int k = chunk * GF_CHUNK + lk;
    unsigned char* base = team_lds + stage * STAGE_BYTES + wave * 1024;
    const bool live = chunk < c_end && k < K;
#pragma unroll
    for (int t = 0; t < 2 * T; ++t) {
      const int row = 16 * t + R;
      const unsigned at = static_cast<unsigned>(row) * static_cast<unsigned>(ldx) * 4u + static_cast<unsigned>(k) * 4u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (GF_LDS(void)*)(base + t * GF_TILE_BYTES), 16,
                                               live && row < m_rows ? at : GF_OOB, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2 * T; ++t) {
      const int row = 16 * t + R;
      const unsigned at = static_cast<unsigned>(row) * static_cast<unsigned>(ldw) * 4u + static_cast<unsigned>(k) * 4u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (GF_LDS(void)*)(base + (2 * T + t) * GF_TILE_BYTES), 16,
                                               live && row < n_rows ? at : GF_OOB, 0, 0, 0);
    }
  };
  unsigned piece_at[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) piece_at[s] = (r >> 2) * 1024 + (r & 3) * 256 + (((4 * s + g) ^ r) * 16);

  // of the range under way, of the half under way, of the first half (one team): [column tile][row tile]
  floatx4 acc[T][T], half[T][T], first[T][T];
#pragma unroll
  for (int j = 0; j < T; ++j)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[j][t] = half[j][t] = first[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  issue(c_begin, 0);
  int range = team * (GF_RANGES / 2);
  for (int turn = 0; turn < turns; ++turn) {
    const int c = c_begin + turn, stage = turn & 1;
    // chunk c has landed for every wave, and every wave is past the products of the turn before
    gf_barrier();
    if (turn + 1 < turns) issue(c + 1, stage ^ 1);
    if (c >= c_end) continue;
    const GF_LDS(unsigned char)* xb = (const GF_LDS(unsigned char)*)(team_lds + stage * STAGE_BYTES + wm * T * GF_TILE_BYTES);
    const GF_LDS(unsigned char)* wb =
        (const GF_LDS(unsigned char)*)(team_lds + stage * STAGE_BYTES + (2 * T + wn * T) * GF_TILE_BYTES);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      floatx4 xf[T], wf[T];
#pragma unroll
      for (int t = 0; t < T; ++t) xf[t] = *reinterpret_cast<const GF_LDS(floatx4)*>(xb + t * GF_TILE_BYTES + piece_at[s]);
#pragma unroll
      for (int j = 0; j < T; ++j) wf[j] = *reinterpret_cast<const GF_LDS(floatx4)*>(wb + j * GF_TILE_BYTES + piece_at[s]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
          for (int t = 0; t < T; ++t)
            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][i], xf[t][i], acc[j][t], 0, 0, 0);
    }
    if (gf_range_begin(range + 1, chunks) == c + 1) {  // the range ends with this chunk
      ++range;
#pragma unroll
      for (int j = 0; j < T; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t) {
          half[j][t] += acc[j][t];
          acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (TEAMS == 1 && c + 1 == middle) {
#pragma unroll
      for (int j = 0; j < T; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t) {
          first[j][t] = half[j][t];
          half[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if constexpr (TEAMS == 2) {
    // the second team's half goes to the first through LDS, which nobody reads any more
    gf_barrier();
    floatx4* meet = reinterpret_cast<floatx4*>(lds) + wave * T * T * PYLON_WAVE + lane;
    if (team == 1) {
#pragma unroll
      for (int j = 0; j < T; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t) meet[(j * T + t) * PYLON_WAVE] = half[j][t];
    }
    gf_barrier();
    if (team == 1) return;
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        first[j][t] = half[j][t];
        half[j][t] = meet[(j * T + t) * PYLON_WAVE];
      }
  }

  const bool wide = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int m = m0 + (wm * T + t) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int n = n0 + (wn * T + j) * 16 + 4 * g;
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

template <int T, int TEAMS>
__global__ __launch_bounds__(TEAMS * 256) void gemm_f32_tiles_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                                     const float* __restrict__ w, int M, int N, int K,
                                                                     long long ldx, long long ldw, long long ldo,
                                                                     int m_tiles, int n_tiles) {
  gemm_f32_tiles_body<T, TEAMS>(out, x, w, M, N, K, ldx, ldw, ldo, m_tiles, n_tiles);
}

template <int T, int TEAMS>
static void launch_tiles(float* out, const float* x, const float* w, int M, int N, int K, long long ldx, long long ldw,
                         long long ldo, hipStream_t stream) {
  const int side = 32 * T, m_tiles = (M + side - 1) / side, n_tiles = (N + side - 1) / side;
  const dim3 grid(static_cast<unsigned>((n_tiles + 7) / 8 * 8) * m_tiles), block(TEAMS * 256);
  hipLaunchKernelGGL((gemm_f32_tiles_kernel<T, TEAMS>), grid, block, 0, stream, out, x, w, M, N, K, ldx, ldw, ldo, m_tiles, n_tiles);
}

// Tiles of 64 x 64 for many rows that fill the chip three times over, else of 32 x 32 (us, 64 against
// 32: 2048 rows 2560 x 9728 993, 1014 and 19456 x 2560 1861, 2057; 600 rows 19456 x 2560 591, 628; but
// 400 rows 451, 440, 270 rows 2560 x 9728 245, 177 and 64 rows 230, 73; tiles of 128 x 128: 1487, 2024,
// 606, 596, 743 and 727).  A launch holds less than 2^32 threads: 0 where neither does.
static int gf_side(int M, int N, int units) {
  auto fits = [&](int side, int threads) {
    const long long groups = static_cast<long long>((M + side - 1) / side) * (((N + side - 1) / side + 7) / 8 * 8);
    return groups * threads < (1ll << 32);
  };
  const bool many = M >= 512 && static_cast<long long>((M + 63) / 64) * ((N + 63) / 64) >= 3ll * units;
  if (!many && fits(32, 512)) return 32;
  return fits(64, 256) ? 64 : 0;
}

// The side of the tiles in which a product of these sizes is computed in float32 (units: compute units), 16 for the
// streaming kernel; 0 where gemm_tiled takes it.  Touches no device.
extern "C" int pylon_gemm_f32_plan(int M, int N, int units, int* side) {
  PYLON_REQUIRE(M >= 1 && N >= 1 && units >= 1 && side != nullptr, "gemm_f32_plan: bad arguments");
  *side = M <= GF_ROWS ? 16 : gf_side(M, N, units);
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
    const dim3 grid((N + 15) / 16), block(GF_RANGES * PYLON_WAVE);
    if (M <= 16)
      hipLaunchKernelGGL((gemm_f32_rows_kernel<1>), grid, block, 0, stream, out, x, w, M, N, K, ldx, ldw, ldo);
    else
      hipLaunchKernelGGL((gemm_f32_rows_kernel<2>), grid, block, 0, stream, out, x, w, M, N, K, ldx, ldw, ldo);
    return true;
  }
  const int side = gf_side(M, N, units);
  if (side == 64)
    launch_tiles<2, 1>(out, x, w, M, N, K, ldx, ldw, ldo, stream);
  else if (side == 32)
    launch_tiles<1, 2>(out, x, w, M, N, K, ldx, ldw, ldo, stream);
  return side != 0;
}
