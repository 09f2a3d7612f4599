// The sums of one 256 x 256 tile of x[rows, K] w[columns, K]^T, bfloat16 operands and float32 sums on the matrix cores, by a
// block of eight waves: the loop that the products of many rows are built on (moe_rows.hip, gemm_block.hip).
//
// What bounds it is the matrix pipe, so the loop keeps it fed. The chunk of 64 columns of K of both operands (64 KB) lies in
// LDS twice, the one being multiplied and the one on its way, copied by the memory pipeline (global_load_lds, rows of 128
// bytes with their 16-byte pieces swizzled, so that no read of LDS meets a bank conflict). A wave's part of the tile is
// 128 x 64 in four quarters of 64 x 32, and its loop four steps, one a quarter: read what the quarter needs that is not in
// registers yet (rows for one step in two, columns the other two), ask for a quarter of the chunk after next, then 16
// matrix instructions. The two waves of a SIMD run half a step apart (the eight-wave "ping-pong" schedule that is published
// for products on CDNA, in the HipKittens paper of 2025 among others), held there by a barrier before and after the
// instructions: while one reads, the other multiplies. A quarter of a chunk is asked for as soon as both waves have read the
// one it overwrites, so about 6 steps (3,000 cycles) before it is read, and every wait leaves what came after it under way.
// Measured on MI355X, us (the vendor library's product): 4096 x 4096 x 4096 101 (112), 4096 rows by 55296 x 4096 1,337 (1,387),
// by 4096 x 27648 590 (589): 1.36 to 1.57 PFLOP/s.
#pragma once
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace block_gemm {
constexpr int TILE = 256, HALF = 128, THREADS = 512;
constexpr int KC = 64;                     // columns of K a chunk holds
constexpr int REGION = HALF * KC * 2;      // bytes of 128 rows of a chunk
constexpr int STAGE = 4 * REGION;          // a chunk: columns' first half, rows' first half, the second halves
constexpr int LDS_BYTES = 2 * STAGE;
constexpr int EXTRA = 16;                  // rows a tile may take beyond its 256: what a step's last few rows are not worth a tile for
constexpr int EXTRA_BYTES = EXTRA * KC * 2;
constexpr int XCDS = 8;

// How the eight waves share a tile: a wave has TR tiles of 16 rows and TC of 16 columns of each quarter, so that a quarter is 128 rows by
// 16 TC CW columns. <4, 2>: two waves by four, 256 x 256. <2, 3>: four by two, 256 rows by 192 columns, for products whose tiles of 256 columns
// would leave a round of the compute units partly idle (a chunk costs it 20 reads of LDS for 48 matrix instructions a wave where the other has 24
// for 64, and 0.8 to 0.87 of the time).
template <int TR, int TC>
struct Shape {
  static constexpr int RW = HALF / (16 * TR), CW = 8 / RW, COLS = 16 * TC * CW;      // COLS: columns of a half
};

// [half of the rows][half of the columns][tile of 16 rows][tile of 16 columns]: a lane holds columns 4 (lane / 16) .. + 3 of
// a tile for its row lane % 16
template <int TR, int TC>
struct AccOf {
  f32x4_t v[2][2][TR][TC];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < TR; ++t)
#pragma unroll
          for (int n = 0; n < TC; ++n) v[i][j][t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
};
using Acc = AccOf<4, 2>;

// Where the lane's part of the tile lies: row `row(i, t)` (of 256) of tile t in half i, first of its four columns
// `column(j, n)` (of 2 COLS). Extra rows: of half j of the columns, one tile of 16 a wave (`extra_column(j)`: the lane's first of four; the
// waves that `has_extra` leaves out have none), row lane % 16.
template <int TR, int TC>
struct PlaceOf {
  using S = Shape<TR, TC>;
  int wr, wc, g, c;
  __device__ __forceinline__ PlaceOf()
      : wr(__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) / S::CW), wc(__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) % S::CW),
        g(threadIdx.x % WAVE / 16), c(threadIdx.x % 16) {}
  __device__ __forceinline__ int row(int i, int t) const { return i * HALF + wr * 16 * TR + t * 16 + c; }
  __device__ __forceinline__ int column(int j, int n) const { return j * S::COLS + wc * 16 * TC + n * 16 + 4 * g; }
  __device__ __forceinline__ bool has_extra() const { return wr < TC; }
  __device__ __forceinline__ int extra_column(int j) const { return j * S::COLS + wc * 16 * TC + wr * 16 + 4 * g; }
};
using Place = PlaceOf<4, 2>;

// The extra rows' sums, by half of the columns.
struct ExtraAcc {
  f32x4_t v[2];
  __device__ __forceinline__ void clear() { v[0] = v[1] = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
};

// What a lane copies of each 128 rows of a chunk: rows `copy_row(q)` (q = 0, 1), from `copy_piece(q)` bytes into the chunk's
// 128 bytes of that row.
__device__ __forceinline__ int copy_row(int q) { return q * 64 + threadIdx.x / 8; }
__device__ __forceinline__ uint32_t copy_piece(int q) { return 16 * ((threadIdx.x % 8) ^ ((copy_row(q) / 2) % 8)); }

__device__ __forceinline__ void phase_barrier() {           // (nothing is moved across it)
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Adds the products to acc. `x_at` and `w_at` [half][q]: this lane's byte offsets from x and w of what it copies of the first
// chunk (row and piece). `chunks` (K / 64): even, at least 2. Every wave of the block comes here, with the same `chunks`.
// MORE: 16 extra rows as well (`more`; `more_at`: as x_at, of rows copy_row(0) up to 15; LDS of LDS_BYTES + 2 EXTRA_BYTES). Waves 0 and 1
// then have a copy more under way, and wait for one more than they need.
template <bool MORE, int TR, int TC>
__device__ __forceinline__ void run_with(AccOf<TR, TC>& acc, ExtraAcc& more, char* lds, const bf16_t* x, const bf16_t* w,
                                         const uint32_t (&x_at)[2][2], const uint32_t (&w_at)[2][2], uint32_t more_at, int chunks) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  using S = Shape<TR, TC>;
  const int wr = wave / S::CW, wc = wave % S::CW, late = wave / 4, g = lane / 16, c = lane % 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const auto copy = [&](int which, int chunk) {             // 0: columns' first half, 1: rows' first half, 2, 3: the second ones
    const int h = which / 2;
    const bf16_t* from = ((which & 1) ? x : w) + (int64_t)chunk * KC;
    const uint32_t to = lds0 + (chunk & 1) * STAGE + which * REGION + wave * 1024;
#pragma unroll
    for (int q = 0; q < 2; ++q) load_to_lds16(from, (which & 1) ? x_at[h][q] : w_at[h][q], to + q * 8192);
    if (MORE && which == 1 && wave < 2) load_to_lds16(from, more_at, lds0 + LDS_BYTES + (chunk & 1) * EXTRA_BYTES + wave * 1024);
  };
  uint32_t at[2];                                           // this lane's 16 bytes of its row of a tile, per 32 of the chunk
#pragma unroll
  for (int s = 0; s < 2; ++s) at[s] = c * (KC * 2) + 16 * ((4 * s + g) ^ ((c / 2) % 8));
  const auto read_rows = [&](bf16x8_t (&a)[2][TR], int half, int chunk) {
    const char* p = lds + (chunk & 1) * STAGE + (1 + 2 * half) * REGION + wr * 16 * TR * KC * 2;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < TR; ++t) a[s][t] = *reinterpret_cast<const bf16x8_t*>(p + t * 16 * KC * 2 + at[s]);
  };
  const auto read_columns = [&](bf16x8_t (&b)[2][TC], int half, int chunk) {
    const char* p = lds + (chunk & 1) * STAGE + 2 * half * REGION + wc * 16 * TC * KC * 2;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < TC; ++t) b[s][t] = *reinterpret_cast<const bf16x8_t*>(p + t * 16 * KC * 2 + at[s]);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  bf16x8_t extra[2];
  const auto multiply = [&](f32x4_t (&d)[TR][TC], const bf16x8_t (&a)[2][TR], const bf16x8_t (&b)[2][TC], auto with) {      // with: the extra
    phase_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < TR; ++t)
#pragma unroll
        for (int n = 0; n < TC; ++n) d[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][n], a[s][t], d[t][n], 0, 0, 0);
    constexpr int J = decltype(with)::value;                // rows too, of half J of the columns (2: not)
    if constexpr (MORE && J < 2) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int n = 0; n < TC; ++n)
          if (wr == n) more.v[J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][n], extra[s], more.v[J], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    phase_barrier();
  };
  // in front of the barrier behind which the other wave of the SIMD may ask for what overwrites what was read
  const auto reads_done = [&] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  bf16x8_t a[2][TR], b[2][2][TC];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int which = 0; which < 4; ++which) copy(which, s);
  wait_loads_but<12>();
  phase_barrier();
  read_columns(b[0], 0, 0);
  reads_done();
  phase_barrier();
  if (late == 1) phase_barrier();                           // half a step behind the other four waves
  // P: k % 2, the set of b that holds the columns' first half. T: 0 while chunks are still asked for, 1 the last but one, 2 the
  // last. A step's wait is for what the next step reads: everything but the copies asked for after it, two a step and wave.
  const auto chunk = [&](auto parity, auto tail, int k) {
    constexpr int P = decltype(parity)::value, T = decltype(tail)::value;
    read_rows(a, 0, k);
    if constexpr (MORE)
#pragma unroll
      for (int s = 0; s < 2; ++s) extra[s] = *reinterpret_cast<const bf16x8_t*>(lds + LDS_BYTES + (k & 1) * EXTRA_BYTES + at[s]);
    if constexpr (T == 0) copy(0, k + 2);
    reads_done();
    wait_loads_but<T == 0 ? 12 : (T == 1 ? 10 : 2)>();
    multiply(acc.v[0][0], a, b[P], c0);
    read_columns(b[1 - P], 1, k);
    if constexpr (T == 0) copy(1, k + 2);
    reads_done();
    wait_loads_but<T == 0 ? 12 : (T == 1 ? 8 : 0)>();
    multiply(acc.v[0][1], a, b[1 - P], c1);
    read_rows(a, 1, k);
    if constexpr (T == 0) copy(2, k + 2);
    reads_done();
    wait_loads_but<T == 0 ? 12 : (T == 1 ? 6 : 0)>();
    multiply(acc.v[1][1], a, b[1 - P], c2);
    if constexpr (T < 2) read_columns(b[1 - P], 0, k + 1);
    if constexpr (T == 0) copy(3, k + 2);
    reads_done();
    wait_loads_but<T == 0 ? 12 : (T == 1 ? 4 : 0)>();
    multiply(acc.v[1][0], a, b[P], c2);
  };
  for (int k = 0; k + 2 < chunks; k += 2) {
    chunk(c0, c0, k);
    chunk(c1, c0, k + 1);
  }
  chunk(c0, c1, chunks - 2);
  chunk(c1, c2, chunks - 1);
  if (late == 0) phase_barrier();                           // (as many barriers as the other four waves)
}

__device__ __forceinline__ void run(Acc& acc, char* lds, const bf16_t* x, const bf16_t* w, const uint32_t (&x_at)[2][2],
                                    const uint32_t (&w_at)[2][2], int chunks) {
  ExtraAcc none;
  run_with<false, 4, 2>(acc, none, lds, x, w, x_at, w_at, 0, chunks);
}

// The tile that block `id` takes of `total`, -1: none. Blocks go to the XCDs in turn; each XCD gets a run of neighbouring
// tiles, whose operands then come out of its own L2.
__device__ __forceinline__ int tile_of_block(int id, int total) {
  const int per = total / XCDS, rest = total % XCDS, xcd = id % XCDS, at = id / XCDS;
  return at < per + (xcd < rest) ? xcd * per + min(xcd, rest) + at : -1;
}

// Neighbouring tiles: four row tiles at a time, all their column tiles in order.
__device__ __forceinline__ void row_and_column(int tile, int row_tiles, int col_tiles, int& row, int& col) {
  constexpr int ROWS = 4;
  const int group = tile / (ROWS * col_tiles), in = tile % (ROWS * col_tiles), rows = min(ROWS, row_tiles - group * ROWS);
  row = group * ROWS + in % rows;
  col = in / rows;
}
}  // namespace block_gemm
