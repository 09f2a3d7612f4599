// Products of many rows (prompts) over untiled weights on 256 x 256 tiles (gemm_block.h), bfloat16 with float32 sums: a gated
// feed-forward's first product with the activation in its epilogue, products whose K is cut into shares over the grid, the shares
// added up by whoever reads them, and several products of one size that do not read one another's results.
//
// A step's last row tile takes up to 16 rows beyond its 256: a portion of 512 tokens beside a few decode rows is two tiles high, not three.
#include "common.h"
#include "gemm_block.h"
#include "holon_hip.h"

namespace {
using namespace block_gemm;

enum { SILU, GELU, PARTS, PLAIN };

constexpr int GROUP_MOST = 4;
struct Operands {                    // PLAIN: a product's each; else the first alone
  const bf16_t* x[GROUP_MOST];
  const bf16_t* w[GROUP_MOST];
  void* y[GROUP_MOST];
};

// What a tile gives, from LDS in whole lines: the gated ones bfloat16 y [M, N], 128 columns a tile (the tile's first half of columns are
// gates and the second ups of w [2 N, K]), PARTS float32 y [splits, M, N], PLAIN bfloat16 y [M, N] of `splits` products.
template <int KIND, int TR, int TC>
__global__ void __launch_bounds__(THREADS, 2) gemm_block_kernel(Operands op, int M, int N, int K, int row_tiles, int col_tiles,
                                                                int splits) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES + 2 * EXTRA_BYTES];
  constexpr bool GATED = KIND == SILU || KIND == GELU;
  using S = Shape<TR, TC>;
  static_assert(GATED || S::COLS == HALF, "products in shares: 256 x 256 tiles alone");
  constexpr int COLS = GATED ? S::COLS : TILE;
  const int tiles = row_tiles * col_tiles;
  int tile = tile_of_block(blockIdx.x, tiles * splits);
  if (tile < 0) return;
  const int split = tile / tiles, share = KIND == PLAIN ? K : K / splits, which = KIND == PLAIN ? split : 0;
  const bf16_t *x = op.x[which], *w = op.w[which];
  void* y = op.y[which];
  tile %= tiles;
  int rt, ct;
  row_and_column(tile, row_tiles, col_tiles, rt, ct);
  const int m0 = rt * TILE, n0 = ct * COLS;
  const bool has_more = rt == row_tiles - 1 && M > row_tiles * TILE;      // rows beyond the last tile's 256
  uint32_t x_at[2][2], w_at[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < 2; ++q) {                    // (rows and columns past the last repeat it: nothing of them is written)
      const int r = copy_row(q);
      x_at[h][q] = (uint32_t)((int64_t)min(m0 + h * HALF + r, M - 1) * K * 2) + copy_piece(q);
      const int64_t column = GATED ? (int64_t)h * N + min(n0 + min(r, COLS - 1), N - 1) : min(n0 + h * HALF + r, N - 1);
      w_at[h][q] = (uint32_t)(column * K * 2) + copy_piece(q);
    }
  const uint32_t more_at = (uint32_t)((int64_t)min(m0 + TILE + copy_row(0) % EXTRA, M - 1) * K * 2) + copy_piece(0);
  AccOf<TR, TC> acc;
  ExtraAcc more;
  acc.clear();
  more.clear();
  const int64_t k0 = KIND == PLAIN ? 0 : (int64_t)split * share;
  if (has_more) run_with<true, TR, TC>(acc, more, lds, x + k0, w + k0, x_at, w_at, more_at, share / KC);
  else run_with<false, TR, TC>(acc, more, lds, x + k0, w + k0, x_at, w_at, 0, share / KC);
  const PlaceOf<TR, TC> at;
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  if constexpr (GATED) {
    constexpr int ACT = KIND == GELU, PITCH = COLS * 2 + 16, ROWS = TILE + EXTRA, PIECES = COLS / 8;
    static_assert(ROWS * PITCH <= LDS_BYTES, "a tile's columns");
    const auto gated = [](f32x4_t gate, f32x4_t up) {                      // the roundings of the product and of the gated kernels
      ushort4 o;
      bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        oe[v] = float_to_bf16(Elem<bf16_t>::round(gate_act<ACT, bf16_t>(Elem<bf16_t>::round(gate[v]))) * Elem<bf16_t>::round(up[v]));
      return o;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < TR; ++t)
#pragma unroll
        for (int n = 0; n < TC; ++n)
          *reinterpret_cast<ushort4*>(lds + at.row(i, t) * PITCH + at.column(0, n) * 2) = gated(acc.v[i][0][t][n], acc.v[i][1][t][n]);
    if (has_more && at.has_extra()) *reinterpret_cast<ushort4*>(lds + (TILE + at.c) * PITCH + at.extra_column(0) * 2) = gated(more.v[0], more.v[1]);
    __syncthreads();
    for (int e = threadIdx.x; e < (has_more ? ROWS : TILE) * PIECES; e += THREADS) {
      const int row = e / PIECES, column = n0 + e % PIECES * 8;
      if (m0 + row < M && column < N)
        *reinterpret_cast<uint4*>((bf16_t*)y + (int64_t)(m0 + row) * N + column) =
            *reinterpret_cast<const uint4*>(lds + row * PITCH + e % PIECES * 16);
    }
  } else if constexpr (KIND == PLAIN) {
    constexpr int PITCH = HALF * 2 + 16, ROWS = TILE + EXTRA;      // half of the columns at a time
    const auto rounded = [](f32x4_t v) {
      ushort4 o;
      o.x = float_to_bf16(v[0]); o.y = float_to_bf16(v[1]); o.z = float_to_bf16(v[2]); o.w = float_to_bf16(v[3]);
      return o;
    };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < TR; ++t)
#pragma unroll
          for (int n = 0; n < TC; ++n)
            *reinterpret_cast<ushort4*>(lds + at.row(i, t) * PITCH + at.column(0, n) * 2) = rounded(acc.v[i][j][t][n]);
      if (has_more && at.has_extra()) *reinterpret_cast<ushort4*>(lds + (TILE + at.c) * PITCH + at.extra_column(0) * 2) = rounded(more.v[j]);
      __syncthreads();
      for (int e = threadIdx.x; e < (has_more ? ROWS : TILE) * 16; e += THREADS) {
        const int row = e / 16, column = n0 + j * HALF + e % 16 * 8;
        if (m0 + row < M && column < N)
          *reinterpret_cast<uint4*>((bf16_t*)y + (int64_t)(m0 + row) * N + column) = *reinterpret_cast<const uint4*>(lds + row * PITCH + e % 16 * 16);
      }
      __syncthreads();
    }
  } else {
    constexpr int PITCH = 144;                       // a wave's own 64 rows of 32 columns at a time
    char* mine = lds + wave * (64 * PITCH);
    float* out = (float*)y + (int64_t)split * M * N;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int n = 0; n < 2; ++n)
            *reinterpret_cast<f32x4_t*>(mine + (t * 16 + at.c) * PITCH + n * 64 + at.g * 16) = acc.v[i][j][t][n];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = u * 8 + lane / 8, m = m0 + i * HALF + at.wr * 64 + r, column = n0 + j * HALF + at.wc * 32 + lane % 8 * 4;
          if (m < M && column < N)
            *reinterpret_cast<f32x4_t*>(out + (int64_t)m * N + column) = *reinterpret_cast<const f32x4_t*>(mine + r * PITCH + lane % 8 * 16);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    if (has_more && m0 + TILE + at.c < M)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int column = n0 + at.extra_column(j);
        if (column < N) *reinterpret_cast<f32x4_t*>(out + (int64_t)(m0 + TILE + at.c) * N + column) = more.v[j];
      }
  }
}

constexpr int SLIM = Shape<2, 3>::COLS;      // a gated product's columns a tile in the form of 192

// Whether a gated product's tiles are 192 columns wide (96 gates and their ups): by the rounds of one tile a compute unit that either takes, of
// which the slim one's lasts 0.8 to 0.87 as long. Measured, us, tiles of 256 columns against 192 (rounds): 12,288 x 4,096 at 256 / 520 / 768 /
// 1,400 / 2,048 / 4,096 rows 85 (1) / 115 (1) / 166 (2) / 255 (3) / 280 (3) / 558 (6) and 78 (1) / 97 (1) / 143 (2) / 224 (3) / 300 (4) / 592 (8);
// 8,192 x 2,048 at 400 / 768 / 2,048 41 (1) / 45 (1) / 105 (2) and 34 (1) / 68 (2) / 124 (3); 9,728 x 2,560 at 520 / 1,024 / 1,400 65 (1) / 119
// (2) / 120 (2) and 58 (1) / 104 (2) / 141 (3). Of 80 products the rule's choice is never the slower one by more than 1 %.
bool slim_pays(int row_tiles, int N) {
  const auto rounds = [&](int wide) { return (row_tiles * ((N + wide - 1) / wide) + 255) / 256; };
  return 0.85f * rounds(SLIM) < rounds(HALF);
}

int row_tiles_of(int M) { return M > TILE && M % TILE && M % TILE <= EXTRA ? M / TILE : (M + TILE - 1) / TILE; }
}  // namespace

// Whether the products serve M rows over w [N or 2 N, K] with K in `splits` shares: shares of whole pairs of chunks, offsets of 32 bits.
extern "C" int holon_gemm_block_supported(int M, int N, int K, int gated, int splits) {
  return M >= 1 && N > 0 && N % 16 == 0 && splits >= 1 && K > 0 && K % (128 * splits) == 0 && (int64_t)M * K < (int64_t)1 << 31 &&
         ((int64_t)N * (gated ? 2 : 1)) * K < (int64_t)1 << 31;
}

static int launch_block(int kind, const void* x, const void* w, void* y, int M, int N, int K, int splits, int width, void* stream) {
  const bool gated = kind == SILU || kind == GELU;
  HOLON_CHECK(holon_gemm_block_supported(M, N, K, gated, splits) && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) == 0,
              "gemm (many rows): M=%d N=%d K=%d in %d shares not served", M, N, K, splits);
  const int rows = row_tiles_of(M);
  const bool slim = gated && (width ? width == SLIM : slim_pays(rows, N));
  const int wide = gated ? (slim ? SLIM : HALF) : TILE, cols = (N + wide - 1) / wide;
  const unsigned blocks = (unsigned)(((int64_t)rows * cols * splits + XCDS - 1) / XCDS * XCDS);      // every XCD as many
  hipStream_t s = (hipStream_t)stream;
  const Operands op{{(const bf16_t*)x}, {(const bf16_t*)w}, {y}};
  switch (kind) {
    case SILU:
      if (slim) gemm_block_kernel<SILU, 2, 3><<<blocks, THREADS, 0, s>>>(op, M, N, K, rows, cols, splits);
      else gemm_block_kernel<SILU, 4, 2><<<blocks, THREADS, 0, s>>>(op, M, N, K, rows, cols, splits);
      break;
    case GELU:
      if (slim) gemm_block_kernel<GELU, 2, 3><<<blocks, THREADS, 0, s>>>(op, M, N, K, rows, cols, splits);
      else gemm_block_kernel<GELU, 4, 2><<<blocks, THREADS, 0, s>>>(op, M, N, K, rows, cols, splits);
      break;
    default: gemm_block_kernel<PARTS, 4, 2><<<blocks, THREADS, 0, s>>>(op, M, N, K, rows, cols, splits); break;
  }
  HOLON_LAUNCH_OK();
  return 0;
}

// y [M, N] = act(x gates^T) * (x ups^T) over w [2 N, K] (gates, then ups); act 0 silu, 1 gelu in its tanh form.
extern "C" int holon_gemm_block_glu_bf16(const void* x, const void* w, void* y, int M, int N, int K, int act, void* stream) {
  return launch_block(act ? GELU : SILU, x, w, y, M, N, K, 1, 0, stream);
}
// The same with the columns of y a tile has, 128 or 96, named (0: by the rule above). The sums are the same.
extern "C" int holon_gemm_block_glu_width_bf16(const void* x, const void* w, void* y, int M, int N, int K, int act, int width, void* stream) {
  HOLON_CHECK(width == 0 || width == HALF || width == SLIM, "gemm (many rows): tiles of %d columns", width);
  return launch_block(act ? GELU : SILU, x, w, y, M, N, K, 1, width, stream);
}

// Whether a product in shares takes this form where gemm_tiles.hip's would serve it too: with its last rows filled up that one's blocks
// read both operands twice as often. Measured with the add + norm that reads the parts, in as many shares, us, that form against this:
// 4096 x 12288 at 129 / 300 / 520 / 768 / 1,024 rows 44 / 64 / 96 / 105 / 117 and 41 / 54 / 64 / 83 / 96; 5120 x 25600 at 256 / 512 /
// 1,000 rows 121 / 172 / 297 and 93 / 148 / 250; 2048 x 8192 at 129 / 512 / 1,000 rows 28 / 35 / 57 and 27 / 35 / 49. A K that eight shares
// of whole pairs of chunks do not divide stays with the other up to 512 rows (2560 x 9728 at 256 / 400 / 600 / 1,000 rows, eight shares there
// against four here: 35 / 50 / 56 / 90 and 48 / 52 / 56 / 63).
extern "C" int holon_gemm_block_parts_serves(int M, int N, int K, int splits) {
  return M > 128 && M <= 1024 && N % TILE == 0 && holon_gemm_block_supported(M, N, K, 0, splits) && (K % 1024 == 0 || M > 512);
}
// The number of shares, a power of two up to eight, that is done first (0: none is served): rounds of a tile's loop a compute unit, and the
// parts' traffic (of 24 products of three widths the choice is at most 6 % from the best).
extern "C" int holon_gemm_block_parts_splits(int M, int N, int K) {
  const int tiles = row_tiles_of(M) * ((N + TILE - 1) / TILE);
  int best = 0;
  float least = 0.f;
  for (int splits = 1; splits <= 8; splits *= 2) {
    if (!holon_gemm_block_parts_serves(M, N, K, splits)) continue;
    const float us = (float)((tiles * splits + 255) / 256) * (0.0203f * K / splits + 6.f) + 1.45e-6f * splits * M * N;
    if (best == 0 || us < least) { best = splits; least = us; }
  }
  return best;
}

// parts [splits, M, N] (float32) = x[:, share s of K] w[:, share s of K]^T.
extern "C" int holon_gemm_block_parts_bf16(const void* x, const void* w, void* parts, int M, int N, int K, int splits, void* stream) {
  return launch_block(PARTS, x, w, parts, M, N, K, splits, 0, stream);
}

// `count` (up to 4) products of one size in one launch, where one of them would leave most compute units without a tile (four of 2,048 x 2,048
// at 2,048 rows are a tile for each of the 256 units: 63 us, 1.1 PFLOP/s; one such product by itself takes 37): y_i [M, N] (bfloat16) = x_i [M, K] w_i [N, K]^T. `operands`: count pointers x, then w,
// then y.
extern "C" int holon_gemm_block_group_bf16(const int64_t* operands, int count, int M, int N, int K, void* stream) {
  HOLON_CHECK(count >= 1 && count <= GROUP_MOST && holon_gemm_block_supported(M, N, K, 0, 1),
              "gemm (many rows, several): %d products of M=%d N=%d K=%d not served", count, M, N, K);
  Operands op{};
  for (int i = 0; i < count; ++i) {
    op.x[i] = (const bf16_t*)operands[i];
    op.w[i] = (const bf16_t*)operands[count + i];
    op.y[i] = (void*)operands[2 * count + i];
    HOLON_CHECK(op.x[i] && op.w[i] && op.y[i] && ((operands[i] | operands[count + i] | operands[2 * count + i]) & 15) == 0,
                "gemm (many rows, several): operands off 16 bytes");
  }
  const int rows = row_tiles_of(M), cols = (N + TILE - 1) / TILE;
  const unsigned blocks = (unsigned)(((int64_t)rows * cols * count + XCDS - 1) / XCDS * XCDS);
  gemm_block_kernel<PLAIN, 4, 2><<<blocks, THREADS, 0, (hipStream_t)stream>>>(op, M, N, K, rows, cols, count);
  HOLON_LAUNCH_OK();
  return 0;
}
