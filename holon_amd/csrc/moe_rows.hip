// The experts of a mixture for steps of many rows (prompts), bfloat16: every expert's products over the rows that chose it
// alone, where the products over all experts multiply every row by every expert and add zeros (2 of 8 experts beside a
// shared one: three times the products). Four launches after the router:
//   lists   which rows chose an expert, in their order, and where a row stands among its own choices (a block an expert)
//   up      tiles of 256 of an expert's rows, gathered, against 128 gates and the same 128 ups (or 256 ups): the activation
//           and the weight in the epilogue, rows of the expert's own -> act
//   down    tiles of act against the expert's columns of the second weight -> a row's part from that expert, float32
//   add     a row's parts in the experts' order, rounded once
// The shared expert's rows are all rows; its tiles come first in `up`'s and `down`'s launches. Which tile a block takes is
// read from the lists on the device, so the launches are the same whatever was chosen: the grid is the most tiles there can
// be, and what is left over ends at once.
//
// Bound by the matrix pipe (gemm_block.h). 4,096 rows of 4,096, 8 experts of 3,072 of which a row takes two, beside a shared
// one: 0.93 TFLOP where the products over all take 2.78.
#include <algorithm>

#include "common.h"
#include "gemm_block.h"
#include "holon_hip.h"
#include "moe_lists.h"

namespace {
using namespace block_gemm;
using namespace moe_lists;
// act of an expert's rows (routed: [rows * top, ff] in the order of the lists) and of the shared expert ([rows, shared]).
template <bool GATED>
__global__ void __launch_bounds__(THREADS, 2) moe_up_rows_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                 bf16_t* __restrict__ act, bf16_t* __restrict__ act_shared,
                                                                 MoeRows p) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  constexpr int COLS = GATED ? HALF : TILE;          // columns of act a tile gives
  const int K = p.hidden, cols = p.experts * p.ff + p.shared;
  RowTile rows;
  const int routed = find_rows<TILE>(p, -1, rows);
  const int per_routed = (p.ff + COLS - 1) / COLS, per_shared = (p.shared + COLS - 1) / COLS;
  const int shared_tiles = p.shared ? (p.rows + TILE - 1) / TILE : 0;
  const int tile = tile_of_block(blockIdx.x, routed * per_routed + shared_tiles * per_shared);
  if (tile < 0) return;
  const int first = shared_tiles * per_shared;
  const bool is_routed = tile >= first;
  int rt, ct;
  if (is_routed) {
    row_and_column(tile - first, routed, per_routed, rt, ct);
    find_rows<TILE>(p, rt, rows);
  } else {
    row_and_column(tile, shared_tiles, per_shared, rt, ct);
    rows = RowTile{p.experts, 0, p.rows, rt * TILE};
  }
  const int width = is_routed ? p.ff : p.shared;     // columns the expert has
  const int* list = p.lists + (int64_t)rows.expert * p.rows;
  const auto token = [&](int i) { return is_routed ? list[i] & ((1 << TOKEN_BITS) - 1) : i; };
  const int64_t w_row = (int64_t)rows.expert * p.ff + ct * COLS;
  uint32_t x_at[2][2], w_at[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < 2; ++q) {                    // (rows and columns past the last repeat it: nothing of them is written)
      const int r = copy_row(q), last = width - 1 - ct * COLS;
      x_at[h][q] = (uint32_t)((int64_t)token(min(rows.row0 + h * HALF + r, rows.count - 1)) * K * 2) + copy_piece(q);
      const int64_t column = GATED ? (int64_t)h * cols + min(r, last) : min(h * HALF + r, last);
      w_at[h][q] = (uint32_t)(column * K * 2) + copy_piece(q);
    }
  Acc acc;
  acc.clear();
  run(acc, lds, x, w + w_row * K, x_at, w_at, K / KC);
  const Place at;
  // through LDS, so that a row's columns leave as whole lines (a lane holds four of them): 128 columns in rows of 256 bytes and
  // a piece, twice where a tile gives 256
  constexpr int PITCH = HALF * 2 + 16;
  static_assert(TILE * PITCH <= LDS_BYTES, "a tile's half of the columns");
  bf16_t* out = is_routed ? act + (int64_t)rows.first * p.ff : act_shared;
#pragma unroll
  for (int j = 0; j < COLS / HALF; ++j) {
    if (j > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = rows.row0 + at.row(i, t);
        const int col = is_routed ? rows.expert : p.shared_col;
        const float weight = r < rows.count && col >= 0 ? p.weights[(int64_t)token(r) * p.stride + col] : 1.f;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          ushort4 o;
          bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
          for (int v = 0; v < 4; ++v) {              // the roundings of moe_gate and of moe_relu2
            float z;
            if constexpr (GATED) {
              const float gate = Elem<bf16_t>::round(acc.v[i][0][t][n][v]), up = Elem<bf16_t>::round(acc.v[i][1][t][n][v]);
              z = Elem<bf16_t>::round(Elem<bf16_t>::round(silu<bf16_t>(gate)) * up) * weight;
            } else {
              const float up = fmaxf(Elem<bf16_t>::round(acc.v[i][j][t][n][v]), 0.f);
              z = up * up * weight;
            }
            oe[v] = float_to_bf16(weight != 0.f ? z : 0.f);
          }
          *reinterpret_cast<ushort4*>(lds + at.row(i, t) * PITCH + at.column(0, n) * 2) = o;
        }
      }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TILE * 16 / THREADS; ++u) {
      const int row = u * (THREADS / 16) + threadIdx.x / 16, r = rows.row0 + row, column = ct * COLS + j * HALF + threadIdx.x % 16 * 8;
      if (r < rows.count && column < width)
        *reinterpret_cast<uint4*>(out + (int64_t)r * width + column) =
            *reinterpret_cast<const uint4*>(lds + row * PITCH + threadIdx.x % 16 * 16);
    }
  }
}

// parts [rows * top + rows, hidden] float32: an expert's share of the results of its rows, in the order of the lists, then the
// shared expert's; which of them are a row's goes into `slots`.
__global__ void __launch_bounds__(THREADS, 2) moe_down_rows_kernel(const bf16_t* __restrict__ act,
                                                                   const bf16_t* __restrict__ act_shared,
                                                                   const bf16_t* __restrict__ w, float* __restrict__ parts,
                                                                   MoeRows p) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int N = p.hidden;
  const int64_t cols = (int64_t)p.experts * p.ff + p.shared;
  RowTile rows;
  const int routed = find_rows<TILE>(p, -1, rows), per = (N + TILE - 1) / TILE;
  const int shared_tiles = p.shared ? (p.rows + TILE - 1) / TILE : 0;
  const int tile = tile_of_block(blockIdx.x, (routed + shared_tiles) * per);
  if (tile < 0) return;
  const bool is_routed = tile >= shared_tiles * per;
  int rt, ct;
  if (is_routed) {
    row_and_column(tile - shared_tiles * per, routed, per, rt, ct);
    find_rows<TILE>(p, rt, rows);
  } else {
    row_and_column(tile, shared_tiles, per, rt, ct);
    rows = RowTile{p.experts, 0, p.rows, rt * TILE};
  }
  const int K = is_routed ? p.ff : p.shared;
  uint32_t x_at[2][2], w_at[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int r = h * HALF + copy_row(q);
      x_at[h][q] = (uint32_t)((int64_t)min(rows.row0 + r, rows.count - 1) * K * 2) + copy_piece(q);
      w_at[h][q] = (uint32_t)(min(ct * TILE + r, N - 1) * cols * 2) + copy_piece(q);
    }
  Acc acc;
  acc.clear();
  run(acc, lds, is_routed ? act + (int64_t)rows.first * K : act_shared, w + (int64_t)rows.expert * p.ff, x_at, w_at, K / KC);
  const Place at;
  float* out = parts + ((int64_t)(is_routed ? rows.first : p.rows * (int64_t)p.top)) * N;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int r = rows.row0 + at.row(i, t);
      if (r >= rows.count) continue;
      if (is_routed && ct == 0 && at.wc == 0 && at.g == 0) {      // (one lane a row)
        const uint32_t entry = p.lists[(int64_t)rows.expert * p.rows + r];
        p.slots[(int64_t)(entry & ((1u << TOKEN_BITS) - 1)) * p.top + (entry >> TOKEN_BITS)] = rows.first + r;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const int column = ct * TILE + at.column(j, n);
          if (column < N) *reinterpret_cast<f32x4_t*>(out + (int64_t)r * N + column) = acc.v[i][j][t][n];
        }
    }
}

}  // namespace

// Whether the products serve `rows` rows of `hidden`: sizes the loop's chunks divide, offsets that 32 bits hold.
extern "C" int holon_moe_rows_supported(int rows, int hidden, int experts, int top, int ff, int shared) {
  const int64_t cols = (int64_t)experts * ff + shared;
  const auto deep = [](int k) { return k >= 128 && k % 128 == 0; };
  return rows >= 1 && rows < 1 << TOKEN_BITS && deep(hidden) && deep(ff) && (shared == 0 || deep(shared)) && experts >= 1 &&
         experts <= MAX_EXPERTS && top >= 1 && top <= experts && top <= MAX_TOP && (int64_t)rows * top * ff < (int64_t)1 << 31 &&
         (int64_t)rows * hidden < (int64_t)1 << 31 && (int64_t)rows * shared < (int64_t)1 << 31 &&
         (cols + HALF) * hidden < (int64_t)1 << 31 && (int64_t)experts * rows < (int64_t)1 << 31;
}

// y [rows, hidden] = the experts' and the shared expert's results of x, over the weights [gates; ups] or [ups] (rows as they
// come, `up`) and the second projections side by side (`down` [hidden, experts ff + shared]). Scratch: lists [experts (rows +
// 1) + rows top] whole numbers, act [rows (top ff + shared)], parts [rows (top + 1), hidden] float32.
extern "C" int holon_moe_rows_bf16(const void* x, const void* up, const void* down, void* y, int* lists, void* act, float* parts,
                                   int rows, int hidden, int experts, int top, int ff, int shared, int gated,
                                   const float* weights, int wstride, int shared_col, void* stream) {
  HOLON_CHECK(holon_moe_rows_supported(rows, hidden, experts, top, ff, shared) && wstride >= experts && shared_col < wstride &&
                  (((uintptr_t)x | (uintptr_t)up | (uintptr_t)down | (uintptr_t)y | (uintptr_t)act | (uintptr_t)parts) & 15) == 0,
              "moe (many rows): %d rows of %d, %d experts of %d (%d a row), %d shared columns not served", rows, hidden, experts,
              ff, top, shared);
  hipStream_t s = (hipStream_t)stream;
  MoeRows p{weights, wstride, rows, hidden, experts, top, ff, shared, shared_col, lists, nullptr, nullptr};
  p.lists = p.counts + experts;
  p.slots = p.lists + (int64_t)experts * rows;
  bf16_t* act_routed = (bf16_t*)act;
  bf16_t* act_shared = act_routed + (int64_t)rows * top * ff;
  const auto tiles = [](int64_t n, int of) { return (n + of - 1) / of; };
  // an expert's last tile is partly empty, and no more tiles than that
  const int64_t routed = std::min<int64_t>((int64_t)rows * top / TILE + experts, (int64_t)experts * tiles(rows, TILE));
  const int cols = gated ? HALF : TILE;
  const int64_t up_tiles = routed * tiles(ff, cols) + tiles(rows, TILE) * tiles(shared, cols);
  const int64_t down_tiles = (routed + (shared ? tiles(rows, TILE) : 0)) * tiles(hidden, TILE);
  const auto blocks = [&](int64_t n) { return (unsigned)(tiles(n, XCDS) * XCDS); };      // every XCD as many
  make_lists(p, s);
  if (gated) moe_up_rows_kernel<true><<<blocks(up_tiles), THREADS, 0, s>>>((const bf16_t*)x, (const bf16_t*)up, act_routed, act_shared, p);
  else moe_up_rows_kernel<false><<<blocks(up_tiles), THREADS, 0, s>>>((const bf16_t*)x, (const bf16_t*)up, act_routed, act_shared, p);
  moe_down_rows_kernel<<<blocks(down_tiles), THREADS, 0, s>>>(act_routed, act_shared, (const bf16_t*)down, parts, p);
  add_parts(p, parts, (bf16_t*)y, s);
  HOLON_LAUNCH_OK();
  return 0;
}
