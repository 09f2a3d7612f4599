// The experts of a mixture in float32, over the rows that chose them: few rows (decode steps) and many (prompts). The products over
// all experts multiply every row by every expert and add zeros; 2 of 8 experts beside a shared one need a third of them, and few
// rows a third of the weights. A row's result is the same bits in both forms: an expert's sums have the order of gemm_f32.h over the
// expert's own columns, and the experts' parts are added in their order, the shared expert's last.
//
// Few rows are bound by memory (blocks of experts that no row chose end at once), many by the matrix cores (tiles of 64 of an expert's
// rows, see moe_rows.hip for the launches). 8 experts of 2,048 x 2,048 (squared ReLU, 2 a row) beside a shared one, us against the
// products over all: one row 53 / 110, 700 rows 460 / 1,199, its two products since then 443 -> 419 (3.1e-7 from 64 bits where those are 4.8e-7).
#include <algorithm>

#include "gemm_f32.h"
#include "holon_hip.h"
#include "moe_lists.h"

namespace {
using namespace f32_sums;
using namespace moe_lists;

// One value of act from the products of its column, as moe_gate and moe_relu2 have it.
template <bool GATED>
__device__ __forceinline__ float weighed(float gate, float up, float weight) {
  if (weight == 0.f) return 0.f;
  if constexpr (GATED) return silu<float>(gate) * up * weight;
  const float z = fmaxf(up, 0.f);
  return z * z * weight;
}

__device__ __forceinline__ float weight_of(const MoeRows& p, int row, int expert) {      // (expert == experts: the shared one)
  const int col = expert < p.experts ? expert : p.shared_col;
  return col >= 0 ? p.weights[(int64_t)row * p.stride + col] : 1.f;
}

// Up to 16 rows. A block 16 columns of act [rows, experts ff + shared]: K in shares over its 16 waves. Blocks of a routed expert that no
// row chose end at once and write nothing.
template <bool GATED>
__global__ void __launch_bounds__(SHARES * WAVE) moe_up_few_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                   float* __restrict__ act, MoeRows p) {
  constexpr int NT = GATED ? 2 : 1;
  __shared__ f32x4_t part[SHARES][NT][WAVE];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  const int n0 = blockIdx.x * 16, cols = p.experts * p.ff + p.shared, expert = min(n0 / p.ff, p.experts);
  const float weight = c < p.rows ? weight_of(p, c, expert) : 0.f;
  if (expert < p.experts && __ballot(weight != 0.f) == 0) return;
  const int K = p.hidden, share = share_length(K), first = wave * share;
  const float *wr[NT], *xr[1] = {x + (int64_t)min(c, p.rows - 1) * K};
#pragma unroll
  for (int u = 0; u < NT; ++u) wr[u] = w + ((int64_t)u * cols + n0 + c) * K;
  f32x4_t acc[1][NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) acc[0][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  share_sums<1, NT, GATED ? 1 : 2, true>(acc, wr, xr, first, min(K, first + share));
#pragma unroll
  for (int u = 0; u < NT; ++u) part[wave][u][lane] = acc[0][u];
  __syncthreads();
  if (wave > 0 || c >= p.rows) return;
  f32x4_t sum[NT], out;
#pragma unroll
  for (int u = 0; u < NT; ++u) sum[u] = sum_shares([&](int i) { return part[i][u][lane]; });
#pragma unroll
  for (int i = 0; i < 4; ++i) out[i] = weighed<GATED>(sum[0][i], sum[NT - 1][i], weight);
  *reinterpret_cast<f32x4_t*>(act + (int64_t)c * cols + n0 + 4 * g) = out;
}

// y [rows, hidden]: a block eight columns (half a tile, see gemm_f32.hip), expert by expert over those that a row chose.
constexpr int AT_ONCE = 3;                       // experts whose shares lie in LDS at a time
__global__ void __launch_bounds__(SHARES * WAVE) moe_down_few_f32_kernel(const float* __restrict__ act, const float* __restrict__ w,
                                                                     float* __restrict__ y, MoeRows p) {
  __shared__ f32x4_t part[AT_ONCE][SHARES][WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  const int n0 = blockIdx.x * 8;
  const int64_t cols = (int64_t)p.experts * p.ff + p.shared;
  const float* wr = w + (int64_t)(n0 + c % 8) * cols;
  const float* xr = act + (int64_t)min(c, p.rows - 1) * cols;
  f32x4_t total = {0.f, 0.f, 0.f, 0.f};
  int held = 0;
  const auto add_held = [&]() {
    __syncthreads();
    if (wave == 0)
      for (int e = 0; e < held; ++e) total += sum_shares([&](int i) { return part[e][i][lane]; });
    __syncthreads();
    held = 0;
  };
  const auto one = [&](int64_t from, int K) {
    const int share = share_length(K), first = wave * share;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    half_sums<2, true>(acc, wr + from, xr + from, first, min(K, first + share));
    part[held][wave][lane] = acc;
    if (++held == AT_ONCE) add_held();
  };
  for (int e0 = 0; e0 < p.experts; e0 += WAVE) {           // (the same in every wave)
    bool any = false;
    if (e0 + lane < p.experts)
      for (int m = 0; m < p.rows; ++m) any |= p.weights[(int64_t)m * p.stride + e0 + lane] != 0.f;
    for (uint64_t mask = __ballot(any); mask != 0; mask &= mask - 1) one((int64_t)(e0 + __builtin_ctzll(mask)) * p.ff, p.ff);
  }
  if (p.shared) one((int64_t)p.experts * p.ff, p.shared);
  if (held > 0) add_held();
  if (wave == 0 && c < p.rows && g < 2) *reinterpret_cast<f32x4_t*>(y + (int64_t)c * p.hidden + n0 + 4 * g) = total;
}

constexpr int ROWS = 64, XCDS = 8;
// Which tile a block takes: of all experts' rows (`rows`; not `routed`: the shared one's, which come first) and the tile of columns `col`.
// take: false where there is none for it; `routed_cols`, `shared_cols`: tiles of columns a routed expert and the shared one have.
struct Taken {
  RowTile rows;
  bool routed;
  int col;
};
__device__ __forceinline__ bool take(const MoeRows& p, int routed_cols, int shared_cols, Taken& out) {
  const int routed = find_rows<ROWS>(p, -1, out.rows), shared_tiles = p.shared ? (p.rows + ROWS - 1) / ROWS : 0;
  const int total = shared_tiles * shared_cols + routed * routed_cols;
  // (blocks go to the XCDs in turn; each gets a run of neighbouring tiles)
  const int per = total / XCDS, rest = total % XCDS, xcd = blockIdx.x % XCDS, at = blockIdx.x / XCDS;
  if (at >= per + (xcd < rest)) return false;
  int tile = xcd * per + min(xcd, rest) + at;
  out.routed = tile >= shared_tiles * shared_cols;
  if (out.routed) {                                        // row tiles of one set of columns side by side: they share its weights
    tile -= shared_tiles * shared_cols;
    out.col = tile / routed;
    find_rows<ROWS>(p, tile % routed, out.rows);
  } else {
    out.col = tile / shared_tiles;
    out.rows = RowTile{p.experts, 0, p.rows, tile % shared_tiles * ROWS};
  }
  return true;
}

// act of an expert's rows (routed: [rows * top, ff] in the order of the lists) and of the shared one ([rows, shared]): tiles of 64 rows
// by 64 columns, GATED 32 gates and the same 32 ups.
template <bool GATED, How HOW>
__global__ void __launch_bounds__(256, HOW == DIRECT ? 5 : 1) moe_up_rows_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              float* __restrict__ act, float* __restrict__ act_shared, MoeRows p) {
  __shared__ __attribute__((aligned(16))) Stage<1, 2, 2> stage;
  constexpr int COLS = GATED ? 32 : 64;
  const auto tiles = [](int n) { return (n + COLS - 1) / COLS; };
  Taken t;
  if (!take(p, tiles(p.ff), tiles(p.shared), t)) return;
  const int width = t.routed ? p.ff : p.shared, K = p.hidden, r0 = threadIdx.x / 8, n0 = t.col * COLS;
  const int64_t cols = (int64_t)p.experts * p.ff + p.shared, w0 = (int64_t)t.rows.expert * p.ff;
  const int* list = p.lists + (int64_t)t.rows.expert * p.rows;
  const auto token = [&](int i) { return t.routed ? list[i] & ((1 << TOKEN_BITS) - 1) : i; };
  const float *xr[2], *wr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xr[i] = x + (int64_t)token(min(t.rows.row0 + r0 + 32 * i, t.rows.count - 1)) * K;
    wr[i] = GATED ? w + (i * cols + w0 + min(n0 + r0, width - 1)) * K : w + (w0 + min(n0 + r0 + 32 * i, width - 1)) * K;
  }
  float* out = t.routed ? act + (int64_t)t.rows.first * p.ff : act_shared;
  if constexpr (!GATED) {
    tile_sums<1, 2, 2, HOW>(stage, xr, wr, K, [&](f32x4_t sum, int row, int column) {
      const int r = t.rows.row0 + row;
      if (r >= t.rows.count || n0 + column >= width) return;
      const float weight = weight_of(p, token(r), t.rows.expert);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] = weighed<false>(0.f, sum[i], weight);
      *reinterpret_cast<f32x4_t*>(out + (int64_t)r * width + n0 + column) = sum;
    });
  } else {
    float* both = &stage[0][0][0];                      // [64 rows][64 columns and 4]: gates, then ups
    static_assert(sizeof(stage) >= ROWS * 68 * sizeof(float), "a tile's gates and ups");
    tile_sums<1, 2, 2, HOW>(stage, xr, wr, K, [&](f32x4_t sum, int row, int column) {      // (behind the last barrier of the sums)
      *reinterpret_cast<f32x4_t*>(both + row * 68 + column) = sum;
    });
    __syncthreads();
    for (int e = threadIdx.x; e < ROWS * 8; e += 256) {
      const int row = e / 8, column = e % 8 * 4, r = t.rows.row0 + row;
      if (r >= t.rows.count || n0 + column >= width) continue;
      const float weight = weight_of(p, token(r), t.rows.expert);
      f32x4_t v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = weighed<true>(both[row * 68 + column + i], both[row * 68 + 32 + column + i], weight);
      *reinterpret_cast<f32x4_t*>(out + (int64_t)r * width + n0 + column) = v;
    }
  }
}

// parts [rows * top + rows, hidden]: an expert's share of the results of its rows, then the shared expert's; slots as in moe_rows.hip.
template <How HOW>
__global__ void __launch_bounds__(256, HOW == DIRECT ? 5 : 1) moe_down_rows_f32_kernel(const float* __restrict__ act, const float* __restrict__ act_shared,
                                                                const float* __restrict__ w, float* __restrict__ parts, MoeRows p) {
  __shared__ __attribute__((aligned(16))) Stage<1, 2, 2> stage;
  const int per = (p.hidden + 63) / 64;
  Taken t;
  if (!take(p, per, per, t)) return;
  const int K = t.routed ? p.ff : p.shared, r0 = threadIdx.x / 8, n0 = t.col * 64;
  const int64_t cols = (int64_t)p.experts * p.ff + p.shared;
  const float* from = t.routed ? act + (int64_t)t.rows.first * K : act_shared;
  const float *xr[2], *wr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xr[i] = from + (int64_t)min(t.rows.row0 + r0 + 32 * i, t.rows.count - 1) * K;
    wr[i] = w + min(n0 + r0 + 32 * i, p.hidden - 1) * cols + (int64_t)t.rows.expert * p.ff;
  }
  if (t.routed && t.col == 0 && threadIdx.x < ROWS && t.rows.row0 + (int)threadIdx.x < t.rows.count) {
    const int r = t.rows.row0 + threadIdx.x;
    const uint32_t entry = p.lists[(int64_t)t.rows.expert * p.rows + r];
    p.slots[(int64_t)(entry & ((1u << TOKEN_BITS) - 1)) * p.top + (entry >> TOKEN_BITS)] = t.rows.first + r;
  }
  float* out = parts + (int64_t)(t.routed ? t.rows.first : (int64_t)p.rows * p.top) * p.hidden;
  tile_sums<1, 2, 2, HOW>(stage, xr, wr, K, [&](f32x4_t sum, int row, int column) {
    const int r = t.rows.row0 + row;
    if (r < t.rows.count && n0 + column < p.hidden) *reinterpret_cast<f32x4_t*>(out + (int64_t)r * p.hidden + n0 + column) = sum;
  });
}
}  // namespace

extern "C" int holon_moe_f32_supported(int rows, int hidden, int experts, int top, int ff, int shared) {
  const int64_t cols = (int64_t)experts * ff + shared;
  return rows >= 1 && rows < 1 << TOKEN_BITS && hidden > 0 && hidden % 16 == 0 && ff > 0 && ff % 16 == 0 && shared >= 0 &&
         shared % 16 == 0 && experts >= 1 && experts <= MAX_EXPERTS && top >= 1 && top <= experts && top <= MAX_TOP &&
         cols * 2 < (int64_t)1 << 31 && (int64_t)experts * rows < (int64_t)1 << 31 && (int64_t)rows * top < (int64_t)1 << 31 &&
         ((int64_t)rows * top / ROWS + experts + (rows + ROWS - 1) / ROWS) * ((cols > hidden ? cols : hidden) / 32 + 1) < (int64_t)1 << 31;
}

// y [rows, hidden]. Up to 16 rows: act [rows, experts ff + shared] (lists and parts are not read). More: lists [experts (rows + 1) + rows
// top] whole numbers, act [rows (top ff + shared)], parts [rows (top + 1), hidden].
extern "C" int holon_moe_f32(const void* x, const void* up, const void* down, void* y, int* lists, void* act, float* parts, int rows,
                             int hidden, int experts, int top, int ff, int shared, int gated, const float* weights, int wstride,
                             int shared_col, void* stream) {
  HOLON_CHECK(holon_moe_f32_supported(rows, hidden, experts, top, ff, shared) && wstride >= experts && shared_col < wstride &&
                  (((uintptr_t)x | (uintptr_t)up | (uintptr_t)down | (uintptr_t)y | (uintptr_t)act | (uintptr_t)parts) & 15) == 0,
              "moe (float32): %d rows of %d, %d experts of %d (%d a row), %d shared columns not served", rows, hidden, experts, ff, top,
              shared);
  hipStream_t s = (hipStream_t)stream;
  MoeRows p{weights, wstride, rows, hidden, experts, top, ff, shared, shared_col, lists, nullptr, nullptr};
  const float *xf = (const float*)x, *wu = (const float*)up, *wd = (const float*)down;
  float* a = (float*)act;
  const int64_t cols = (int64_t)experts * ff + shared;
  if (rows <= 16) {
    if (gated) moe_up_few_f32_kernel<true><<<(unsigned)(cols / 16), SHARES * WAVE, 0, s>>>(xf, wu, a, p);
    else moe_up_few_f32_kernel<false><<<(unsigned)(cols / 16), SHARES * WAVE, 0, s>>>(xf, wu, a, p);
    moe_down_few_f32_kernel<<<hidden / 8, SHARES * WAVE, 0, s>>>(a, wd, (float*)y, p);
    HOLON_LAUNCH_OK();
    return 0;
  }
  p.lists = p.counts + experts;
  p.slots = p.lists + (int64_t)experts * rows;
  float* act_shared = a + (int64_t)rows * top * ff;
  const auto tiles = [](int64_t n, int of) { return (n + of - 1) / of; };
  const int64_t routed = std::min<int64_t>((int64_t)rows * top / ROWS + experts, (int64_t)experts * tiles(rows, ROWS));
  const int64_t shared_rows = shared ? tiles(rows, ROWS) : 0;
  const int width = gated ? 32 : 64;
  const auto blocks = [&](int64_t n) { return (unsigned)(tiles(n, XCDS) * XCDS); };      // every XCD as many
  const unsigned up_blocks = blocks(routed * tiles(ff, width) + shared_rows * tiles(shared, width));
  make_lists(p, s);
#define UP(GATED, HOW) moe_up_rows_f32_kernel<GATED, HOW><<<up_blocks, 256, 0, s>>>(xf, wu, a, act_shared, p)
  if (hidden % CHUNK == 0) { if (gated) UP(true, DIRECT); else UP(false, DIRECT); }
  else { if (gated) UP(true, BY_FOUR); else UP(false, BY_FOUR); }
#undef UP
  const unsigned down_blocks = blocks((routed + shared_rows) * tiles(hidden, 64));
  if (ff % CHUNK == 0 && shared % CHUNK == 0) moe_down_rows_f32_kernel<DIRECT><<<down_blocks, 256, 0, s>>>(a, act_shared, wd, parts, p);
  else moe_down_rows_f32_kernel<BY_FOUR><<<down_blocks, 256, 0, s>>>(a, act_shared, wd, parts, p);
  add_parts(p, parts, (float*)y, s);
  HOLON_LAUNCH_OK();
  return 0;
}
