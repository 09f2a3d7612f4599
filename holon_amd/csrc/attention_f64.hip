// Paged causal softmax attention of the 32-bit path on the float64 matrix cores: heads of 64 and 128 whose keys and
// values have one width, pages of whole tiles of 16 tokens. Operands are float32, both long sums (a score over the head, the
// values over the keys) float64, scores and softmax float32. The general kernel (softmax_attention.hip: options and layout of
// the pages as there) serves every other geometry. Which of the two a model's attention takes depends on the geometry alone and not
// on the step: a position's result is then the same bits in a prompt, in its portions, decoded, and whatever else is in the step.
//
// A block takes 16 columns, the heads of one kv head's group at consecutive tokens of a row, so a key is read once for all of them.
// Its eight waves walk tiles of 16 keys, wave w the tiles w, w + 8, ... counted from key 0, each with a running
// maximum, sum and values; they are combined at the end in a fixed order. Tiles that a token does not see change nothing of
// its column, so every sum's order depends on the token's position alone.
//   S^T = K Q^T: 16 keys x 4 dimensions a product. Lane l holds row or column l % 16 at k = l / 16 of either operand, and
//     rows 4 r + l / 16 of the result in register r. Keys enter in the order that leaves a lane keys 4 (l / 16) + r, dimensions
//     four neighbours a lane, so that both operands are 16-byte loads;
//   O^T = V^T P^T: 16 dimensions x 4 keys, the weights straight from the registers that hold them, values (transposed inside a
//     page) as 16-byte loads of the same four keys.
//
// Bound by the float64 products, 64 of 75 cycles each a tile of 16 keys and 128 dimensions, and the conversions beside them
// (a tile's keys and values, and the queries again, which as float64 would take registers that spill). us against the general
// kernel, 16 heads of 128 on 4: prompts of one row of 37 / 64 / 128 / 700 tokens 12 / 13 / 17 / 104 and 10 / 13 / 29 / 401, 12 decode rows
// behind 600 beside a prompt of 500 129 and 234; 8 heads of 64 on one, 700 tokens 33 and 114. A decode row fills a part of the columns
// alone and its block's waves are few: one behind 150 / 700 / 6,000 tokens 16 / 41 / 293 and 12 / 30 / 256, 16 behind 700 44 and 36, 64
// behind 500 41 and 70. Each head its own keys, a column a token: 37 / 700 tokens 21 / 142 and 10 / 412.
#include <float.h>

#include <type_traits>

#include "common.h"
#include "holon_hip.h"

typedef double f64x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace {
constexpr int WAVES = 8, KEYS = 16;

struct AttnF64 {
  const float* q;                  // [tokens, heads, dim]
  float* out;
  const float* pages;              // a page: kv_heads planes of keys [P, dim], kv_heads / v_share planes of values [dim, P]
  const int32_t* table;            // [table_rows, table_stride]
  int table_stride, table_rows;
  const int32_t* slots;            // a token's row of the table: slots[token_row[t]]
  const int32_t* token_row;
  const int32_t* positions;
  int tokens, heads, kv_heads, page_size, num_pages;
  float scale;
  int window;                      // see first_seen
  const float* sink;               // nullable, [heads]
  float softcap;                   // 0: none
  const float* r1;                 // nullable: the distance bias's two numbers a head
  const float* r2;
  int v_share;
  int per;                         // tokens a block takes
  double* part_o;                  // SPLIT: [tokens, heads, WAVES, dim] and [tokens, heads, WAVES, 2]
  float* part_ml;
};

// DT: head_dim / 16. MOD: a cap or a distance bias on the scores. SPLIT: the block is wave blockIdx.z alone, and leaves what the waves
// exchange at the end in memory for `attention_f64_merge_kernel`: a decode row's few blocks then fill more than a few compute units (one row
// behind 700 tokens, 16 heads of 128 on 4: 45 us, split 23.1 + 4.6).
template <int DT, bool MOD, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? WAVE : WAVES * WAVE, SPLIT ? 1 : 2) attention_f64_kernel(AttnF64 a) {
  constexpr int D = DT * 16;
  __shared__ double red[SPLIT ? 1 : WAVES / 2][SPLIT ? 1 : D][17];
  __shared__ float ml_s[WAVES][16][2];
  __shared__ float den_s[16];
  const int w = SPLIT ? (int)blockIdx.z : __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  const int group = a.heads / a.kv_heads, side = min(group, 16), blocks = (group + 15) / 16;      // columns a token takes
  const int hk = blockIdx.y / blocks, h_at = blockIdx.y % blocks * 16 + c % side;
  const int P = a.page_size;
  // The block's tokens: from t0 on those of one row up to a position that is a multiple of `per`. A token that follows the one before
  // it there lies in another block, and its own ends at once; rows that meet, and decode rows, have blocks of their own. (Every
  // per-th token first, an odd number of them: blocks are dealt to the XCDs and their parts in turn, and those that stay would share a
  // few of them, 12 decode rows of 16 kv heads beside a prompt of 500 tokens 900 us for 250.)
  const int sets = gridDim.x / a.per, t0 = blockIdx.x % sets * a.per + blockIdx.x / sets;
  if (t0 >= a.tokens) return;
  const int row = a.token_row[t0], pos0 = a.positions[t0];
  const auto follows = [&](int t) {
    return a.positions[t] > 0 && a.positions[t] % a.per != 0 && a.token_row[t] == a.token_row[t - 1] &&
           a.positions[t] == a.positions[t - 1] + 1;
  };
  if (t0 > 0 && follows(t0)) return;
  const int nth = c / side, t = t0 + nth;
  const bool mine = h_at < group && t < a.tokens &&
                    (nth == 0 || (pos0 >= 0 && pos0 % a.per + nth < a.per && a.token_row[t] == row && a.positions[t] == pos0 + nth &&
                                  follows(t)));
  const int head = hk * group + h_at, pos = mine ? pos0 + nth : -1;
  const bool live = pos >= 0;                              // (a padded row's token: position -1, and 0 is written)
  f32x4_t q[DT];                                           // dimensions 16 m + 4 g .. + 3
#pragma unroll
  for (int m = 0; m < DT; ++m)
    q[m] = mine ? *reinterpret_cast<const f32x4_t*>(a.q + ((int64_t)t * a.heads + head) * D + 16 * m + 4 * g) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float b1 = mine && a.r1 ? a.r1[head] : 0.f, b2 = mine && a.r1 ? a.r2[head] : 0.f;
  const int64_t page_len = (int64_t)(a.kv_heads + a.kv_heads / a.v_share) * P * D;
  const int64_t values = ((int64_t)a.kv_heads + hk / a.v_share) * P * D;
  const int first = pos >= 0 ? max(0, first_seen(pos, a.window)) : 0;

  int last = live ? pos : -1, least = live ? pos : 0x7fffffff, from = live ? first : 0x7fffffff, whole_from = live ? first : 0;
  const auto columns = [&](auto distance) {                // over the 16 lanes of a group of columns
    constexpr int O = decltype(distance)::value;
    last = max(last, lane_xor<O>(last));
    least = min(least, lane_xor<O>(least));
    from = min(from, lane_xor<O>(from));
    whole_from = max(whole_from, lane_xor<O>(whole_from));
  };
  columns(std::integral_constant<int, 1>{});
  columns(std::integral_constant<int, 2>{});
  columns(std::integral_constant<int, 4>{});
  columns(std::integral_constant<int, 8>{});
  last = __builtin_amdgcn_readfirstlane(last);
  from = __builtin_amdgcn_readfirstlane(from);
  const int slot = min(max(a.slots[row], 0), a.table_rows - 1);
  const int32_t* trow = a.table + (int64_t)slot * a.table_stride;
  const auto page_of = [&](int tile) {                   // -1: the table does not hold the tile, its keys are not seen
    const int at = tile * KEYS / P;
    if (tile * KEYS > last || at >= a.table_stride) return -1;
    const int page = __builtin_amdgcn_readfirstlane(trow[at]);
    return page >= 0 && page < a.num_pages ? page : -1;
  };
  const auto load_keys = [&](int tile, int page, f32x4_t (&k)[DT]) {
    const float* p = a.pages + page * page_len + ((int64_t)hk * P + tile * KEYS % P + 4 * (c % 4) + c / 4) * D + 4 * g;
#pragma unroll
    for (int m = 0; m < DT; ++m) k[m] = *reinterpret_cast<const f32x4_t*>(p + 16 * m);
  };
  f64x4_t acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f64x4_t{0, 0, 0, 0};
  float m = -INFINITY, l = 0.f;
  int tile = from / KEYS;                                // (from: no live column: 0x7fffffff, and last is -1)
  tile += (w - tile % WAVES + WAVES) % WAVES;
  int page = last >= 0 ? page_of(tile) : -1;
  f32x4_t k[DT];
  if (page >= 0) load_keys(tile, page, k);
  while (last >= 0 && tile * KEYS <= last) {
    const int next = tile + WAVES, next_page = page_of(next);
    f32x4_t v[DT];
    if (page >= 0) {
      const float* p = a.pages + page * page_len + values + (int64_t)c * P + tile * KEYS % P + 4 * g;
#pragma unroll
      for (int d = 0; d < DT; ++d) v[d] = *reinterpret_cast<const f32x4_t*>(p + (int64_t)d * 16 * P);
    }
    if (page >= 0) {
      f64x4_t s2[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        asm volatile("" : "+v"(q[i]));                    // (converted again each tile: as float64 they take twice the registers)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          s2[u % 2] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)k[i][u], (double)q[i][u], s2[u % 2], 0, 0, 0);
      }
      if (next_page >= 0) load_keys(next, next_page, k);      // under way while the weights and the values are worked on
      const int key0 = tile * KEYS, mine0 = key0 + 4 * g;
      float s[4], mx = -INFINITY;
      bool seen[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        seen[r] = live && mine0 + r <= pos && mine0 + r >= first;
        s[r] = (float)(s2[0][r] + s2[1][r]) * a.scale;
        if (MOD && a.softcap > 0.f) s[r] = a.softcap * tanhf(s[r] / a.softcap);
        if (MOD && a.r1 != nullptr) s[r] -= b1 * log1pf(b2 * (float)max(pos - mine0 - r, 0));
        if (seen[r]) mx = fmaxf(mx, s[r]);
      }
      mx = xor_max<16>(mx);
      mx = xor_max<32>(mx);
      const float m_new = fmaxf(m, mx), at = m_new == -INFINITY ? 0.f : m_new;    // (a score that is NaN stays one)
      const float alpha = expf(m - at);
      float p[4], sum = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[r] = seen[r] ? expf(s[r] - at) : 0.f;
        sum += p[r];
      }
      sum = xor_sum<16>(sum);
      sum = xor_sum<32>(sum);
      l = l * alpha + sum;
      if (__any(m_new != m)) {
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[d] *= (double)alpha;
      }
      m = m_new;
      bool bad = false;
      if (!(key0 + KEYS - 1 <= least && key0 >= whole_from)) {     // some column does not see all of the tile
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (mine0 + r > last || mine0 + r < from) v[d][r] = 0.f;             // held by no one: may be anything
            bad |= !(fabsf(v[d][r]) <= FLT_MAX);
          }
      }
      if (__any(bad)) {
        // a value that is not finite would reach columns that do not see it as 0 times itself: a token's columns at a time, over
        // the values that it sees
        for (int at_token = 0; at_token < a.per; ++at_token) {
          const int its_pos = __builtin_amdgcn_readlane(live ? pos : -1, at_token * side);
          const int its_first = __builtin_amdgcn_readlane(first, at_token * side);
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            f64x4_t one = acc[d];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const double value = mine0 + r <= its_pos && mine0 + r >= its_first ? (double)v[d][r] : 0.0;
              one = __builtin_amdgcn_mfma_f64_16x16x4f64(value, (double)p[r], one, 0, 0, 0);
            }
            if (c / side == at_token) acc[d] = one;
          }
        }
      } else {
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          asm volatile("" : "+v"(v[d]));
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[d] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)v[d][r], (double)p[r], acc[d], 0, 0, 0);
        }
      }
    } else if (next_page >= 0) {
      load_keys(next, next_page, k);
    }
    tile = next;
    page = next_page;
  }
  if constexpr (SPLIT) {
    if (!mine) return;
    const int64_t cell = ((int64_t)t * a.heads + head) * WAVES + w;
    if (g == 0) { a.part_ml[cell * 2] = m; a.part_ml[cell * 2 + 1] = l; }
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) a.part_o[cell * D + d * 16 + 4 * r + g] = acc[d][r];
    return;
  }
  // the waves' sums, in one order: 0 + 4, 1 + 5, 2 + 6, 3 + 7, then those from the first on
  if (g == 0) { ml_s[w][c][0] = m; ml_s[w][c][1] = l; }
  __syncthreads();
  float top = a.sink && mine ? a.sink[head] : -INFINITY;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) top = fmaxf(top, ml_s[i][c][0]);
  const auto share = [&](float max) { return max == -INFINITY ? 0.f : expf(max - top); };
  if (w == 0 && g == 0) {
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) den = fmaf(ml_s[i][c][1], share(ml_s[i][c][0]), den);
    if (a.sink && mine) den += expf(a.sink[head] - top);
    den_s[c] = den;
  }
  const double f = (double)share(m);
  if (w < WAVES / 2) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[w][d * 16 + 4 * r + g][c] = __dmul_rn(acc[d][r], f);
  }
  __syncthreads();
  if (w >= WAVES / 2) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double& to = red[w - WAVES / 2][d * 16 + 4 * r + g][c];
        to = fma(acc[d][r], f, to);
      }
  }
  __syncthreads();
  const uint64_t to_write = __ballot(mine), with_keys = __ballot(live);       // (bit c: column c; the same in every wave)
  for (int e = threadIdx.x; e < 16 * D; e += WAVES * WAVE) {
    const int col = e / D, d = e % D;
    if (!(to_write >> col & 1)) continue;
    double sum = 0;
#pragma unroll
    for (int i = 0; i < WAVES / 2; ++i) sum += red[i][d][col];
    const float den = den_s[col];
    const float y = (float)(den > 0.f ? sum / (double)den : sum * 0.0);      // (no weights: 0)
    a.out[(((int64_t)t0 + col / side) * a.heads + hk * group + blockIdx.y % blocks * 16 + col % side) * D + d] =
        with_keys >> col & 1 ? y : 0.f;
  }
}

// What the waves of a block do at its end, from their sums in memory: the same operations in the same order.
__global__ void __launch_bounds__(128) attention_f64_merge_kernel(AttnF64 a, int dim) {
  const int t = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  const int64_t cell = ((int64_t)t * a.heads + head) * WAVES;
  float m[WAVES], l[WAVES];
  double o[WAVES];
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    m[i] = a.part_ml[(cell + i) * 2];
    l[i] = a.part_ml[(cell + i) * 2 + 1];
    o[i] = a.part_o[(cell + i) * dim + d];
  }
  float top = a.sink ? a.sink[head] : -INFINITY;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) top = fmaxf(top, m[i]);
  float den = 0.f;
  double sum = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    m[i] = m[i] == -INFINITY ? 0.f : expf(m[i] - top);
    den = fmaf(l[i], m[i], den);
  }
  if (a.sink) den += expf(a.sink[head] - top);
#pragma unroll
  for (int i = 0; i < WAVES / 2; ++i) sum += fma(o[i + WAVES / 2], (double)m[i + WAVES / 2], __dmul_rn(o[i], (double)m[i]));
  const float y = (float)(den > 0.f ? sum / (double)den : sum * 0.0);
  a.out[((int64_t)t * a.heads + head) * dim + d] = a.positions[t] >= 0 ? y : 0.f;
}
}  // namespace

extern "C" int holon_softmax_attention_f64_supported(int heads, int kv_heads, int dim, int vdim, int page_size) {
  return dim == vdim && (dim == 64 || dim == 128) && page_size > 0 && page_size % KEYS == 0 && kv_heads > 0 && heads % kv_heads == 0 &&
         (int64_t)kv_heads * ((heads / kv_heads + 15) / 16) <= 65535;
}

static int f64_launch(const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
                                           int table_rows, const int32_t* slots, const int32_t* token_row,
                                           const int32_t* positions, int tokens, int heads, int kv_heads, int dim, int vdim,
                                           int page_size, int num_pages, const float* sink, float scale, int window, int dtype,
                                           float softcap, const float* r1, const float* r2, int keep_first, int v_share,
                                           double* part_o, float* part_ml, void* stream) {
  HOLON_CHECK(holon_softmax_attention_f64_supported(heads, kv_heads, dim, vdim, page_size) && dtype == HOLON_F32 &&
                  (uintptr_t)q % 16 == 0 && (uintptr_t)pages % 16 == 0,
              "softmax_attention (float64 sums): heads of %d / %d, pages of %d, type %d, or pointers that are not at 16 bytes", dim,
              vdim, page_size, dtype);
  HOLON_CHECK(v_share >= 1 && kv_heads % v_share == 0, "softmax_attention: %d key heads do not share value heads by %d",
              kv_heads, v_share);
  HOLON_CHECK(tokens >= 0 && num_pages > 0 && window > -0x7fffffff && table_stride > 0 && table_rows > 0 && softcap >= 0.f &&
                  (window <= 0 || keep_first == 0) && (r1 == nullptr) == (r2 == nullptr),
              "softmax_attention: %d pages, a window of %d, a cap of %g, %d kept tokens", num_pages, window, softcap, keep_first);
  if (tokens == 0) return 0;
  HOLON_CHECK(tokens < 1 << 30, "softmax_attention: %d tokens exceed one launch", tokens);
  const int group = heads / kv_heads, side = group < 16 ? group : 16, per = 16 / side;
  const AttnF64 a{(const float*)q, (float*)out, (const float*)pages, table, table_stride, table_rows, slots, token_row, positions,
                  tokens, heads, kv_heads, page_size, num_pages, scale, window, sink, softcap, r1, r2, v_share, per, part_o, part_ml};
  const bool split = part_o != nullptr;
  const dim3 grid(((tokens + per - 1) / per | 1) * per, kv_heads * ((group + 15) / 16), split ? WAVES : 1);
  const bool mod = softcap > 0.f || r1 != nullptr;
  hipStream_t s = (hipStream_t)stream;
#define F64(DT, MOD)                                                                   \
  do {                                                                                 \
    if (split) attention_f64_kernel<DT, MOD, true><<<grid, WAVE, 0, s>>>(a);           \
    else attention_f64_kernel<DT, MOD, false><<<grid, WAVES * WAVE, 0, s>>>(a);        \
  } while (0)
  if (dim == 64 && !mod) F64(4, false);
  else if (dim == 64) F64(4, true);
  else if (!mod) F64(8, false);
  else F64(8, true);
#undef F64
  HOLON_LAUNCH_OK();
  if (split) {
    attention_f64_merge_kernel<<<dim3(tokens, heads), dim, 0, s>>>(a, dim);
    HOLON_LAUNCH_OK();
  }
  return 0;
}

// Arguments as holon_softmax_attention's; float32, no kept first tokens under a window.
extern "C" int holon_softmax_attention_f64(const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
                                           int table_rows, const int32_t* slots, const int32_t* token_row,
                                           const int32_t* positions, int tokens, int heads, int kv_heads, int dim, int vdim,
                                           int page_size, int num_pages, const float* sink, float scale, int window, int dtype,
                                           float softcap, const float* r1, const float* r2, int keep_first, int v_share,
                                           void* stream) {
  return f64_launch(q, out, pages, table, table_stride, table_rows, slots, token_row, positions, tokens, heads, kv_heads, dim, vdim,
                    page_size, num_pages, sink, scale, window, dtype, softcap, r1, r2, keep_first, v_share, nullptr, nullptr, stream);
}

// The same bits with a block's eight waves in blocks of their own and a second kernel behind them: part_o [tokens, heads, 8, dim] float64,
// part_ml [tokens, heads, 8, 2] float32.
extern "C" int holon_softmax_attention_f64_split(const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
                                                 int table_rows, const int32_t* slots, const int32_t* token_row,
                                                 const int32_t* positions, int tokens, int heads, int kv_heads, int dim, int vdim,
                                                 int page_size, int num_pages, const float* sink, float scale, int window, int dtype,
                                                 float softcap, const float* r1, const float* r2, int keep_first, int v_share,
                                                 double* part_o, float* part_ml, void* stream) {
  HOLON_CHECK(part_o != nullptr && part_ml != nullptr && heads <= 65535, "softmax_attention (float64 sums): no room for the waves' sums");
  return f64_launch(q, out, pages, table, table_stride, table_rows, slots, token_row, positions, tokens, heads, kv_heads, dim, vdim,
                    page_size, num_pages, sink, scale, window, dtype, softcap, r1, r2, keep_first, v_share, part_o, part_ml, stream);
}
