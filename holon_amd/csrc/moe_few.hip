// The experts of a mixture for steps of up to 16 rows, bfloat16: two products that read the weights of the chosen experts
// alone. All experts' first projections are the rows of one weight, their second ones the columns of another (see
// parts/ffn.py); which experts any row of the step chose is read from the router's weights on the device, so the launches
// are the same whatever was chosen (a step may be replayed from a graph). Every sum has the order that gemm_skinny.hip's product of
// that size gives it, so the results are bit for bit those of the products over all experts.
//
// Both stream weights in the tile layout of gemm_skinny.hip ([N / 16, K / 32, 64 lanes, 8]) and are bound by memory: one
// row that chooses 2 of 8 experts beside a shared one reads 3 of 9 parts. Over experts of 2,048 by 2,048 at one row: 11.8 us for
// gates, ups and activation and 9.6 for the second product (2.1 and 2.6 TB/s: a kernel's first loads wait for the router's
// choice); all experts' products take 25.4 and 18.4 and the activation between them 4.5.
#include <type_traits>

#include "common.h"
#include "holon_hip.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace {
constexpr int MAX_EXPERTS = 1024;

struct Chosen {
  const float* weights;        // [M, stride] float32: 0 where a row did not choose an expert
  int stride, experts, ff, shared, shared_col;   // shared_col < 0: the shared expert's weight is 1
  // The weight of column `col` (of experts * ff + shared) for row m.
  __device__ __forceinline__ float of(int m, int col) const {
    if (col < experts * ff) return weights[(int64_t)m * stride + col / ff];
    return shared_col >= 0 ? weights[(int64_t)m * stride + shared_col] : 1.f;
  }
};

__device__ __forceinline__ bf16x8_t row_values(const bf16_t* at, bool have) {
  bf16x8_t v;
  if (have) {
    v = *reinterpret_cast<const bf16x8_t*>(at);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (__bf16)0.f;
  }
  return v;
}

// `steps` products of a wave over H weight tiles, added to acc in order: the loads of UNROLL of them into one of two sets of
// registers while the other set is multiplied; what is left over, at the end, in a set by itself.
template <int H, int UNROLL, typename At, typename Tokens>
__device__ __forceinline__ void in_two_sets(f32x4_t (&acc)[H], int steps_, At at, Tokens tokens) {
  const int steps = __builtin_amdgcn_readfirstlane(steps_);      // (a matrix instruction runs whatever lanes are off: its
                                                                 // conditions have to be branches of the whole wave)
  bf16x8_t wf[2][H][UNROLL], xf[2][UNROLL];
  const auto ask = [&](auto set, int s) {
    constexpr int B = decltype(set)::value;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
        wf[B][h][u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(at(h, min(s + u, steps - 1))));
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) xf[B][u] = tokens(min(s + u, steps - 1));
  };
  const auto use = [&](auto set, int s) {
    constexpr int B = decltype(set)::value;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      if (s + u < steps)
#pragma unroll
        for (int h = 0; h < H; ++h) acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[B][h][u], xf[B][u], acc[h], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  ask(even, 0);
  for (int s = 0; s < steps; s += 2 * UNROLL) {
    if (s + UNROLL < steps) ask(odd, s + UNROLL);
    use(even, s);
    if (s + UNROLL < steps) {
      if (s + 2 * UNROLL < steps) ask(even, s + 2 * UNROLL);
      use(odd, s + UNROLL);
    }
  }
}

// One block 16 columns of the experts' activations: gate and up tile over all of K, split over the block's waves in order,
// then round(round(round(silu(gate)) * up) * weight); GATED false: one tile and round(max(up, 0)^2 * weight). Blocks of a
// routed expert that no row chose end at once and write nothing. 0 where the weight is 0.
template <int WPB, bool GATED>
__global__ void __launch_bounds__(WPB * 64) moe_up_few_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              bf16_t* __restrict__ y, int M, int cols, int K, Chosen ch) {
  constexpr int H = GATED ? 2 : 1;
  __shared__ f32x4_t red[WPB > 1 ? (WPB - 1) * H * WAVE : 1];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16;
  const bool have = c < M;
  const float weight = have ? ch.of(c, blockIdx.x * 16) : 0.f;      // (16 columns are one expert's)
  // The second product leaves out the experts that no row chose, never the shared one: its columns are written whatever its
  // weights are, zeros where its gate has come to 0 for every row.
  if (blockIdx.x * 16 < ch.experts * ch.ff && __ballot(weight != 0.f) == 0) return;
  const int steps = K / 32 / WPB;
  const bf16_t* wp[H];
#pragma unroll
  for (int h = 0; h < H; ++h)
    wp[h] = w + (((int64_t)h * (cols / 16) + blockIdx.x) * (K / 32) + (int64_t)wave * steps) * 512 + lane * 8;
  const bf16_t* xp = x + (int64_t)c * K + (int64_t)wave * steps * 32 + 8 * g;
  f32x4_t acc[H];
#pragma unroll
  for (int h = 0; h < H; ++h) acc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  in_two_sets<H, 4>(acc, steps, [&](int h, int s) { return wp[h] + (int64_t)s * 512; },
                    [&](int s) { return row_values(xp + s * 32, have); });
  if (WPB > 1) {
    if (wave > 0) {
#pragma unroll
      for (int h = 0; h < H; ++h) red[((wave - 1) * H + h) * WAVE + lane] = acc[h];
    }
    __syncthreads();
    if (wave > 0) return;
    for (int ww = 1; ww < WPB; ++ww)
#pragma unroll
      for (int h = 0; h < H; ++h) acc[h] += red[((ww - 1) * H + h) * WAVE + lane];
  }
  if (!have) return;
  ushort4 o;
  bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v;
    if constexpr (GATED) {
      const float gate = Elem<bf16_t>::round(acc[0][r]), up = Elem<bf16_t>::round(acc[H - 1][r]);
      v = Elem<bf16_t>::round(Elem<bf16_t>::round(silu<bf16_t>(gate)) * up) * weight;
    } else {
      const float up = fmaxf(Elem<bf16_t>::round(acc[0][r]), 0.f);
      v = up * up * weight;
    }
    oe[r] = float_to_bf16(weight != 0.f ? v : 0.f);
  }
  *reinterpret_cast<ushort4*>(y + (int64_t)c * cols + blockIdx.x * 16 + 4 * g) = o;
}

// y[M, N] = act[M, cols] w[N, cols]^T over the columns of the experts that a row of the step chose, and the shared one's. A
// block 16 columns of y; all columns, 32 at a time, lie in RUNS equal runs in order, and a run leaves out those of experts that no
// row chose (they would add zeros). The runs that have any are dealt out to the block's eight waves, which have room for a
// run's worth of loads under way; the runs' sums are added in order.
// A wave's first weights wait for the choice, so that comes in one round of memory latency: a lane an expert, the rows' weights asked for
// together: 25 MB into 2,048 columns at 1 / 4 / 8 / 16 rows 9.4 / 10.0 / 11.0 / 13.3 us (9.5 / 11.0 / 13.2 / 17.8 with one row's looked at
// behind the other's).
constexpr int DOWN_WAVES = 8;
struct Down {
  const bf16_t* act;
  const bf16_t* w;
  bf16_t* y;
  int M, N, cols;
  Chosen ch;
};
template <int RUNS>
__device__ __forceinline__ void down_tile(const Down& d, int tile, f32x4_t (*sums)[WAVE]) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16;
  const bool have = c < d.M;
  const Chosen& ch = d.ch;
  const int per = ch.ff / 32, run = d.cols / 32 / RUNS, routed = ch.experts * per;      // steps of 32 columns an expert, a run, all experts
  const auto chosen = [&](int e0) {                        // which of experts e0 .. e0 + 63 any row chose
    const float* at = ch.weights + min(e0 + lane, ch.experts - 1);
    float v[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) v[m] = at[(int64_t)min(m, d.M - 1) * ch.stride];
    bool any = false;
#pragma unroll
    for (int m = 0; m < 16; ++m) any |= v[m] != 0.f;
    return __ballot(any && e0 + lane < ch.experts);
  };
  const uint64_t first = chosen(0);
  bool mine = false;                                       // lane r: whether run r has columns to add
  {
    const int e_first = lane * run / per, e_last = min(((lane + 1) * run - 1) / per, ch.experts - 1);
    mine = (lane + 1) * run > routed;
    for (int e0 = 0; e0 < ch.experts; e0 += WAVE) {
      const uint64_t mask = e0 == 0 ? first : chosen(e0);
      const int lo = max(e_first - e0, 0), hi = min(e_last - e0, WAVE - 1);
      if (lo <= hi) mine |= (mask >> lo & (hi - lo == WAVE - 1 ? ~0ull : (1ull << (hi - lo + 1)) - 1)) != 0;
    }
    mine = mine && lane < RUNS;
  }
  const uint64_t active = __ballot(mine);
  const bf16_t* wp = d.w + (int64_t)tile * (d.cols / 32) * 512 + lane * 8;
  const bf16_t* xp = d.act + (int64_t)c * d.cols + 8 * g;
  int turn = 0;
  for (uint64_t left = active; left != 0; left &= left - 1, ++turn) {
    if (turn % DOWN_WAVES != wave) continue;
    const int r = __builtin_ctzll(left), lo = r * run, hi = lo + run;
    f32x4_t acc[1] = {{0.f, 0.f, 0.f, 0.f}};
    const auto part = [&](int from, int to) {
      if (from < to)
        in_two_sets<1, 12>(acc, to - from, [&](int, int s) { return wp + (int64_t)(from + s) * 512; },
                           [&](int s) { return row_values(xp + (from + s) * 32, have); });
    };
    const int e_last = min((hi - 1) / per, ch.experts - 1);
    int from = -1, to = -1;                                // columns side by side, one product
    for (int e0 = lo / per / WAVE * WAVE; e0 <= e_last; e0 += WAVE) {
      uint64_t mask = e0 == 0 ? first : chosen(e0);        // (bits outside the run: cut off by its borders)
      if (lo / per > e0) mask &= ~0ull << (lo / per - e0);
      if (e_last - e0 < WAVE - 1) mask &= (1ull << (e_last - e0 + 1)) - 1;
      for (; mask != 0; mask &= mask - 1) {
        const int at = (e0 + __builtin_ctzll(mask)) * per;
        if (max(lo, at) != to) {
          part(from, to);
          from = max(lo, at);
        }
        to = min(hi, at + per);
      }
    }
    if (hi > routed) {                                     // the shared one's
      if (max(lo, routed) != to) {
        part(from, to);
        from = max(lo, routed);
      }
      to = hi;
    }
    part(from, to);
    sums[r][lane] = acc[0];
  }
  __syncthreads();
  if (wave > 0 || !have) return;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < RUNS; ++r)
    if (active >> r & 1) acc += sums[r][lane];
  ushort4 o;
  o.x = float_to_bf16(acc[0]); o.y = float_to_bf16(acc[1]); o.z = float_to_bf16(acc[2]); o.w = float_to_bf16(acc[3]);
  *reinterpret_cast<ushort4*>(d.y + (int64_t)c * d.N + tile * 16 + 4 * g) = o;
}
template <int RUNS>
__global__ void __launch_bounds__(DOWN_WAVES * 64) moe_down_few_kernel(Down d) {
  __shared__ f32x4_t sums[RUNS][WAVE];
  down_tile<RUNS>(d, blockIdx.x, sums);
}

// The second product beside another one of the same rows that reads nothing of it (the output projection of the sublayer beside): over
// 2,048 columns either leaves half of the units without a block. The other product's blocks come behind, 16 waves' worth of K two to a
// wave, every sum in the order that gemm_skinny.hip gives it. Two of 8 experts of 2,048 beside a shared one, with 2,048 x 2,048 at 1 / 4 / 8 / 16
// rows 9.8 / 10.4 / 11.3 / 13.5 us (one after the other 13.6 / 14.5 / 15.8 / 18.7), with 4,096 x 4,096 12.7 / 13.9 / 15.4 / 18.0 (16.7 / 17.5 /
// 18.9 / 22.4).
struct Beside {
  const bf16_t* x;
  const bf16_t* w;              // tiled
  void* y;
  int N, K, waves, form;        // waves a tile; form as out_f32 of holon_gemm_skinny_bf16
};
template <int RUNS>
__global__ void __launch_bounds__(DOWN_WAVES * 64) moe_down_beside_kernel(Down d, Beside b) {
  __shared__ f32x4_t sums[16][WAVE];
  if ((int)blockIdx.x < d.N / 16) {
    down_tile<RUNS>(d, blockIdx.x, sums);
    return;
  }
  const int all = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  const int sides = b.waves == 16 ? 2 : 1, own = b.waves == 16 ? 8 : b.waves;      // slices of K a wave; waves of the block a tile
  const int wave = all % own, tile = ((int)blockIdx.x - d.N / 16) * (DOWN_WAVES / own) + all / own;
  const bool have = c < d.M, mine = tile < b.N / 16;
  const int steps = b.K / 32 / b.waves;
  if (mine)
    for (int side = 0; side < sides; ++side) {
      const int slice = wave + side * 8;
      const bf16_t* wp = b.w + ((int64_t)tile * (b.K / 32) + (int64_t)slice * steps) * 512 + lane * 8;
      const bf16_t* xp = b.x + (int64_t)c * b.K + (int64_t)slice * steps * 32 + 8 * g;
      f32x4_t acc[1] = {{0.f, 0.f, 0.f, 0.f}};
      in_two_sets<1, 8>(acc, steps, [&](int, int s) { return wp + (int64_t)s * 512; }, [&](int s) { return row_values(xp + s * 32, have); });
      sums[all + side * 8][lane] = acc[0];
    }
  __syncthreads();
  if (wave > 0 || !mine || !have) return;
  f32x4_t acc = sums[all][lane];
  for (int ww = 1; ww < b.waves; ++ww) acc += sums[all + ww][lane];
  const int64_t at = (int64_t)c * b.N + tile * 16 + 4 * g;
  ushort4 o;
  bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
  for (int r = 0; r < 4; ++r) oe[r] = float_to_bf16(acc[r]);
  if (b.form == 2) {
    f32x4_t wide;
#pragma unroll
    for (int r = 0; r < 4; ++r) wide[r] = bf16_to_float(oe[r]);
    *reinterpret_cast<f32x4_t*>((float*)b.y + at) = wide;
    return;
  }
  if (b.form == 4)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = fmaxf(bf16_to_float(oe[r]), 0.f);
      oe[r] = float_to_bf16(v * v);
    }
  *reinterpret_cast<ushort4*>((bf16_t*)b.y + at) = o;
}
}  // namespace

// Whether the two products serve `rows` rows of `hidden` over `experts` experts of `ff` columns and `shared` shared ones.
extern "C" int holon_moe_few_supported(int rows, int hidden, int experts, int ff, int shared) {
  return rows >= 1 && rows <= 16 && hidden > 0 && hidden % 32 == 0 && experts >= 1 && experts <= MAX_EXPERTS && ff > 0 &&
         ff % 32 == 0 && shared >= 0 && shared % 32 == 0 && (int64_t)experts * ff + shared <= 0x7fffffff / 16;
}

// act [rows, experts ff + shared] = what moe_gate (gated) or moe_relu2 leaves of x [rows, hidden] times the tiled weight
// ([gates; ups] or [ups]); columns of experts that no row chose are left as they are.
extern "C" int holon_moe_up_few_bf16(const void* x, const void* w_tiled, void* act, int rows, int hidden, int experts, int ff,
                                     int shared, int gated, const float* weights, int wstride, int shared_col, void* stream) {
  HOLON_CHECK(holon_moe_few_supported(rows, hidden, experts, ff, shared) && wstride >= experts && shared_col < wstride,
              "moe (few rows): %d rows of %d, %d experts of %d, %d shared columns not served", rows, hidden, experts, ff, shared);
  const Chosen ch{weights, wstride, experts, ff, shared, shared_col};
  const int cols = experts * ff + shared;
  hipStream_t s = (hipStream_t)stream;
#define MOE_UP(WPB)                                                                                                       \
  case WPB:                                                                                                               \
    if (gated) moe_up_few_kernel<WPB, true><<<cols / 16, WPB * 64, 0, s>>>((const bf16_t*)x, (const bf16_t*)w_tiled,       \
                                                                           (bf16_t*)act, rows, cols, hidden, ch);          \
    else moe_up_few_kernel<WPB, false><<<cols / 16, WPB * 64, 0, s>>>((const bf16_t*)x, (const bf16_t*)w_tiled,            \
                                                                      (bf16_t*)act, rows, cols, hidden, ch);               \
    break
  switch (skinny_waves((gated ? 2 : 1) * (cols / 16), hidden)) { MOE_UP(16); MOE_UP(8); MOE_UP(4); MOE_UP(2); MOE_UP(1); }
#undef MOE_UP
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_moe_down_few_bf16(const void* act, const void* w_tiled, void* y, int rows, int hidden, int experts,
                                       int ff, int shared, const float* weights, int wstride, void* stream) {
  HOLON_CHECK(holon_moe_few_supported(rows, hidden, experts, ff, shared) && wstride >= experts,
              "moe (few rows): %d rows of %d, %d experts of %d, %d shared columns not served", rows, hidden, experts, ff, shared);
  const int cols = experts * ff + shared;
  const Down d{(const bf16_t*)act, (const bf16_t*)w_tiled, (bf16_t*)y, rows, hidden, cols, {weights, wstride, experts, ff, shared, -1}};
#define MOE_DOWN(RUNS) \
  case RUNS: moe_down_few_kernel<RUNS><<<hidden / 16, DOWN_WAVES * 64, 0, (hipStream_t)stream>>>(d); break
  switch (skinny_waves(hidden / 16, cols)) { MOE_DOWN(16); MOE_DOWN(8); MOE_DOWN(4); MOE_DOWN(2); MOE_DOWN(1); }
#undef MOE_DOWN
  HOLON_LAUNCH_OK();
  return 0;
}

// The same, and py [rows, N] = px [rows, K] times a tiled weight [N, K] in one launch; `form`: 0 bfloat16, 2 float32 values that were rounded
// to bfloat16 first, 4 bfloat16 max(product, 0)^2.
extern "C" int holon_moe_down_beside_bf16(const void* act, const void* w_tiled, void* y, int rows, int hidden, int experts,
                                          int ff, int shared, const float* weights, int wstride, const void* px, const void* pw, void* py,
                                          int N, int K, int form, void* stream) {
  HOLON_CHECK(holon_moe_few_supported(rows, hidden, experts, ff, shared) && wstride >= experts,
              "moe (few rows): %d rows of %d, %d experts of %d, %d shared columns not served", rows, hidden, experts, ff, shared);
  HOLON_CHECK(N > 0 && N % 16 == 0 && K >= 32 && K % 32 == 0 && (form == 0 || form == 2 || form == 4) &&
                  (((uintptr_t)px | (uintptr_t)pw | (uintptr_t)py) & 15) == 0,
              "moe (few rows) beside a product: N=%d K=%d form %d not served (N %% 16, K %% 32, operands at 16 bytes)", N, K, form);
  const int cols = experts * ff + shared;
  const Down d{(const bf16_t*)act, (const bf16_t*)w_tiled, (bf16_t*)y, rows, hidden, cols, {weights, wstride, experts, ff, shared, -1}};
  const Beside b{(const bf16_t*)px, (const bf16_t*)pw, py, N, K, skinny_waves(N / 16, K), form};
  const int per = b.waves >= 8 ? 1 : DOWN_WAVES / b.waves, blocks = hidden / 16 + (N / 16 + per - 1) / per;
#define MOE_DOWN(RUNS) \
  case RUNS: moe_down_beside_kernel<RUNS><<<blocks, DOWN_WAVES * 64, 0, (hipStream_t)stream>>>(d, b); break
  switch (skinny_waves(hidden / 16, cols)) { MOE_DOWN(16); MOE_DOWN(8); MOE_DOWN(4); MOE_DOWN(2); MOE_DOWN(1); }
#undef MOE_DOWN
  HOLON_LAUNCH_OK();
  return 0;
}
