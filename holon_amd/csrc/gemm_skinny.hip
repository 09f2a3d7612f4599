// y[M, N] = x[M, K] w[N, K]^T for up to 16 rows (decode steps): bfloat16 operands, float32 accumulation on the matrix
// cores, memory-bound on the weights. A workgroup owns 16 weight rows; its waves split K evenly and add their partial
// tiles through LDS in wave order, so the result does not depend on M or on anything but the shapes.
//
// v_mfma_f32_16x16x32_bf16 with the weights as A (16 rows x 32 k: lane l reads 16 contiguous bytes of row l%16) and
// the activations as B (32 k x 16 tokens: lane l reads 16 contiguous bytes of token l%16); the result tile has weight
// rows 4*(l/16)+r of token l%16 in lane l, i.e. 4 consecutive outputs of one token: one 8- or 16-byte store.
//
// Two weight layouts: rows [N, K] as the checkpoint stores them, and tiles [N/16, K/32, 64 lanes, 8] in which the
// 16 bytes lane l needs for one product are at lane l's place, so that a wave's load is one contiguous kilobyte and a
// tile's whole K extent is one contiguous run (measured: 6 to 7 TB/s against 4 to 5 for the row layout).
#include <type_traits>

#include "common.h"
#include "holon_hip.h"
#include "moe_router.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// A norm folded into the product that reads it. With RMSNorm y = x * rsqrt(mean(x^2) + eps) * g in front of a product
// with W, the product of the un-normed rows with W * diag(g) (folded into the tiled copy once, after loading), scaled
// per row by rsqrt(mean(x^2) + eps) in the epilogue, is the same number with one rounding moved from the normed
// activations to the folded weights; and the norm's kernel, which moves next to nothing and costs as much as a
// quarter of a projection, is gone. The sums of squares come as partial sums `stats` [parts, 16] (float32, row m of
// the step in column m): the kernel that last wrote the rows leaves one partial per 16 columns it owned, and the
// reader adds them in a fixed order (every wave a share in ascending order, the waves in wave order, the four lane
// groups in order).
struct RowScale {
  const float* stats;   // nullptr: rows are used as they are
  int parts;
  float eps, inv_dim;
};

// The sums of squares are read 16 parts at a time: lane l of a wave takes four floats of part 16 k + l / 4, columns
// 4 (l % 4) .. + 3, so a wave's load is one contiguous kilobyte; wave w takes chunks k = w, w + WPB, ... and adds them
// in that order. The values are asked for a few at a time, at the top of each round of the weight loop, and added one
// round later: loads return in the order they were issued, so by then they have arrived behind the weights that the
// round before waited for, and the sum never makes the stream wait.
template <int WPB>
struct RowSums {
  static constexpr int Q = 4;   // loads in flight per lane
  const f32x4_t* at;            // this lane's four floats of the next chunk
  int part, parts;              // the part they belong to; how many there are
  int n;                        // loads in flight
  f32x4_t v[Q], ss;
  __device__ __forceinline__ void start(const RowScale& rs, int wave, int lane) {
    at = reinterpret_cast<const f32x4_t*>(rs.stats) + wave * 64 + lane;
    part = wave * 16 + lane / 4;
    parts = rs.stats != nullptr ? rs.parts : 0;
    n = 0;
    ss = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void turn() {   // add what the last turn asked for, ask for the next
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (q < n) ss += v[q];
    n = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (part + q * 16 * WPB < parts) {
        v[q] = at[(int64_t)q * 64 * WPB];
        n = q + 1;
      }
    at += (int64_t)n * 64 * WPB;
    part += n * 16 * WPB;
  }
  __device__ __forceinline__ f32x4_t finish() {
    do turn(); while (n > 0);
    return ss;
  }
};
// After the waves' shares have been added: the sum over the 16 lanes that hold the same four columns (lanes l, l ^ 4,
// l ^ 8, l ^ 16, l ^ 32, in that order), then column c out of lane c / 4. Every lane of column c gets the same sum.
__device__ __forceinline__ float row_sum_of_column(f32x4_t v, int c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = xor_sum<32>(xor_sum<16>(xor_sum<8>(xor_sum<4>(v[i]))));
  const float t0 = __shfl(v[0], c / 4, WAVE), t1 = __shfl(v[1], c / 4, WAVE), t2 = __shfl(v[2], c / 4, WAVE),
              t3 = __shfl(v[3], c / 4, WAVE);
  return c % 4 == 0 ? t0 : (c % 4 == 1 ? t1 : (c % 4 == 2 ? t2 : t3));
}
// The four lane groups' shares of row c, added in order; every lane of column c gets the same sum.
__device__ __forceinline__ float over_lane_groups(float v, int c) {
  const float a = __shfl(v, c, WAVE), b = __shfl(v, 16 + c, WAVE), d = __shfl(v, 32 + c, WAVE), e = __shfl(v, 48 + c, WAVE);
  return ((a + b) + d) + e;
}

// A wave's run of `steps` products over NT weight tiles, added to acc. UNROLL products' loads wait in one of two sets of
// registers while the other set's are asked for: a wave that asks for all, waits for all and multiplies has nothing under way
// for part of its time. (One row of 2,048 / 8,192 / 18,432 against 2,048 columns, 16 waves a tile: 8 loads in one set 5.1, 11.6,
// 24.2 us; two sets of 4 4.35, 9.7, 21.7.)
// REST: steps is no multiple of UNROLL; what is left over is asked for while the last whole set is multiplied, where one load after
// the other behind it took 20 % of a short K's time (18432 x 704 at one row 9.7 us and 6.6 so; gated, 5120 x 1280, 6.9 and 6.2).
// Without it the conditions are not there: they cost up to 15 % where nothing is left over (4096 x 2048, gated: 6.6 and 7.8).
template <int NT, int UNROLL, bool REST, typename Tokens, typename Turn>
__device__ __forceinline__ void stream_tiles(f32x4_t (&acc)[NT], const bf16_t* const (&wp)[NT], int wstep, int steps,
                                             Tokens tokens, Turn turn) {
  bf16x8_t wf[2][NT][UNROLL], xf[2][UNROLL];
  const auto ask = [&](auto set, int s, int n) {
    constexpr int B = decltype(set)::value;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
        if (u < n) wf[B][j][u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(wp[j] + (int64_t)(s + u) * wstep));
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      if (u < n) xf[B][u] = tokens(s + u);
  };
  const auto use = [&](auto set, int n) {
    constexpr int B = decltype(set)::value;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      if (u < n)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[B][j][u], xf[B][u], acc[j], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  const int rounds = steps / UNROLL, end = rounds * UNROLL, rest = steps - end;      // (the same in all lanes)
  if (rounds > 0) ask(even, 0, UNROLL);
  else if (REST) ask(even, 0, rest);
  for (int r = 0; r < rounds; r += 2) {
    turn();
    if (r + 1 < rounds) ask(odd, (r + 1) * UNROLL, UNROLL);
    else if (REST) ask(odd, end, rest);
    use(even, UNROLL);
    if (r + 1 < rounds) {
      if (r + 2 < rounds) ask(even, (r + 2) * UNROLL, UNROLL);
      else if (REST) ask(even, end, rest);
      use(odd, UNROLL);
    }
  }
  if (REST) {
    if (rounds % 2) use(odd, rest);
    else use(even, rest);
  }
}

// RESID: y is the residual stream, y = round(y + round(product)) in place: the add that the next norm's kernel would
// have done, with its roundings.
// NT: tiles of 16 weight rows a block owns, next to one another; its waves run them side by side over one copy of the
// activations, which halves what the activations cost where every block reads all of them. A tile's sums are the same
// whatever NT is.
template <int NT, int WPB, int UNROLL, bool TWICE, bool REST, typename OutT, bool TILED, bool RESID = false>
__global__ void __launch_bounds__(WPB * 64) gemm_skinny_kernel(const bf16_t* __restrict__ x,
                                                                const bf16_t* __restrict__ w, OutT* __restrict__ y,
                                                                int M, int N, int K, int round_first, RowScale rs,
                                                                float* __restrict__ stats_out) {
  __shared__ f32x4_t red[WPB > 1 ? (WPB - 1) * NT * WAVE : 1];
  __shared__ f32x4_t red_ss[WPB > 1 ? (WPB - 1) * WAVE : 1];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16;
  const int tile0 = blockIdx.x * NT;
  const int kw = K / WPB;                       // this wave's slice of K (a multiple of 32)
  const int steps = kw / 32;
  const bf16_t* wp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wp[j] = TILED ? w + ((int64_t)(tile0 + j) * (K / 32) + (int64_t)wave * steps) * 512 + lane * 8
                  : w + (int64_t)((tile0 + j) * 16 + c) * K + (int64_t)wave * kw + 8 * g;
  constexpr int WSTEP = TILED ? 512 : 32;       // elements between one product's weights and the next
  const bf16_t* xp = x + (int64_t)c * K + (int64_t)wave * kw + 8 * g;
  const bool have = c < M;                      // token c of the step exists
  f32x4_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  RowSums<WPB> sums;
  sums.start(rs, wave, lane);
  ushort4 before[NT];                           // RESID: the residual values this lane will add to, asked for now so
  if constexpr (RESID) {                        // that they are here when the sums are
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (wave == 0 && have) before[j] = *reinterpret_cast<const ushort4*>(y + (int64_t)c * N + (tile0 + j) * 16 + 4 * g);
  }
  auto tokens = [&](int s) -> bf16x8_t {        // the activations of product s: zeros for a token that is not there
    bf16x8_t xf;
    if (have) {
      xf = *reinterpret_cast<const bf16x8_t*>(xp + s * 32);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) xf[i] = (__bf16)0.f;
    }
    return xf;
  };

  if constexpr (TWICE) {
    stream_tiles<NT, UNROLL, REST>(acc, wp, WSTEP, steps, tokens, [&] { sums.turn(); });
  } else {
    int s = 0;
    for (; s + UNROLL <= steps; s += UNROLL) {
      sums.turn();
      bf16x8_t wf[NT][UNROLL], xf[UNROLL];
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
          wf[j][u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(wp[j] + (int64_t)(s + u) * WSTEP));
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) xf[u] = tokens(s + u);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][u], xf[u], acc[j], 0, 0, 0);
    }
    for (; s < steps; ++s) {
      const bf16x8_t xf = tokens(s);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const bf16x8_t wf = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(wp[j] + (int64_t)s * WSTEP));
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, acc[j], 0, 0, 0);
      }
    }
  }
  f32x4_t ss = sums.finish();
  if (WPB > 1) {
    if (wave > 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j) red[((wave - 1) * NT + j) * WAVE + lane] = acc[j];
      red_ss[(wave - 1) * WAVE + lane] = ss;
    }
    __syncthreads();
    if (wave > 0) return;
    for (int ww = 1; ww < WPB; ++ww) {
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] += red[((ww - 1) * NT + j) * WAVE + lane];
      ss += red_ss[(ww - 1) * WAVE + lane];
    }
  }
  if (rs.stats != nullptr) {                     // the norm's scale of row c, on the float32 sums before they are rounded
    const float inv = 1.0f / sqrtf(row_sum_of_column(ss, c) * rs.inv_dim + rs.eps);
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] *= inv;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    float mine = 0.f;                            // RESID with stats_out: the squares of the residual values written
    if (have) {
      OutT* yp = y + (int64_t)c * N + (tile0 + j) * 16 + 4 * g;
      if constexpr (sizeof(OutT) == 4) {
        f32x4_t o = acc[j];
        if (round_first) {      // the bfloat16 product, widened: what the vendor product of more rows gives, cast up
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = bf16_to_float(float_to_bf16(o[r]));
        }
        *reinterpret_cast<f32x4_t*>(yp) = o;
      } else {
        ushort4 o;
        o.x = float_to_bf16(acc[j][0]); o.y = float_to_bf16(acc[j][1]);
        o.z = float_to_bf16(acc[j][2]); o.w = float_to_bf16(acc[j][3]);
        if (round_first == 4) {      // the squared ReLU of the rounded product, rounded: the two kernels' roundings in one
          const float v0 = fmaxf(bf16_to_float(o.x), 0.f), v1 = fmaxf(bf16_to_float(o.y), 0.f);
          const float v2 = fmaxf(bf16_to_float(o.z), 0.f), v3 = fmaxf(bf16_to_float(o.w), 0.f);
          o.x = float_to_bf16(v0 * v0); o.y = float_to_bf16(v1 * v1);
          o.z = float_to_bf16(v2 * v2); o.w = float_to_bf16(v3 * v3);
        }
        if constexpr (RESID) {
          const ushort4 r = before[j];
          o.x = float_to_bf16(bf16_to_float(r.x) + bf16_to_float(o.x));
          o.y = float_to_bf16(bf16_to_float(r.y) + bf16_to_float(o.y));
          o.z = float_to_bf16(bf16_to_float(r.z) + bf16_to_float(o.z));
          o.w = float_to_bf16(bf16_to_float(r.w) + bf16_to_float(o.w));
          const float v0 = bf16_to_float(o.x), v1 = bf16_to_float(o.y), v2 = bf16_to_float(o.z), v3 = bf16_to_float(o.w);
          mine = ((v0 * v0 + v1 * v1) + v2 * v2) + v3 * v3;
        }
        *reinterpret_cast<ushort4*>(yp) = o;
      }
    }
    if constexpr (RESID) {
      if (stats_out != nullptr) {                // a tile's 16 columns of every row: one partial per row
        const float part = over_lane_groups(mine, c);
        if (g == 0) stats_out[(int64_t)(tile0 + j) * 16 + c] = part;
      }
    }
  }
}

template <int NT, int WPB, int UNROLL, bool TWICE, bool REST, typename OutT, bool RESID>
static void launch_skinny(const void* x, const void* w, void* y, int M, int N, int K, bool tiled, hipStream_t s,
                          int round_first, RowScale rs, float* stats_out) {
  const dim3 grid(N / 16 / NT), block(WPB * 64);
  if constexpr (RESID)
    gemm_skinny_kernel<NT, WPB, UNROLL, TWICE, REST, OutT, true, true><<<grid, block, 0, s>>>((const bf16_t*)x, (const bf16_t*)w,
                                                                                (OutT*)y, M, N, K, round_first, rs, stats_out);
  else if (tiled)
    gemm_skinny_kernel<NT, WPB, UNROLL, TWICE, REST, OutT, true><<<grid, block, 0, s>>>((const bf16_t*)x, (const bf16_t*)w,
                                                                          (OutT*)y, M, N, K, round_first, rs, stats_out);
  else
    gemm_skinny_kernel<NT, WPB, UNROLL, TWICE, REST, OutT, false><<<grid, block, 0, s>>>((const bf16_t*)x, (const bf16_t*)w,
                                                                           (OutT*)y, M, N, K, round_first, rs, stats_out);
}

// How many waves share a tile, from the shapes alone (a result never depends on M): 16 up to 319 tiles, 8 from there. How many
// tiles a block owns and how many loads wait in which form changes no result, so it may follow M. Measured on MI355X, in us at
// 1 / 8 / 16 rows (in brackets: 8 loads in one set of registers, two tiles a block from 320 to 512 tiles and, from 10 rows
// up, beyond 4,096):
//   up to 319 tiles: one, two sets of 4 loads. 2048 x 8192 9.7 / 11.4 / 14.5 (11.6 / 12.4 / 15.3), 4096 x 4096 7.8 / 8.3 / 9.3
//     (8.3 / 8.5 / 10.0). Where the residual is added, 8 loads in one set: behind the kernels of a step of four rows, which leave
//     4096 x 4096 and 4096 x 12288 cold, two sets took 13.9 on average and one 13.4.
//     (8 waves where K is no multiple of 512: two sets of 4 up to 256 tiles, 4096 x 11008 17.5 / 19.2 / 22.6 (18.9 / 21.2 / 23.4;
//     two tiles, half the units without a block, 22.7 / 25.5 / 29.1), 2816 x 2816 6.3 / 6.8 / 7.8 (6.8 / 7.4 / 8.0; 9.0 / 9.7 / 9.6);
//     from there one set of 4, 5104 x 3328 10.1 / 11.3 / 13.5 (11.4 / 12.0 / 14.8; two sets 10.7 / 11.9 / 14.7), and above 8 rows
//     two tiles, 4608 x 2816 at 16 rows 10.0 (12.6; one tile 12.3).)
//   320 to 511: two (at 512, one: 8192 x 4096 13.8 / 15.1 / 16.0, two 15.0 / 16.1 / 16.0); two sets of 4 loads a tile up to 8 rows,
//     of 2 above: 6144 x 4096 11.5 / 12.8 / 12.7 (12.0 / 12.9 / 14.3), 6144 x 5120 13.3 / 14.8 / 15.4 (16.8 / 17.8 / 19.1).
//   from 1,024, and K below 4,096 or more than 8 rows: two, two sets of 2 loads a tile: 18432 x 2048 15.5 / 16.0 / 17.7 (15.6 /
//     16.8 / 20.0), 36864 x 2048 26.2 / 26.3 / 28.4 (26.3 / 29.0 / 34.7), 24576 x 3072 26.3 / 26.5 / 28.6 (29.6 / 32.4 / 39.4).
//   otherwise one, 4 loads in one set, which is what 8 waves a block and several blocks a unit need least registers for: 12288 x
//     4096 19.4 / 20.0 / 23.3 (19.5 / 20.6 / 25.3; two tiles 22.8 / 23.6 / 24.7), 9216 x 2048 9.5 / 10.1 / 11.5 (9.7 / 10.7 /
//     12.6), 151936 x 4096 182 / 190 (184 / 199; two tiles, for 16 rows, 206, where one takes 243 and took 225).
//   fewer than 8 waves: one, two sets of 8 loads up to 1,024 waves in all, of 4 from there, where registers bound how many of them are
//     on the chip: 5632 x 1472 6.3 / 6.8 / 7.4 (12.3 / 12.6 / 13.0; sets of 4 7.2 / 7.4 / 7.8), 18432 x 704 6.6 / 7.0 / 8.2 (8.1 / 8.4
//     / 9.4; sets of 8 8.0 / 8.3 / 9.6), 7168 x 2688 9.2 / 9.7 / 11.6 (13.9 / 14.3 / 14.9; sets of 8 9.9 / 10.9 / 12.3).
static bool skinny_two(int tiles, int K, int M) {
  return skinny_waves(tiles, K) == 8 && tiles % 2 == 0 &&
         ((tiles >= (M > 8 ? 257 : 320) && tiles < 512) || (tiles >= 1024 && (K < 4096 || M > 8)));
}

template <typename OutT, bool RESID = false>
static int pick_waves(const void* x, const void* w, void* y, int M, int N, int K, bool tiled, hipStream_t s,
                      int round_first = 0, RowScale rs = RowScale{nullptr, 0, 0.f, 0.f}, float* stats_out = nullptr) {
  const int tiles = N / 16;
  const int wpb = skinny_waves(tiles, K);
  const bool two = skinny_two(tiles, K, M);
  const int steps = K / 32 / wpb;
#define SKINNY(NT, WPB, U, TWICE, REST) \
  launch_skinny<NT, WPB, U, TWICE, REST, OutT, RESID>(x, w, y, M, N, K, tiled, s, round_first, rs, stats_out)
#define SKINNY_TWICE(NT, WPB, U)                      \
  do {                                                \
    if (steps % U) SKINNY(NT, WPB, U, true, true);    \
    else SKINNY(NT, WPB, U, true, false);             \
  } while (0)
  switch (wpb) {
    case 16:
      if constexpr (RESID) { SKINNY(1, 16, 8, false, false); } else { SKINNY_TWICE(1, 16, 4); }
      break;
    case 8:
      if (tiles <= 256) SKINNY_TWICE(1, 8, 4);
      else if (!two) SKINNY(1, 8, 4, false, false);
      else if (tiles < 512 && M <= 8) SKINNY_TWICE(2, 8, 4);
      else SKINNY_TWICE(2, 8, 2);
      break;
    // (fewer than 8: an odd number of steps a wave)
    case 4: if (tiles <= 256) SKINNY(1, 4, 8, true, true); else SKINNY(1, 4, 4, true, true); break;
    case 2: if (tiles <= 512) SKINNY(1, 2, 8, true, true); else SKINNY(1, 2, 4, true, true); break;
    default: SKINNY(1, 1, 8, true, true); break;
  }
#undef SKINNY_TWICE
#undef SKINNY
  return 0;
}

// How many tiles of 16 columns a block owns.
extern "C" int holon_gemm_skinny_tiles(int M, int N, int K) { return skinny_two(N / 16, K, M) ? 2 : 1; }

extern "C" int holon_gemm_skinny_supported(int M, int N, int K) {
  return M >= 1 && M <= 16 && N % 16 == 0 && K % 32 == 0 && K >= 32;
}

// out_f32: 0 writes bfloat16, 1 float32 straight from the accumulators, 2 float32 values that were rounded to bfloat16
// first (the product in the operands' type, cast up), 4 bfloat16 again: max(product, 0)^2 of the rounded product (a
// feed-forward's squared ReLU in the product's epilogue). tiled: 1 when `w` is in the tile layout (see holon_tile_weight_bf16).
extern "C" int holon_gemm_skinny_bf16(const void* x, const void* w, void* y, int M, int N, int K, int out_f32,
                                      int tiled, void* stream) {
  HOLON_CHECK(holon_gemm_skinny_supported(M, N, K), "gemm (few rows): M=%d N=%d K=%d not served (M <= 16, N %% 16, K %% 32)",
              M, N, K);
  hipStream_t s = (hipStream_t)stream;
  HOLON_CHECK(out_f32 == 0 || out_f32 == 1 || out_f32 == 2 || out_f32 == 4, "gemm (few rows): no output form %d", out_f32);
  if (out_f32 == 4) pick_waves<bf16_t>(x, w, y, M, N, K, tiled != 0, s, 4);
  else if (out_f32) pick_waves<float>(x, w, y, M, N, K, tiled != 0, s, out_f32 == 2);
  else pick_waves<bf16_t>(x, w, y, M, N, K, tiled != 0, s);
  HOLON_LAUNCH_OK();
  return 0;
}

// The same product over rows that a folded norm has yet to scale: `w_tiled` holds W * diag(g), x the un-normed rows,
// `stats` [parts, 16] the partial sums of squares of x's rows; row m of the result is scaled by
// rsqrt(sum(stats[:, m]) / K + eps) before it is rounded.
extern "C" int holon_gemm_skinny_scaled_bf16(const void* x, const void* w_tiled, void* y, int M, int N, int K,
                                             int out_f32, const float* stats, int parts, float eps, void* stream) {
  HOLON_CHECK(holon_gemm_skinny_supported(M, N, K) && stats != nullptr && parts >= 1,
              "gemm (few rows, folded norm): M=%d N=%d K=%d parts=%d not served (M <= 16, N %% 16, K %% 32)", M, N, K, parts);
  const RowScale rs{stats, parts, eps, 1.0f / (float)K};
  hipStream_t s = (hipStream_t)stream;
  if (out_f32) pick_waves<float>(x, w_tiled, y, M, N, K, true, s, out_f32 == 2, rs);
  else pick_waves<bf16_t>(x, w_tiled, y, M, N, K, true, s, 0, rs);
  HOLON_LAUNCH_OK();
  return 0;
}

// residual[M, N] += x[M, K] w^T in place (the product rounded, then the sum rounded) over tiled weights: the output
// projection's product and the residual add that follows it, in one kernel. With `stats_out` ([N / 16, 16] float32)
// it also leaves, per block of 16 columns, the sums of squares of the residual values it wrote: what a norm over the
// new rows needs.
extern "C" int holon_gemm_skinny_add_bf16(const void* x, const void* w_tiled, void* residual, int M, int N, int K,
                                          float* stats_out, void* stream) {
  HOLON_CHECK(holon_gemm_skinny_supported(M, N, K),
              "gemm (few rows, added to the residual): M=%d N=%d K=%d not served (M <= 16, N %% 16, K %% 32)", M, N, K);
  pick_waves<bf16_t, true>(x, w_tiled, residual, M, N, K, true, (hipStream_t)stream, 0,
                           RowScale{nullptr, 0, 0.f, 0.f}, stats_out);
  HOLON_LAUNCH_OK();
  return 0;
}

// Several products of the same up to 16 rows that do not read one another's results, in one launch: each with operands, sizes and an output
// form of its own, every sum in the order that the product by itself has. What bounds them one by one is not the weights: 2048 x 2048 by
// itself takes 4.6 us in a step, of which its 8 MB are 1.2, the rest the kernel's start and end and a round of memory latency. Measured in a
// step of one row, us, against the products one after the other: seven of 2,048 to 3,072 columns and one of 64 over 2,048 of K 12.5 (34);
// 3,072 and 8,192 columns over 2,048 10.5 (12.9); 2,048 columns over 2,048 and over 8,192 of K 10.2 (13.9): 4.1 to 4.4 TB/s.
// A block holds 16 waves: one tile of 16 columns whose K goes over 16 waves, two of 8 waves and so on; blocks with the most columns of K a
// wave come first. SHORT: no wave has more than four steps of K, so that its loads need half the registers and a unit holds two blocks.
constexpr int GROUP_MOST = 8, GROUP_WAVES = 16;
struct GroupItem {
  const bf16_t* x;
  const bf16_t* w;             // tiled
  void* y;
  int N, K, waves, form;       // waves a tile; form as out_f32 of holon_gemm_skinny_bf16
  int first;                   // the item's first block
};
struct GroupItems {
  GroupItem at[GROUP_MOST];
  int count, M;
};
// A mixture's router over the same number of rows, a block a row in front of the products' blocks: by itself it is one wave's chain of
// choices behind the logits' round of memory latency, 4.8 to 6.1 us in which nothing else runs.
struct GroupRoute {
  const bf16_t* x;
  const float* router;
  const float* bias;
  float* weights;
  int width, experts, rows_r, top, groups, keep, score;
  float scale;
};

template <bool SHORT, bool REST, bool ROUTE>
__global__ void __launch_bounds__(GROUP_WAVES * 64, SHORT && !ROUTE ? 8 : 4) gemm_skinny_group_kernel(GroupItems items, GroupRoute route) {
  __shared__ f32x4_t red[GROUP_WAVES * WAVE];
  int block = blockIdx.x;
  if constexpr (ROUTE) {
    static_assert(moe_router::BLOCK_WAVES == GROUP_WAVES && sizeof(moe_router::Lds) <= sizeof(red), "the router's block");
    if (block < items.M) {
      moe_router::Lds& lds = *reinterpret_cast<moe_router::Lds*>(red);
      if (route.score < 0)
        moe_router::few_token<bf16_t, 1>(lds, block, route.x, route.router, route.bias, route.weights, route.width, route.experts,
                                         route.rows_r, route.top, route.groups, route.keep, route.score, route.scale);
      else
        moe_router::few_token<bf16_t, 4>(lds, block, route.x, route.router, route.bias, route.weights, route.width, route.experts,
                                         route.rows_r, route.top, route.groups, route.keep, route.score, route.scale);
      return;
    }
    block -= items.M;
  }
  const int all = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  int n = 0;
  while (n + 1 < items.count && block >= items.at[n + 1].first) ++n;
  const GroupItem it = items.at[n];
  const int wave = all % it.waves, tile = (block - it.first) * (GROUP_WAVES / it.waves) + all / it.waves;
  const bool have = c < items.M, mine = tile < it.N / 16;
  const int steps = mine ? it.K / 32 / it.waves : 0;
  f32x4_t acc[1] = {{0.f, 0.f, 0.f, 0.f}};
  const bf16_t* const wp[1] = {it.w + ((int64_t)tile * (it.K / 32) + (int64_t)wave * steps) * 512 + lane * 8};
  const bf16_t* xp = it.x + (int64_t)c * it.K + (int64_t)wave * steps * 32 + 8 * g;
  const auto tokens = [&](int s) -> bf16x8_t {
    bf16x8_t xf;
    if (have) {
      xf = *reinterpret_cast<const bf16x8_t*>(xp + s * 32);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) xf[i] = (__bf16)0.f;
    }
    return xf;
  };
  if constexpr (SHORT) {
    bf16x8_t wf[4], xf[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < steps) {
        wf[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(wp[0] + (int64_t)u * 512));
        xf[u] = tokens(u);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < steps) acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf[u], acc[0], 0, 0, 0);
  } else {
    stream_tiles<1, 4, REST>(acc, wp, 512, steps, tokens, [] {});
  }
  red[all * WAVE + lane] = acc[0];
  __syncthreads();
  if (wave > 0 || !mine) return;
  for (int ww = 1; ww < it.waves; ++ww) acc[0] += red[(all + ww) * WAVE + lane];
  if (!have) return;
  const int64_t at = (int64_t)c * it.N + tile * 16 + 4 * g;
  ushort4 o;
  bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
  for (int r = 0; r < 4; ++r) oe[r] = float_to_bf16(acc[0][r]);
  if (it.form == 2) {
    f32x4_t wide;
#pragma unroll
    for (int r = 0; r < 4; ++r) wide[r] = bf16_to_float(oe[r]);
    *reinterpret_cast<f32x4_t*>((float*)it.y + at) = wide;
    return;
  }
  if (it.form == 4)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = fmaxf(bf16_to_float(oe[r]), 0.f);
      oe[r] = float_to_bf16(v * v);
    }
  *reinterpret_cast<ushort4*>((bf16_t*)it.y + at) = o;
}

// `items`: `count` (up to 8) of 3 pointers (x [M, K], w tiled, y [M, N]) and 3 sizes (N, K, form: 0 bfloat16, 2 float32 values that were
// rounded to bfloat16 first, 4 bfloat16 max(product, 0)^2). `route` (nullable): 4 pointers (x [M, width], router [rows, width], bias or 0,
// weights [M, rows]) and 7 numbers (width, experts, rows, top, groups, keep, score) of a router as holon_moe_router (score -1) and
// holon_moe_router_top have them, of up to 64 experts.
extern "C" int holon_gemm_skinny_group_bf16(const int64_t* items, int count, int M, const int64_t* route, float scale, void* stream) {
  HOLON_CHECK(count >= 1 && count <= GROUP_MOST && M >= 1 && M <= 16, "gemm (few rows, several): %d products of %d rows", count, M);
  GroupItems g{};
  g.count = count;
  g.M = M;
  for (int i = 0; i < count; ++i) {
    const int64_t* v = items + 6 * i;
    GroupItem it{(const bf16_t*)v[0], (const bf16_t*)v[1], (void*)v[2], (int)v[3], (int)v[4], 0, (int)v[5], 0};
    HOLON_CHECK(holon_gemm_skinny_supported(M, it.N, it.K) && ((v[0] | v[1] | v[2]) & 15) == 0 &&
                    (it.form == 0 || it.form == 2 || it.form == 4),
                "gemm (few rows, several): M=%d N=%d K=%d form %d not served (N %% 16, K %% 32, operands at 16 bytes)", M, it.N, it.K, it.form);
    it.waves = skinny_waves(it.N / 16, it.K);
    int at = i;                                             // longest runs of K first
    for (; at > 0 && g.at[at - 1].K / g.at[at - 1].waves < it.K / it.waves; --at) g.at[at] = g.at[at - 1];
    g.at[at] = it;
  }
  int blocks = 0;
  bool is_short = true, rest = false;
  for (int i = 0; i < count; ++i) {
    GroupItem& it = g.at[i];
    const int per = GROUP_WAVES / it.waves, steps = it.K / 32 / it.waves;
    it.first = blocks;
    blocks += (it.N / 16 + per - 1) / per;
    is_short = is_short && steps <= 4;
    rest = rest || steps % 4 != 0;
  }
  hipStream_t s = (hipStream_t)stream;
  GroupRoute r{};
  if (route != nullptr) {
    r = {(const bf16_t*)route[0], (const float*)route[1], (const float*)route[2], (float*)route[3], (int)route[4], (int)route[5], (int)route[6],
         (int)route[7], (int)route[8], (int)route[9], (int)route[10], scale};
    HOLON_CHECK(r.x && r.router && r.weights && r.width >= 1 && r.width <= 12288 && r.experts >= 1 && r.experts <= WAVE && r.top >= 1 &&
                    r.top <= r.experts && (r.rows_r == r.experts || (r.score >= 0 && r.rows_r == r.experts + 1)) && r.score >= -1 && r.score <= 2 &&
                    (r.groups <= 1 || (r.experts % r.groups == 0 && r.keep >= 1 && r.keep <= r.groups &&
                                       (r.score < 0 || r.top <= r.keep * (r.experts / r.groups)))),
                "gemm (few rows, several): a router of width %d, top %d of %d experts, %d rows, %d of %d groups, score %d not served", r.width,
                r.top, r.experts, r.rows_r, r.keep, r.groups, r.score);
    blocks += M;
  }
#define GROUP(SHORT, REST)                                                                                       \
  do {                                                                                                           \
    if (route != nullptr) gemm_skinny_group_kernel<SHORT, REST, true><<<blocks, GROUP_WAVES * 64, 0, s>>>(g, r); \
    else gemm_skinny_group_kernel<SHORT, REST, false><<<blocks, GROUP_WAVES * 64, 0, s>>>(g, r);                 \
  } while (0)
  if (is_short) GROUP(true, false);
  else if (rest) GROUP(false, true);
  else GROUP(false, false);
#undef GROUP
  HOLON_LAUNCH_OK();
  return 0;
}

// The gated form: w = [gate rows; up rows] (2I rows), y[M, I] = round(act(round(x gate^T))) * round(x up^T), act silu or
// (ACT 1) the tanh form of gelu, the roundings of the two-kernel composition. A block owns gate tile t and up tile t + I/16 and streams both.
template <int WPB, int UNROLL, bool REST, bool TILED, int ACT>
__global__ void __launch_bounds__(WPB * 64) gemm_skinny_glu_kernel(const bf16_t* __restrict__ x,
                                                                    const bf16_t* __restrict__ w,
                                                                    bf16_t* __restrict__ y, int M, int I, int K,
                                                                    RowScale rs) {
  __shared__ f32x4_t red[WPB > 1 ? (WPB - 1) * 2 * WAVE : 1];
  __shared__ f32x4_t red_ss[WPB > 1 ? (WPB - 1) * WAVE : 1];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16;
  const int n0 = blockIdx.x * 16;
  const int kw = K / WPB, steps = kw / 32;
  const bf16_t* wp[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t tile = blockIdx.x + (int64_t)h * (I / 16);
    wp[h] = TILED ? w + (tile * (K / 32) + (int64_t)wave * steps) * 512 + lane * 8
                  : w + (tile * 16 + c) * K + (int64_t)wave * kw + 8 * g;
  }
  constexpr int WSTEP = TILED ? 512 : 32;
  const bf16_t* xp = x + (int64_t)c * K + (int64_t)wave * kw + 8 * g;
  const bool have = c < M;
  f32x4_t acc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
  RowSums<WPB> sums;
  sums.start(rs, wave, lane);
  auto tokens = [&](int s) -> bf16x8_t {
    bf16x8_t xf;
    if (have) {
      xf = *reinterpret_cast<const bf16x8_t*>(xp + s * 32);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) xf[i] = (__bf16)0.f;
    }
    return xf;
  };
  stream_tiles<2, UNROLL, REST>(acc, wp, WSTEP, steps, tokens, [&] { sums.turn(); });
  f32x4_t ss = sums.finish();
  if (WPB > 1) {
    if (wave > 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) red[((wave - 1) * 2 + h) * WAVE + lane] = acc[h];
      red_ss[(wave - 1) * WAVE + lane] = ss;
    }
    __syncthreads();
    if (wave > 0) return;
    for (int ww = 1; ww < WPB; ++ww) {
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[h] += red[((ww - 1) * 2 + h) * WAVE + lane];
      ss += red_ss[(ww - 1) * WAVE + lane];
    }
  }
  if (rs.stats != nullptr) {
    const float inv = 1.0f / sqrtf(row_sum_of_column(ss, c) * rs.inv_dim + rs.eps);
    acc[0] *= inv;
    acc[1] *= inv;
  }
  if (!have) return;
  ushort4 o;
  bf16_t* oe = reinterpret_cast<bf16_t*>(&o);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float gate = bf16_to_float(float_to_bf16(acc[0][r]));
    const float up = bf16_to_float(float_to_bf16(acc[1][r]));
    const float sg = bf16_to_float(float_to_bf16(gate_act<ACT, bf16_t>(gate)));
    oe[r] = float_to_bf16(sg * up);
  }
  *reinterpret_cast<ushort4*>(y + (int64_t)c * I + n0 + 4 * g) = o;
}

// `stats` (nullable, with `parts` and `eps`): x holds un-normed rows and `w` the tiled weights with the norm's weight
// folded in; rows are scaled as in holon_gemm_skinny_scaled_bf16 (tiled).
template <int ACT>
static int skinny_glu(const void* x, const void* w, void* y, int M, int I, int K, int tiled, const float* stats, int parts,
                      float eps, void* stream) {
  HOLON_CHECK(M >= 1 && M <= 16 && I % 16 == 0 && K % 128 == 0, "gated gemm (few rows): M=%d I=%d K=%d not served", M, I, K);
  HOLON_CHECK(stats == nullptr || (tiled && parts >= 1), "gated gemm (few rows, folded norm): tiled=%d parts=%d", tiled, parts);
  const RowScale rs{stats, parts, eps, 1.0f / (float)K};
  hipStream_t s = (hipStream_t)stream;
  // few tile pairs: four waves share each; otherwise two. At 1 / 8 / 16 rows 768 pairs over K = 4,096 take 34.4 / 34.3 / 35.0 us,
  // 384 over 2,048 11.6 / 12.3 / 13.3 (35.4 / 35.7 / 36.6 and 12.1 / 13.3 / 14.6 with 8 loads in one set of registers).
  const bool few = I / 16 < 512;
#define GLU(WPB, U, REST)                                                                                              \
  do {                                                                                                                 \
    if (tiled) gemm_skinny_glu_kernel<WPB, U, REST, true, ACT><<<I / 16, WPB * 64, 0, s>>>((const bf16_t*)x, (const bf16_t*)w, \
                                                                                     (bf16_t*)y, M, I, K, rs);         \
    else gemm_skinny_glu_kernel<WPB, U, REST, false, ACT><<<I / 16, WPB * 64, 0, s>>>((const bf16_t*)x, (const bf16_t*)w,      \
                                                                                (bf16_t*)y, M, I, K, rs);              \
  } while (0)
  const bool rest = K / 32 / (few ? 4 : 2) % 4 != 0;
  if (few && rest) GLU(4, 4, true);
  else if (few) GLU(4, 4, false);
  else if (rest) GLU(2, 4, true);
  else GLU(2, 4, false);
#undef GLU
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_gemm_skinny_glu_bf16(const void* x, const void* w, void* y, int M, int I, int K, int tiled,
                                          const float* stats, int parts, float eps, void* stream) {
  return skinny_glu<0>(x, w, y, M, I, K, tiled, stats, parts, eps, stream);
}

// The same with the tanh form of gelu in place of silu.
extern "C" int holon_gemm_skinny_geglu_bf16(const void* x, const void* w, void* y, int M, int I, int K, int tiled,
                                            void* stream) {
  return skinny_glu<1>(x, w, y, M, I, K, tiled, nullptr, 0, 0.f, stream);
}

// tiled[t][s][l][e] = w[16 t + l % 16][32 s + 8 (l / 16) + e]: the layout the few-row product streams.
// With `scale` [K]: tiled holds round(w[n][k] * scale[k]), a norm's weight folded into the columns it multiplies.
__global__ void tile_weight_kernel(const bf16_t* __restrict__ w, bf16_t* __restrict__ tiled, int N, int K,
                                   const bf16_t* __restrict__ scale) {
  const int64_t chunks = (int64_t)N * K / 8;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < chunks; i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i % 64);
    const int64_t ts = i / 64;
    const int64_t step = ts % (K / 32), tile = ts / (K / 32);
    const int64_t col = step * 32 + 8 * (lane / 16);
    const int64_t src = (tile * 16 + lane % 16) * K + col;
    uint4 v = *reinterpret_cast<const uint4*>(w + src);
    if (scale != nullptr) {
      bf16_t* e = reinterpret_cast<bf16_t*>(&v);
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = float_to_bf16(bf16_to_float(e[j]) * bf16_to_float(scale[col + j]));
    }
    *reinterpret_cast<uint4*>(tiled + i * 8) = v;
  }
}

extern "C" int holon_tile_weight_bf16(const void* w, void* tiled, int N, int K, const void* scale, void* stream) {
  HOLON_CHECK(N > 0 && K > 0 && N % 16 == 0 && K % 32 == 0, "tile_weight: N=%d K=%d must be multiples of 16 and 32", N, K);
  tile_weight_kernel<<<4096, 256, 0, (hipStream_t)stream>>>((const bf16_t*)w, (bf16_t*)tiled, N, K, (const bf16_t*)scale);
  HOLON_LAUNCH_OK();
  return 0;
}
