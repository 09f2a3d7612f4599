// y[M, N] = x[M, K] w[N, K]^T in true float32: float32 operands on the matrix cores (v_mfma_f32_16x16x4_f32: no
// reduced-precision mode), float32 accumulation. This is the product of the 32-bit path.
//
// Its point is a fixed order of summation, the same in all forms of shares below: K is cut into 16 shares of equal length
// (64, or a larger multiple of 32; the last ones shorter or empty); a share's sum runs over its k in groups of 16 (the instruction adds
// k, k + 4, k + 8 and k + 12 of a group at a time), four shares are added up one after the other, and so are the four
// quarters that makes. None of it depends on M, on where the row lies in the batch, or on the tile of the output the
// element falls in (rows and columns beyond the edge repeat the last one and are never stored; what lies beyond K is
// taken as zeros, which add nothing). So a token's result is bit for bit the same whether it runs alone, in a portion
// of a prompt or in a batch of others.
//
// A lane of a matrix instruction's operand holds one float of row lane % 16; here it reads four neighbours in k at once
// (16 bytes, k = 4 (lane / 16) .. + 3 of a group) and spends them on four instructions.
#include "gemm_f32.h"
#include "holon_hip.h"

namespace {
using namespace f32_sums;

// Steps of few rows. A block owns MT x NT tiles of 16 x 16 results; each of its 16 waves takes one share of K, and the waves' sums are added in
// order through LDS. Operands go from memory straight to registers, DEPTH groups of k of a wave under way at a time; 16
// waves on four SIMDs cover each other's loads, so nothing is staged and no wave waits for another before the end. With
// few rows that streams the weights (bound by memory: a lane has DEPTH 16-byte loads in flight); with many the matrix
// cores bound it, as a group of k is 4 MT NT instructions of 32 cycles for MT + NT loads.
template <int MT, int NT, int DEPTH, bool VEC>
__global__ void __launch_bounds__(SHARES * WAVE) gemm_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                  float* __restrict__ y, int M, int N, int K) {
  __shared__ f32x4_t part[SHARES][MT * NT][WAVE];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16;
  const int n0 = blockIdx.x * NT * 16, m0 = blockIdx.y * MT * 16;
  const int share = share_length(K);
  const int first = wave * share, last = min(K, first + share);
  const float *wr[NT], *xr[MT];
#pragma unroll
  for (int u = 0; u < NT; ++u) wr[u] = w + (int64_t)min(n0 + u * 16 + c, N - 1) * K;
#pragma unroll
  for (int t = 0; t < MT; ++t) xr[t] = x + (int64_t)min(m0 + t * 16 + c, M - 1) * K;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  share_sums<MT, NT, DEPTH, VEC>(acc, wr, xr, first, last);
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) part[wave][t * NT + u][lane] = acc[t][u];
  __syncthreads();
  // lane holds columns 4 g .. 4 g + 3 of row c of tile `wave`
  if (wave >= MT * NT) return;
  const f32x4_t sum = sum_shares([&](int i) { return part[i][wave][lane]; });
  store4(y, sum, m0 + wave / NT * 16 + c, n0 + wave % NT * 16 + 4 * g, M, N);
}

// Up to 16 rows over at most 128 tiles of 16 columns, which a block each leave half the compute units idle: a block half a tile. Tiles
// against halves at 1 / 16 rows, us: 2048 x 2048 7.4 / 10.4 and 6.3 / 9.2, 2048 x 8192 27.6 / 38.5 and 20.2 / 28.7, 2048 x 18432 55 / 85
// and 44 / 59; of 192 tiles (3072 x 2048) 9.2 / 12.5 and 10.8 / 14.3. More loads under way change nothing in either form.
constexpr int HALF_TILES = 128;
template <int DEPTH, bool VEC>
__global__ void __launch_bounds__(SHARES * WAVE) gemm_f32_half_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                  float* __restrict__ y, int M, int N, int K) {
  __shared__ f32x4_t part[SHARES][WAVE];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int g = lane / 16, c = lane % 16, n0 = blockIdx.x * 8, share = share_length(K);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  half_sums<DEPTH, VEC>(acc, w + (int64_t)min(n0 + c % 8, N - 1) * K, x + (int64_t)min(c, M - 1) * K, wave * share,
                        min(K, (wave + 1) * share));
  part[wave][lane] = acc;
  __syncthreads();
  if (wave > 0 || g > 1) return;
  const f32x4_t sum = sum_shares([&](int i) { return part[i][lane]; });
  store4(y, sum, c, n0 + 4 * g, M, N);
}

template <int SIDE, int MT, int NT, How HOW>
__global__ void __launch_bounds__(SIDE * 256, SIDE > 1 ? 4 : (MT == 2 && NT == 2 && HOW == DIRECT ? 5 : 1)) gemm_f32_kernel(
    const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) Stage<SIDE, MT, NT> stage;
  const int m0 = blockIdx.y * 32 * MT, n0 = blockIdx.x * 32 * NT, r0 = threadIdx.x % 256 / 8;
  const float *xr[MT], *wr[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xr[i] = x + (int64_t)min(m0 + r0 + 32 * i, M - 1) * K;
#pragma unroll
  for (int i = 0; i < NT; ++i) wr[i] = w + (int64_t)min(n0 + r0 + 32 * i, N - 1) * K;
  tile_sums<SIDE, MT, NT, HOW>(stage, xr, wr, K, [&](f32x4_t sum, int row, int column) { store4(y, sum, m0 + row, n0 + column, M, N); });
}

// Long sums into many columns: one running sum over k = 0, 1, 2, ... (v_mfma_f32_32x32x2_f32 adds its two k one after the
// other), the order of a plain float32 product. What the 32-bit path of a model of these sizes is held against is the same model
// in plain float32 products, and the rounding of those alone, most of it the query and key projection's (6,144 columns over K =
// 4,096), is 2.1e-5 of the logits' rms at 36 layers: sums in shares come 3 times closer to 64 bits (8e-6) and lie 2.1e-5 from
// the plain model where 2e-5 are allowed; these lie 1.9e-5 from it. (A product that is exact would lie 2.1e-5 from it too.) The order
// costs time, most with few rows, as nothing shares K: 6144 x 4096 takes 223 / 273 / 285 / 433 us at 1 / 64 / 300 / 704 rows, in
// shares 27 / 67 / 158 / 387.
// A workgroup of four waves owns a 64 x 64 tile of the output, each wave a 32 x 32 quarter. Per step the workgroup stages 64
// rows of x and 64 rows of w, 32 k wide, in LDS (rows padded to 33 floats: a wave's 32 rows then fall in 32 different banks).
constexpr int TM = 64, TN = 64, TK = 32, PAD = 1;
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__host__ __device__ __forceinline__ bool sums_in_order(int N, int K) { return K >= 4096 && N > K; }

// VEC: K is a multiple of 4 and both operands are 16-byte aligned, so rows are read four floats at a time.
template <bool VEC>
__device__ __forceinline__ void stage_rows(const float* __restrict__ src, int rows, int K, int row0, int k0,
                                           float (*dst)[TK + PAD]) {
  // 64 rows x 32 floats = 512 groups of four; 256 threads take two each
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int idx = threadIdx.x + it * 256;
    const int r = idx / (TK / 4), c = (idx % (TK / 4)) * 4;
    const int row = row0 + r, k = k0 + c;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row < rows) {
      const float* p = src + (int64_t)row * K + k;
      if (VEC) {
        if (k < K) v = *reinterpret_cast<const float4*>(p);      // K % 4 == 0: a group is inside or outside whole
      } else {
        if (k + 0 < K) v.x = p[0];
        if (k + 1 < K) v.y = p[1];
        if (k + 2 < K) v.z = p[2];
        if (k + 3 < K) v.w = p[3];
      }
    }
    dst[r][c + 0] = v.x; dst[r][c + 1] = v.y; dst[r][c + 2] = v.z; dst[r][c + 3] = v.w;
  }
}

template <bool VEC>
__global__ void __launch_bounds__(256) gemm_f32_in_order_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       float* __restrict__ y, int M, int N, int K) {
  __shared__ float xs[TM][TK + PAD];
  __shared__ float ws[TN][TK + PAD];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int wm = wave / 2, wn = wave % 2;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int r = lane % 32, half = lane / 32;
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  for (int k0 = 0; k0 < K; k0 += TK) {
    stage_rows<VEC>(x, M, K, m0, k0, xs);
    stage_rows<VEC>(w, N, K, n0, k0, ws);
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; kk += 2) {
      const float a = xs[wm * 32 + r][kk + half];
      const float b = ws[wn * 32 + r][kk + half];
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
    }
    __syncthreads();
  }
  // lane holds column n = r of rows 8 (i / 4) + 4 half + i % 4
  const int n = n0 + wn * 32 + r;
  if (n >= N) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int m = m0 + wm * 32 + 8 * (i / 4) + 4 * half + i % 4;
    if (m < M) y[(int64_t)m * N + n] = acc[i];
  }
}

// Which form a product takes: the one that is done first by a fit on MI355X over 400 products of K = 32 to 18,432, N = 64 to 16,384 and M =
// 17 to 2,048, weights from memory (1.6 GB of them in turn: back to back over three weights that stay in the last-level cache, staged forms
// look up to a third faster than behind a model's other products), in us: a start, and so much for every round of one block a CU, linear in K.
// Tiles straight from memory add a part of K to that; of staged ones a block that has its unit to itself takes longer than its share of a full
// one, `start_k` a k. The choice is 0.3 % from the best form on average and 9 % at most; over 2,850 products that the fit has not seen 0.6 and 11 %
// from K = 512 on, up to 24 % below (of 3 to 15 us, where K is 64 or less). In us, best and others: 2048 x 2048 takes 1 x 1 tiles up to 32 rows (10; with a 64 x 64 tile a
// block and no split of K it took 118), 1 x 2 at 64 (16), 2 x 4 at 145 (34; staged 39 to 48), quarters side by side from 300 rows (39; one
// after the other 48), blocks of 32 rows at 700 (65; of 64 rows 76, whose second round is mostly empty); 2048 x 9248 at 704 rows blocks of
// 32 (274; of 64 312); 16384 x 2048 1 x 1 tiles up to 16 rows (5.0 TB/s at one row), blocks of 32 at 150 (117; of 64 122), of 64 at 825
// (493; of 32 596); 9248 x 256 at 2,048 rows of 64 one after the other (102; side by side 143).
struct Form { int mt, nt; float start, start_k, round, round_k; };
enum { SIDE_BY_SIDE = 4, IN_TURN = 5, IN_TURN_32 = 6, KINDS = 7 };
constexpr Form FORMS[KINDS] = {{1, 1, 1.7f, 6.67e-4f, 0.425f, 3.27e-3f},  {1, 2, 2.06f, 7.5e-4f, 0.613f, 5.89e-3f},
                               {2, 2, 2.34f, 1.28e-3f, 0.911f, 7.33e-3f}, {2, 4, 1.0f, 1.24e-3f, 3.19f, 1.36e-2f},
                               {4, 4, 0.872f, 6.47e-3f, 3.39f, 1.69e-2f}, {4, 4, 3.63f, 2.16e-2f, 0.607f, 1.72e-2f},
                               {2, 4, 1.73f, 1.98e-2f, 0.657f, 1.03e-2f}};
// Operands that cannot be copied straight into LDS (K off a multiple of 32, or not on 16 bytes) pass registers, in tiles of 64 x 64: a fit of
// their own (1,149 products), each time the sum of all its terms; within 1 % of the best on average over the 400 above, too.
constexpr Form BY_REGISTERS[KINDS - 1] = {{1, 1, 2.6f, 2e-4f, 0.43f, 3.25e-3f}, {1, 2, 2.5f, 2e-4f, 0.63f, 5.0e-3f},
                                          {2, 2, 2.5f, 7e-4f, 0.90f, 7.35e-3f}, {2, 4, 1.2f, 5e-4f, 3.0f, 1.31e-2f},
                                          {4, 4, 1.2f, 0.f, 3.2f, 1.86e-2f},    {4, 4, 2.1f, 8.0e-3f, 1.1f, 1.66e-2f}};

int pick_form(int M, int N, int K, bool direct) {
  int best = 0;
  float least = INFINITY;
  for (int i = 0; i < (direct ? KINDS : KINDS - 1); ++i) {
    const Form& f = direct ? FORMS[i] : BY_REGISTERS[i];
    if (i > 0 && M <= 16) break;
    if (f.mt < 4 && (M + 16 * f.mt - 1) / (16 * f.mt) > 65535) continue;
    const int64_t blocks = (int64_t)((M + 16 * f.mt - 1) / (16 * f.mt)) * ((N + 16 * f.nt - 1) / (16 * f.nt));
    const float rounds = (float)((blocks + 255) / 256) * (f.round + f.round_k * K), lone = f.start_k * K;
    const float cost = f.start + (direct && i >= SIDE_BY_SIDE ? fmaxf(lone, rounds) : lone + rounds);
    if (cost < least) { least = cost; best = i; }
  }
  return best;
}

template <bool VEC, How HOW>
void launch(const float* x, const float* w, float* y, int M, int N, int K, hipStream_t s) {
  const int best = pick_form(M, N, K, HOW == DIRECT);
  const dim3 grid((N + 16 * FORMS[best].nt - 1) / (16 * FORMS[best].nt), (M + 16 * FORMS[best].mt - 1) / (16 * FORMS[best].mt));
  switch (best) {
    case 0:
      if (M <= 16 && (N + 15) / 16 <= HALF_TILES) gemm_f32_half_kernel<2, VEC><<<(N + 7) / 8, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K);
      else gemm_f32_rows_kernel<1, 1, 2, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K);
      break;
    case 1: gemm_f32_rows_kernel<1, 2, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 2: gemm_f32_rows_kernel<2, 2, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 3: gemm_f32_rows_kernel<2, 4, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case SIDE_BY_SIDE: gemm_f32_kernel<4, 2, 2, HOW><<<grid, 1024, 0, s>>>(x, w, y, M, N, K); break;
    case IN_TURN_32:
      if constexpr (HOW == DIRECT) gemm_f32_kernel<1, 1, 2, HOW><<<grid, 256, 0, s>>>(x, w, y, M, N, K);
      break;
    default: gemm_f32_kernel<1, 2, 2, HOW><<<grid, 256, 0, s>>>(x, w, y, M, N, K); break;
  }
}
}  // namespace

// Which form serves M rows of operands on 16 bytes: 0 to 3 tiles of 1 x 1, 1 x 2, 2 x 2 and 2 x 4 a block straight from memory; 4 to 6 staged
// ones, 64 x 64 a block with the quarters of K side by side (4) or one after the other (5), and 32 x 64 one after the other (6, whole
// chunks of K alone); -1 one running sum.
extern "C" int holon_gemm_f32_form(int M, int N, int K) { return sums_in_order(N, K) ? -1 : pick_form(M, N, K, K % CHUNK == 0); }

extern "C" int holon_gemm_f32(const void* x, const void* w, void* y, int M, int N, int K, void* stream) {
  HOLON_CHECK(M >= 0 && N > 0 && K > 0, "gemm (float32): M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  HOLON_CHECK((M + 63) / 64 <= 65535, "gemm (float32): M=%d rows exceed one launch (%d)", M, 65535 * 64);
  const bool vec = K % 4 == 0 && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0);
  if (sums_in_order(N, K)) {
    const dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
    hipStream_t s = (hipStream_t)stream;
    if (vec) gemm_f32_in_order_kernel<true><<<grid, 256, 0, s>>>((const float*)x, (const float*)w, (float*)y, M, N, K);
    else gemm_f32_in_order_kernel<false><<<grid, 256, 0, s>>>((const float*)x, (const float*)w, (float*)y, M, N, K);
  } else if (vec && K % CHUNK == 0) launch<true, DIRECT>((const float*)x, (const float*)w, (float*)y, M, N, K, (hipStream_t)stream);
  else if (vec) launch<true, BY_FOUR>((const float*)x, (const float*)w, (float*)y, M, N, K, (hipStream_t)stream);
  else launch<false, BY_VALUE>((const float*)x, (const float*)w, (float*)y, M, N, K, (hipStream_t)stream);
  HOLON_LAUNCH_OK();
  return 0;
}
