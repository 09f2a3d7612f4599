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
#include "common.h"
#include "holon_hip.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace {
constexpr int SHARES = 16, QUARTERS = 4;
constexpr int GROUP = 16;              // k values of one 16-byte load of every lane
constexpr int CHUNK = 32;              // k values staged at a time, and what shares are a multiple of

constexpr int SHORTEST = 64;           // a share's least length: up to 1,024 of K fewer waves share it

__host__ __device__ __forceinline__ int share_length(int K) {
  const int even = (K + SHARES * CHUNK - 1) / (SHARES * CHUNK) * CHUNK;
  return even > SHORTEST ? even : SHORTEST;
}

// s[0] .. s[15] in the order above.
template <typename F>
__device__ __forceinline__ f32x4_t sum_shares(F s) {
  f32x4_t total;
#pragma unroll
  for (int q = 0; q < QUARTERS; ++q) {
    f32x4_t quarter = s(4 * q);
#pragma unroll
    for (int i = 1; i < 4; ++i) quarter += s(4 * q + i);
    total = q ? total + quarter : quarter;
  }
  return total;
}

// Four results of a row, columns n .. n + 3.
__device__ __forceinline__ void store4(float* __restrict__ y, f32x4_t v, int m, int n, int M, int N) {
  if (m >= M) return;
  float* out = y + (int64_t)m * N + n;
  if (N % 4 == 0 && (uintptr_t)y % 16 == 0) {
    if (n < N) *reinterpret_cast<f32x4_t*>(out) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) if (n + i < N) out[i] = v[i];
  }
}

// Four floats of a row at k. VEC: K is a multiple of 4 and rows are 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ f32x4_t load4(const float* __restrict__ row, int k, int K) {
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    if (k < K) v = *reinterpret_cast<const f32x4_t*>(row + k);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) if (k + i < K) v[i] = row[k + i];
  }
  return v;
}

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
  for (int k0 = first; k0 < last; k0 += DEPTH * GROUP) {
    f32x4_t a[DEPTH][NT], b[DEPTH][MT];
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {                     // (beyond the share: zeros, which add nothing)
      const int k = k0 + s * GROUP + 4 * g;
#pragma unroll
      for (int u = 0; u < NT; ++u) a[s][u] = load4<VEC>(wr[u], k, last);
#pragma unroll
      for (int t = 0; t < MT; ++t) b[s][t] = load4<VEC>(xr[t], k, last);
    }
#pragma unroll
    for (int s = 0; s < DEPTH; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int u = 0; u < NT; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][u][i], b[s][t][i], acc[t][u], 0, 0, 0);
  }
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

// More rows: bound by the matrix cores. A block owns 64 x 64 results; four waves (32 x 32 each) walk a run of K whose rows of x and
// w they stage in LDS, CHUNK of k at a time, into one of two buffers while the other is multiplied; pieces of 16 bytes lie at
// place p ^ (row % 8) of their row. SIDE 4: sixteen waves, the four quarters of K side by side: what fills the chip where an output of
// some hundred rows has few tiles, four waves a SIMD covering each other's barriers. SIDE 1: four waves, the quarters one after the
// other: several blocks share a unit, so that one's first loads and its stores lie under the others' products; that is the better
// one where there are tiles for it, the more the shorter K. Either ends at K (what lies behind it would add zeros).
template <int SIDE, bool VEC>
__global__ void __launch_bounds__(SIDE * 256) gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              float* __restrict__ y, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) float stage[SIDE][2][2][64 * CHUNK];       // quarter, buffer, x or w
  const int quarter = SIDE > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / 256) : 0, tid = threadIdx.x % 256;
  const int wave = tid / WAVE, lane = tid % WAVE;
  const int g = lane / 16, c = lane % 16;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int share = share_length(K), first = quarter * 4 * share, per_share = share / CHUNK;
  const int chunks = (min(K, (SIDE > 1 ? 4 : 16) * share) + CHUNK - 1) / CHUNK;      // (of the block: the first quarter's)
  // what this thread stages: rows tid / 8 and 32 more, piece tid % 8
  const int r0 = tid / 8, p0 = tid % 8;
  const float *xr[2], *wr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xr[i] = x + (int64_t)min(m0 + r0 + 32 * i, M - 1) * K;
    wr[i] = w + (int64_t)min(n0 + r0 + 32 * i, N - 1) * K;
  }
  const int put = r0 * CHUNK + 4 * (p0 ^ (r0 % 8));
  f32x4_t held[2][2];
  auto fetch = [&](int chunk) {
    const int k = first + chunk * CHUNK + 4 * p0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      held[0][i] = load4<VEC>(xr[i], k, K);
      held[1][i] = load4<VEC>(wr[i], k, K);
    }
  };
  auto keep = [&](int buf) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4_t*>(&stage[quarter][buf][o][put + 32 * i * CHUNK]) = held[o][i];
  };
  // where this lane reads: row 32 (half) + 16 t + c, pieces g and 4 + g
  const int xrow = wave / 2 * 32 + c, wrow = wave % 2 * 32 + c;
  const int at[2] = {4 * (g ^ (c % 8)), 4 * ((4 + g) ^ (c % 8))};
  // the sums of a share, of a quarter's shares so far (SIDE 1), and of all that is behind them
  f32x4_t acc[2][2], part[SIDE > 1 ? 1 : 2][2], total[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) acc[t][u] = total[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int left = per_share, shares = 0;
  const auto end_share = [&]() {
    const bool begins = SIDE > 1 ? shares == 0 : shares % 4 == 0, ends = shares % 4 == 3, first_quarter = shares < 4;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if constexpr (SIDE > 1) {
          total[t][u] = begins ? acc[t][u] : total[t][u] + acc[t][u];
        } else {
          part[t][u] = begins ? acc[t][u] : part[t][u] + acc[t][u];
          if (ends) total[t][u] = first_quarter ? part[t][u] : total[t][u] + part[t][u];
        }
        acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    left = per_share;
    ++shares;
  };
  fetch(0);
  keep(0);
  if (chunks > 1) fetch(1);
  lds_barrier();
  for (int ch = 0; ch < chunks; ++ch) {
    if (ch + 1 < chunks) keep((ch + 1) & 1);              // (read last in front of the barrier behind us)
    if (ch + 2 < chunks) fetch(ch + 2);
    if (SIDE == 1 || first + ch * CHUNK < K) {
      const float* xs = stage[quarter][ch & 1][0];
      const float* ws = stage[quarter][ch & 1][1];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        f32x4_t b[2], a[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) b[t] = *reinterpret_cast<const f32x4_t*>(&xs[(xrow + 16 * t) * CHUNK + at[s]]);
#pragma unroll
        for (int u = 0; u < 2; ++u) a[u] = *reinterpret_cast<const f32x4_t*>(&ws[(wrow + 16 * u) * CHUNK + at[s]]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[t][i], acc[t][u], 0, 0, 0);
      }
      if (--left == 0) end_share();
    }
    lds_barrier();                                        // (what was fetched stays under way)
  }
  if (left < per_share) end_share();                      // (K ends inside a share)
  if constexpr (SIDE > 1) {
    // the quarters' sums through LDS: tile (4 t' + u') of the block's 16, one a wave
    f32x4_t(*sums)[16][WAVE] = reinterpret_cast<f32x4_t(*)[16][WAVE]>(&stage[0][0][0][0]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) sums[quarter][(wave / 2 * 2 + t) * 4 + wave % 2 * 2 + u][lane] = total[t][u];
    __syncthreads();
    const int tile = quarter * 4 + wave;
    f32x4_t sum = sums[0][tile][lane];
#pragma unroll
    for (int q = 1; q < QUARTERS; ++q) sum += sums[q][tile][lane];
    store4(y, sum, m0 + tile / 4 * 16 + c, n0 + tile % 4 * 16 + 4 * g, M, N);
  } else {
    const bool pending = shares % 4 != 0, only = shares < 4;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const f32x4_t sum = pending ? (only ? part[t][u] : total[t][u] + part[t][u]) : total[t][u];
        store4(y, sum, m0 + (wave / 2 * 2 + t) * 16 + c, n0 + (wave % 2 * 2 + u) * 16 + 4 * g, M, N);
      }
  }
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

// Which form a product takes: the one that is done first by a fit over K = 48 to 18,432, N = 64 to 16,384 and M = 17 to 2,048 on
// MI355X (1,149 products, each in all forms, weights from memory): in us, a start and so much for every round of one block a CU, both
// linear in K. Where the best form takes more than 15 us the choice is 0.1 % from it on average and 6 % at most. In us, best and others:
// 2048 x 2048 takes 1 x 1 tiles up to 32 rows (10; with a 64 x 64 tile a block and no split of K it took 118), quarters side by side
// from 300 rows (42; one after the other 54, 2 x 2 tiles 50), one after the other at 2,048 (157; 163); 2048 x 9248 and 2048 x 18432 at
// 704 rows quarters side by side (345 and 672; 2 x 4 tiles, which a fit up to K = 4,096 took there, 396 and 767); 16384 x 2048 1 x 1
// tiles up to 16 rows (5.0 TB/s at one row), quarters side by side from 64 (46; 58), one after the other from 150 (125; 130); 9248 x 256
// at 2,048 rows one after the other (103; side by side 180).
struct Form { int mt, nt; float start, start_k, round, round_k; };
constexpr Form FORMS[6] = {{1, 1, 2.6f, 2e-4f, 0.43f, 3.25e-3f}, {1, 2, 2.5f, 2e-4f, 0.63f, 5.0e-3f},
                           {2, 2, 2.5f, 7e-4f, 0.90f, 7.35e-3f}, {2, 4, 1.2f, 5e-4f, 3.0f, 1.31e-2f},
                           {4, 4, 1.2f, 0.f, 3.2f, 1.86e-2f},    {4, 4, 2.1f, 8.0e-3f, 1.1f, 1.66e-2f}};

int pick_form(int M, int N, int K) {
  int best = 0;
  float least = INFINITY;
  for (int i = 0; i < 6; ++i) {
    const Form& f = FORMS[i];
    if (i > 0 && M <= 16) break;
    if (f.mt < 4 && (M + 16 * f.mt - 1) / (16 * f.mt) > 65535) continue;
    const int64_t blocks = (int64_t)((M + 16 * f.mt - 1) / (16 * f.mt)) * ((N + 16 * f.nt - 1) / (16 * f.nt));
    const float cost = f.start + f.start_k * K + (float)((blocks + 255) / 256) * (f.round + f.round_k * K);
    if (cost < least) { least = cost; best = i; }
  }
  return best;
}

template <bool VEC>
void launch(const float* x, const float* w, float* y, int M, int N, int K, hipStream_t s) {
  const int best = pick_form(M, N, K);
  const dim3 grid((N + 16 * FORMS[best].nt - 1) / (16 * FORMS[best].nt), (M + 16 * FORMS[best].mt - 1) / (16 * FORMS[best].mt));
  switch (best) {
    case 0: gemm_f32_rows_kernel<1, 1, 2, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 1: gemm_f32_rows_kernel<1, 2, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 2: gemm_f32_rows_kernel<2, 2, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 3: gemm_f32_rows_kernel<2, 4, 1, VEC><<<grid, SHARES * WAVE, 0, s>>>(x, w, y, M, N, K); break;
    case 4: gemm_f32_kernel<4, VEC><<<grid, 1024, 0, s>>>(x, w, y, M, N, K); break;
    default: gemm_f32_kernel<1, VEC><<<grid, 256, 0, s>>>(x, w, y, M, N, K); break;
  }
}
}  // namespace

// Which form serves M rows: 0 to 3 tiles of 1 x 1, 1 x 2, 2 x 2 and 2 x 4 a block, 4 quarters of K side by side, 5 one after the
// other; -1 one running sum.
extern "C" int holon_gemm_f32_form(int M, int N, int K) { return sums_in_order(N, K) ? -1 : pick_form(M, N, K); }

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
  } else if (vec) launch<true>((const float*)x, (const float*)w, (float*)y, M, N, K, (hipStream_t)stream);
  else launch<false>((const float*)x, (const float*)w, (float*)y, M, N, K, (hipStream_t)stream);
  HOLON_LAUNCH_OK();
  return 0;
}
