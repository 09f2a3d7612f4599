// The gated delta rule over prompt rows, in blocks of 16 tokens on the float32 matrix cores. Token by token (recurrent.hip, which
// keeps decode rows and short portions, also where a step has longer rows beside them) the rule is S <- g_t S; u_t = beta_t (v_t - S^T k_t); S <- S + k_t u_t^T; o_t = S^T q_t. Over a block that
// starts from S0, with G_t the product of g up to t, f(t, i) the product of g behind i up to t and E_i = f(last, i):
//   u   = T R,  R_t = beta_t v_t - beta_t G_t S0^T k_t,  T = (I + L)^-1,  L[t][i] = beta_t f(t, i) k_t . k_i below the diagonal
//   o_t = G_t S0^T q_t + sum over i <= t of (f(t, i) q_t . k_i) u_i
//   S   = G S0 + sum_i E_i k_i u_i^T
// T and the scores f(t, i) q_t . k_i are 16 x 16 matrices of a block and head that do not depend on S: `delta_blocks` forms them
// for all blocks of the step at once, and only products with S are left in the chain from block to block. Every decay is a product of
// g between two tokens and so at most 1; nothing is divided by one.
//
// Rows of more than a piece's tokens run in pieces side by side: a piece is linear in the state it starts from, S -> A S + B. The first
// pass runs every piece but a row's last on the D columns of the identity with values of zero (A) and on the V value columns from zero
// (B); `delta_walk` goes over a row's pieces in order; the second pass starts every piece from its true state and writes outputs.
//
// What bounds it is the chain: a block costs its wave 3 D / 4 + 8 matrix instructions of 32 cycles (1.4 us at D = 128), one wave a
// SIMD. A wave owns 16 value columns, S's D x 16 part in its accumulators, whose layout is that of the second operand of the products over
// S's rows: nothing is moved between lanes. Four waves a block share K, Q and the transposed decayed K through LDS (more waves a
// block leave fewer blocks than compute units: 16 heads of 128 by 128 over 2,048 tokens are 256 blocks of four). Measured, 16 heads of
// 128 by 128, us (token by token in registers, rows of 512 and more in pieces): one row of 64 / 300 / 1,024 / 2,048 tokens 28 / 70 / 120 / 159
// (41 / 170 / 405 / 709), rows of 1,400, 700, 900 and 1,000 in one step 259 (1,443). Against 64 bits o is off by 8.2e-8 (1.03e-7), the state by
// 5.1e-8 to 7.3e-8 (5.0e-8 to 7.2e-8).
//
// v_mfma_f32_16x16x4_f32: A 16x4 (lane l: row l % 16, k = l / 16), B 4x16 (lane l: column l % 16, k = l / 16), result in lane l: rows
// 4 (l / 16) + i of column l % 16. Product i of a group of 16 inner values takes k = 4 (l / 16) + i.
#include "common.h"
#include "holon_hip.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {
constexpr int TB = 16;                       // tokens a block
constexpr int NW = 4, THREADS = NW * WAVE;
constexpr int ROW_BETA = 512, ROW_BG = 528, ROW_G = 544, ROW_E = 560, BLOCK_FLOATS = 576;      // a block's matrices: T, scores, then factors by token

struct DeltaRows {
  const float* qn;             // [T, G, D]
  const float* kn;
  const float* beta;           // [T, H]
  const float* g;
  const int32_t* slots;
  const int32_t* starts;
  const int32_t* query_start;
  int heads, kv_heads, dim, vdim;
  int piece;                   // tokens a piece, a multiple of 16
  const int32_t* piece_of;     // [rows]: the same row by row, 0: the row goes token by token; null: `piece` for all
  const int32_t* base;         // [rows]: the number of row b's first piece among all pieces of the step
  float* blocks;               // [T / 16 + rows, H, BLOCK_FLOATS]
  float* a;                    // [pieces, H, KD, KD], the key size padded with zeros
  float* sin;                  // [pieces, H, D, V]: B, then the state behind the piece; a row's last piece's place: the state it starts from
};

__device__ __forceinline__ int piece_tokens(const DeltaRows& r, int b) { return r.piece_of ? r.piece_of[b] : r.piece; }
__device__ __forceinline__ int pieces_of(int tokens, int piece) { return piece > 0 ? (tokens + piece - 1) / piece : 0; }
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }
__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Where the matrices of the block that starts at token `first` of row b lie: rows' blocks never share a place, as a row's first token's
// sixteenth is at least that of the row before's last one.
__device__ __forceinline__ int64_t block_place(const DeltaRows& r, int first, int b, int h) {
  return ((int64_t)(first / TB + b) * r.heads + h) * BLOCK_FLOATS;
}

// Four neighbouring key channels of a token's head; channels from dim on are zero.
template <bool WHOLE>
__device__ __forceinline__ f32x4 four(const float* __restrict__ row, int d, int dim) {
  if constexpr (WHOLE) return d < dim ? *reinterpret_cast<const f32x4*>(row + d) : f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 x;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = d + i < dim ? row[d + i] : 0.f;
  return x;
}

// A wave a block of tokens and head. WHOLE: key sizes are multiples of four, so a token's channels come as 16-byte loads.
template <bool WHOLE>
__global__ void __launch_bounds__(THREADS) delta_blocks_kernel(DeltaRows r) {
  __shared__ __attribute__((aligned(16))) double below[NW][TB][TB];
  const int b = blockIdx.x, h = blockIdx.y, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, g4 = lane / 16, c = lane % 16;
  const int lo = r.query_start[b], hi = r.query_start[b + 1], t0 = lo + (blockIdx.z * NW + wave) * TB;
  if (t0 >= hi || piece_tokens(r, b) == 0) return;         // (waves of a block share nothing)
  const int n = min(TB, hi - t0), hk = h / (r.heads / r.kv_heads);
  const bool in = c < n;
  const int64_t row = ((int64_t)(t0 + min(c, n - 1)) * r.kv_heads + hk) * r.dim;
  const float gv = in ? r.g[(int64_t)(t0 + c) * r.heads + h] : 1.f, bv = in ? r.beta[(int64_t)(t0 + c) * r.heads + h] : 0.f;
  double kk[4] = {0., 0., 0., 0.}, qk[4] = {0., 0., 0., 0.};
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  for (int d = 4 * g4; d - 4 * g4 < r.dim; d += 16) {
    const f32x4 ka = four<WHOLE>(r.kn + row, d, r.dim), qa = four<WHOLE>(r.qn + row, d, r.dim);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float ki = in ? ka[i] : 0.f;
      const f32x4 ks = mfma(ki, ki, none), qs = mfma(in ? qa[i] : 0.f, ki, none);
#pragma unroll
      for (int n = 0; n < 4; ++n) { kk[n] += ks[n]; qk[n] += qs[n]; }
    }
  }
  // Rows t = 4 g4 + i of column c. All of this in 64 bits, each value rounded once: what is off here is off for a whole row of outputs
  // or all of the state at once (with q . k and k . k summed in 32 bits o's error over 2,048 tokens is 1.09e-7).
  double f[4] = {0., 0., 0., 0.}, run = 1., upto = 1., behind = 1.;
#pragma unroll
  for (int m = 0; m < TB; ++m) {
    const double gm = __shfl(gv, m, WAVE);
    if (m > c) { run *= gm; behind *= gm; }
    if (m <= c) upto *= gm;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (m == 4 * g4 + i) f[i] = run;
  }
  float* to = r.blocks + block_place(r, t0, b, h);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 4 * g4 + i;
    to[TB * TB + t * TB + c] = c <= t ? (float)(f[i] * qk[i]) : 0.f;
    const float bt = __shfl(bv, t, WAVE);
    below[wave][t][c] = c < t ? bt * (f[i] * kk[i]) : 0.;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (a wave's LDS operations complete in order; its own rows)
  double x[TB];                                            // column c of T, row after row; the four groups of lanes do the same
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    double s = t == c ? 1. : 0.;
#pragma unroll
    for (int i = 0; i < t; ++i) s -= below[wave][t][i] * x[i];
    x[t] = s;
    if (t / 4 == g4) to[t * TB + c] = t == c ? 0.f : (float)s;
  }
  if (g4 == 0) {
    to[ROW_BETA + c] = bv;
    to[ROW_BG + c] = (float)(bv * upto);
    to[ROW_G + c] = (float)upto;
    to[ROW_E + c] = (float)behind;
  }
}

// A block: one (piece, head) and 64 columns. PASS 1: columns 0 .. V - 1 form B, the D behind them A; PASS 2: outputs.
template <int KD, int PASS, bool WHOLE, typename T>
__global__ void __launch_bounds__(THREADS, KD <= 128 ? 2 : 1) delta_chain_kernel(const T* __restrict__ qkv, int qkv_stride, int v_offset,
                                                                                float* __restrict__ state, float* __restrict__ out,
                                                                                DeltaRows r) {
  constexpr bool OUT = PASS == 2;
  constexpr int DT = KD / 16, KP = KD + 4, TP = TB + 4, PER = TB * KD / 4 / THREADS;
  static_assert(TB * KD % (4 * THREADS) == 0 || KD == 32, "whole rounds of 16-byte pieces");
  constexpr int ROUNDS = PER > 0 ? PER : 1;                // (a key size of 32: half of the threads have a piece)
  __shared__ __attribute__((aligned(16))) float ks[TB * KP], qs[OUT ? TB * KP : 4], kt[KD * TP];
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, g4 = lane / 16, c = lane % 16;
  const int dim = r.dim, vdim = r.vdim, hk = h / (r.heads / r.kv_heads);
  const int columns = OUT ? vdim : vdim + dim, col_blocks = (columns + 16 * NW - 1) / (16 * NW);
  const int piece = blockIdx.z / col_blocks, j = (blockIdx.z % col_blocks) * 16 * NW + 16 * wave + c;      // this lane's column
  int lo = r.query_start[b], hi = r.query_start[b + 1];
  const int tokens = piece_tokens(r, b), pieces = pieces_of(hi - lo, tokens);
  if (piece >= pieces || (!OUT && piece == pieces - 1)) return;
  lo += piece * tokens;
  hi = min(hi, lo + tokens);
  const int64_t piece_no = r.base[b] + piece;
  float* held = state + ((int64_t)r.slots[b] * r.heads + h) * dim * vdim;
  const float* before = pieces == 1 ? held : r.sin + ((piece_no + (piece == 0 ? pieces : 0) - 1) * r.heads + h) * dim * vdim;
  const bool some = OUT && (piece > 0 || r.starts[b] > 0);  // whether there is a state to start from
  const bool value = j < vdim;
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * dt + 4 * g4 + i;
      if constexpr (OUT) S[dt][i] = some && value && d < dim ? before[(int64_t)d * vdim + j] : 0.f;
      else S[dt][i] = !value && d == j - vdim ? 1.f : 0.f;
    }
  // The operands of a block of tokens on their way; a thread's pieces of K and Q are all of token tid % 16. Places past a row's end are
  // read from its last token and made harmless when the values are used, so that nothing here waits for a load.
  f32x4 nk[ROUNDS], nq[ROUNDS], nt, np, nb, nbg, ng;
  float ne, nall;
  T nv[4];
  const auto ask = [&](int t0) {
    const int64_t row = ((int64_t)min(t0 + tid % TB, hi - 1) * r.kv_heads + hk) * dim;
#pragma unroll
    for (int e = 0; e < ROUNDS; ++e) {
      const int d = 4 * (tid / TB + e * (THREADS / TB));
      if (KD >= 64 || d < KD) {
        nk[e] = four<WHOLE>(r.kn + row, d, dim);
        if constexpr (OUT) nq[e] = four<WHOLE>(r.qn + row, d, dim);
      }
    }
    const float* m = r.blocks + block_place(r, t0, b, h);
    nt = *reinterpret_cast<const f32x4*>(m + c * TB + 4 * g4);
    if constexpr (OUT) np = *reinterpret_cast<const f32x4*>(m + TB * TB + c * TB + 4 * g4);
    nb = *reinterpret_cast<const f32x4*>(m + ROW_BETA + 4 * g4);
    nbg = *reinterpret_cast<const f32x4*>(m + ROW_BG + 4 * g4);
    if constexpr (OUT) ng = *reinterpret_cast<const f32x4*>(m + ROW_G + 4 * g4);
    ne = m[ROW_E + tid % TB];
    nall = m[ROW_G + TB - 1];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      nv[i] = qkv[(int64_t)min(t0 + 4 * g4 + i, hi - 1) * qkv_stride + v_offset + h * vdim + min(j, vdim - 1)];
  };
  ask(lo);
  for (int t0 = lo; t0 < hi; t0 += TB) {
    const bool in = t0 + tid % TB < hi;
#pragma unroll
    for (int e = 0; e < ROUNDS; ++e) {
      const int d = 4 * (tid / TB + e * (THREADS / TB)), t = tid % TB;
      if (KD >= 64 || d < KD) {
        const f32x4 none = {0.f, 0.f, 0.f, 0.f}, key = in ? nk[e] : none;
        *reinterpret_cast<f32x4*>(&ks[t * KP + d]) = key;
        if constexpr (OUT) *reinterpret_cast<f32x4*>(&qs[t * KP + d]) = in ? nq[e] : none;
#pragma unroll
        for (int i = 0; i < 4; ++i) kt[(d + i) * TP + t] = key[i] * ne;
      }
    }
    const f32x4 ta = nt, pa = np, beta = nb, bg = nbg, gt = ng;
    const float all = nall;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = t0 + 4 * g4 + i < hi && value ? Elem<T>::load(nv[i]) : 0.f;
    lds_barrier();
    if (t0 + TB < hi) ask(t0 + TB);
    // Sums over S's rows in chains of 8 values, four side by side: a chain rounds at the size of what it holds (in chains of 32 o's
    // error over 2,048 tokens is 2.1e-7).
    f32x4 read, from;
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
      f32x4 rc[4], fc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) rc[i] = fc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = d0; dt < d0 + 2; ++dt) {
        const f32x4 ka = *reinterpret_cast<const f32x4*>(&ks[c * KP + 16 * dt + 4 * g4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) rc[i] = mfma(ka[i], S[dt][i], rc[i]);
        if constexpr (OUT) {
          const f32x4 qa = *reinterpret_cast<const f32x4*>(&qs[c * KP + 16 * dt + 4 * g4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) fc[i] = mfma(qa[i], S[dt][i], fc[i]);
        }
      }
      const f32x4 rs = (rc[0] + rc[1]) + (rc[2] + rc[3]), fs = (fc[0] + fc[1]) + (fc[2] + fc[3]);
      read = d0 ? read + rs : rs;
      from = d0 ? from + fs : fs;
    }
    // A row of R or u that is not finite belongs into its own token's and the later ones': the products, where it would meet the
    // earlier ones' zeros, go without it, and it is added below them: T from the row behind its own, as its diagonal is left out of `m` and
    // R itself is added to u (an infinity stays one, for its token's u and for the state), and never in rows behind the portion's end.
    const auto lower = [&](const f32x4& a, const f32x4& x, int matrix) {
      f32x4 clean, sum = {0.f, 0.f, 0.f, 0.f};
      bool all_finite = true;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        clean[i] = finite(x[i]) ? x[i] : 0.f;
        all_finite = all_finite && finite(x[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sum = mfma(a[i], clean[i], sum);
      if (__ballot(!all_finite) != 0) {
        const float* m = r.blocks + block_place(r, t0, b, h) + matrix * TB * TB;
#pragma nounroll
        for (int n = 0; n < TB; ++n) {
          const f32x4 every = x;
          const float mine = n % 4 == 0 ? every[0] : (n % 4 == 1 ? every[1] : (n % 4 == 2 ? every[2] : every[3]));
          const float val = __shfl(mine, (n / 4) * 16 + c, WAVE);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!finite(val) && n < 4 * g4 + i + matrix && t0 + 4 * g4 + i < hi) sum[i] += m[(4 * g4 + i) * TB + n] * val;
        }
      }
      return sum;
    };
    f32x4 R;
#pragma unroll
    for (int i = 0; i < 4; ++i) R[i] = t0 + 4 * g4 + i < hi ? beta[i] * v[i] - bg[i] * read[i] : 0.f;
    const f32x4 u = R + lower(ta, R, 0);
    if constexpr (OUT) {
      const f32x4 o = from * gt + lower(pa, u, 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = t0 + 4 * g4 + i;
        if (t < hi && value) out[((int64_t)t * r.heads + h) * vdim + j] = o[i];
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const f32x4 ka = *reinterpret_cast<const f32x4*>(&kt[(16 * dt + c) * TP + 4 * g4]);
      S[dt] *= all;
#pragma unroll
      for (int i = 0; i < 4; ++i) S[dt] = mfma(ka[i], u[i], S[dt]);
    }
    lds_barrier();                                         // the next block's operands go where these were read
  }
  const bool to_slot = OUT && piece == pieces - 1;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * dt + 4 * g4 + i;
      if constexpr (OUT) {
        if (to_slot && value && d < dim) held[(int64_t)d * vdim + j] = S[dt][i];
      } else if (value) {
        if (d < dim) r.sin[((piece_no * r.heads + h) * dim + d) * vdim + j] = S[dt][i];
      } else if (j < columns) {
        r.a[((piece_no * r.heads + h) * KD + d) * KD + j - vdim] = S[dt][i];
      }
    }
}

// Between the passes: a row's pieces in order, S <- A S + B, 16 columns of S a block, a tile of 16 of S's rows a wave in turn; S goes round
// through LDS, columns as rows. (A's columns from dim on are not written: they meet S's rows there, which are zero, as zeros.) sin[p]
// becomes the state piece p + 1 starts from, and the last piece's place, which nothing is added to, takes the state the row starts from: the
// slot may no longer hold it when piece 0 comes to read it, as the last piece writes it in the same launch.
template <int KD>
__global__ void __launch_bounds__(THREADS) delta_walk_kernel(const float* __restrict__ state, DeltaRows r) {
  constexpr int DT = KD / 16, TILES = (DT + NW - 1) / NW, SP = KD + 4;
  __shared__ __attribute__((aligned(16))) float st[2][16 * SP];
  const int b = blockIdx.x, h = blockIdx.y, j0 = blockIdx.z * 16, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, g4 = lane / 16, c = lane % 16;
  const int dim = r.dim, vdim = r.vdim, j = j0 + c;
  const int pieces = pieces_of(r.query_start[b + 1] - r.query_start[b], piece_tokens(r, b));
  if (pieces < 2) return;
  const float* held = state + ((int64_t)r.slots[b] * r.heads + h) * dim * vdim;
  const bool carried = r.starts[b] > 0;
  for (int e = threadIdx.x; e < KD * 16; e += THREADS) {
    const int d = e / 16, jj = e % 16;
    const float s = carried && d < dim && j0 + jj < vdim ? held[(int64_t)d * vdim + j0 + jj] : 0.f;
    st[0][jj * SP + d] = s;
    if (d < dim && j0 + jj < vdim) r.sin[((((int64_t)r.base[b] + pieces - 1) * r.heads + h) * dim + d) * vdim + j0 + jj] = s;
  }
  f32x4 na[TILES][DT], nb[TILES];
  const auto ask = [&](int p) {
    const int64_t at = ((int64_t)r.base[b] + p) * r.heads + h;
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      const int rt = wave + u * NW;
      if (rt >= DT) continue;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) na[u][dt] = *reinterpret_cast<const f32x4*>(r.a + (at * KD + 16 * rt + c) * KD + 16 * dt + 4 * g4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * rt + 4 * g4 + i;
        nb[u][i] = d < dim && j < vdim ? r.sin[(at * dim + d) * vdim + j] : 0.f;
      }
    }
  };
  ask(0);
  __syncthreads();
  for (int p = 0; p + 1 < pieces; ++p) {
    const int64_t at = ((int64_t)r.base[b] + p) * r.heads + h;
    const float* from = st[p % 2];
    float* to = st[(p + 1) % 2];
    f32x4 acc[TILES][2];
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      acc[u][0] = nb[u];
      acc[u][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(&from[c * SP + 16 * dt + 4 * g4]);
#pragma unroll
      for (int u = 0; u < TILES; ++u) {
        if (wave + u * NW >= DT) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][i % 2] = mfma(16 * dt + 4 * g4 + i < dim ? na[u][dt][i] : 0.f, s[i], acc[u][i % 2]);
      }
    }
    if (p + 2 < pieces) ask(p + 1);
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      const int rt = wave + u * NW;
      if (rt >= DT) continue;
      const f32x4 s = acc[u][0] + acc[u][1];
      *reinterpret_cast<f32x4*>(&to[c * SP + 16 * rt + 4 * g4]) = s;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * rt + 4 * g4 + i;
        if (d < dim && j < vdim) r.sin[(at * dim + d) * vdim + j] = s[i];
      }
    }
    lds_barrier();                                         // S is whole; the other buffer is read by nobody any more
  }
}

template <int KD, bool WHOLE, typename T>
void chain(int pass, dim3 grid, hipStream_t s, const void* qkv, int stride, int v_offset, float* state, float* out, const DeltaRows& r) {
  if (pass == 1) delta_chain_kernel<KD, 1, WHOLE, T><<<grid, THREADS, 0, s>>>((const T*)qkv, stride, v_offset, state, out, r);
  else delta_chain_kernel<KD, 2, WHOLE, T><<<grid, THREADS, 0, s>>>((const T*)qkv, stride, v_offset, state, out, r);
}
}  // namespace

// The rows of holon_delta_scan that `piece_of` gives pieces (null: every row; it has checked the arguments).
int holon_delta_scan_pieces(const float* qn, const float* kn, const void* qkv, int qkv_stride, int v_offset, const float* beta,
                            const float* g, float* state, float* out, const int32_t* slots, const int32_t* starts,
                            const int32_t* query_start, int rows, int heads, int kv_heads, int dim, int vdim, int dtype,
                            int piece_tokens, int max_pieces, const int32_t* piece_base, const int32_t* piece_of, float* blocks,
                            float* a, float* sin, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  const DeltaRows r{qn, kn, beta, g, slots, starts, query_start, heads, kv_heads, dim, vdim, piece_tokens, piece_of, piece_base, blocks, a, sin};
  const bool whole = dim % 4 == 0 && (((uintptr_t)qn | (uintptr_t)kn) & 15) == 0;
  const int64_t groups = ((int64_t)max_pieces * piece_tokens / TB + NW - 1) / NW;
  const int out_cols = (vdim + 16 * NW - 1) / (16 * NW), all_cols = (vdim + dim + 16 * NW - 1) / (16 * NW);
  HOLON_CHECK(groups <= 65535 && (int64_t)all_cols * max_pieces <= 65535, "delta_scan: %d pieces a row exceed one launch", max_pieces);
  if (whole) delta_blocks_kernel<true><<<dim3(rows, heads, (unsigned)groups), THREADS, 0, s>>>(r);
  else delta_blocks_kernel<false><<<dim3(rows, heads, (unsigned)groups), THREADS, 0, s>>>(r);
  HOLON_LAUNCH_OK();
#define CHAIN_T(PASS, KD, GRID)                                                                                              \
  do {                                                                                                                       \
    if (dtype == HOLON_F32) {                                                                                                \
      if (whole) chain<KD, true, float>(PASS, GRID, s, qkv, qkv_stride, v_offset, state, out, r);                            \
      else chain<KD, false, float>(PASS, GRID, s, qkv, qkv_stride, v_offset, state, out, r);                                 \
    } else {                                                                                                                 \
      if (whole) chain<KD, true, bf16_t>(PASS, GRID, s, qkv, qkv_stride, v_offset, state, out, r);                           \
      else chain<KD, false, bf16_t>(PASS, GRID, s, qkv, qkv_stride, v_offset, state, out, r);                                \
    }                                                                                                                        \
  } while (0)
#define CHAIN(PASS, GRID)                                                                                                    \
  do {                                                                                                                       \
    if (dim <= 32) CHAIN_T(PASS, 32, GRID);                                                                                  \
    else if (dim <= 64) CHAIN_T(PASS, 64, GRID);                                                                             \
    else if (dim <= 128) CHAIN_T(PASS, 128, GRID);                                                                           \
    else CHAIN_T(PASS, 256, GRID);                                                                                           \
  } while (0)
  if (max_pieces > 1) {
    CHAIN(1, dim3(rows, heads, all_cols * max_pieces));
    HOLON_LAUNCH_OK();
    const dim3 walk(rows, heads, (vdim + 15) / 16);
    if (dim <= 32) delta_walk_kernel<32><<<walk, THREADS, 0, s>>>(state, r);
    else if (dim <= 64) delta_walk_kernel<64><<<walk, THREADS, 0, s>>>(state, r);
    else if (dim <= 128) delta_walk_kernel<128><<<walk, THREADS, 0, s>>>(state, r);
    else delta_walk_kernel<256><<<walk, THREADS, 0, s>>>(state, r);
    HOLON_LAUNCH_OK();
  }
  CHAIN(2, dim3(rows, heads, out_cols * max_pieces));
#undef CHAIN
#undef CHAIN_T
  HOLON_LAUNCH_OK();
  return 0;
}
