// The matrix memory of xLSTM (mLSTM) along each row's tokens. Per (row, head): a matrix S [D, V], a vector n [D] and a
// running maximum m, float32, carried in the request's slot (a row that starts at position 0 starts from S = 0, n = 0
// and a maximum of 0, whatever the slot holds). With log gates i and f of the token:
//   m' = max(f + m, i);  S' = exp(f + m - m') S + exp(i - m') k v^T;  n' = exp(f + m - m') n + exp(i - m') k
//   o = S'^T q / (max(|n' . q|, exp(-m')) + 1e-6)
// The gates come as pre-activations a of a projection and a bias: i = cap tanh((a_i + b_i) / cap),
// f = logsigmoid(cap tanh((a_f + b_f) / cap)); q is scaled by D^-0.5. q, k, v and the gates are columns of one
// projection's rows.
//
// n is kept as one more column of S (the column of a value that is always 1), so the state is S [D, V + 1] and the
// kernel leaves the numerators S'^T q [V] and the denominator max(|n' . q|, exp(-m')) + 1e-6 of every token; the
// read-out kernel that follows divides. S's columns never meet, so a wave owns 8 of them, eight lanes a column with an
// eighth of the key rows each; what a token needs of a whole column is summed over a lane's rows in four interleaved
// chains and then over the eight lanes in a fixed order. A batch of tokens' operands travels from memory to LDS while
// the batch before is worked through; the gates' functions are taken then, off the recurrence's path.
// The blocks of a head (one for every 8 columns) all need m and do not wait for each other, so each keeps a copy of
// its own in the slot, m [H, ceil((V + 1) / 8)]: a block reads and writes nothing that another block touches.
//
// Long rows run in pieces side by side. The maxima depend on the gates alone, m' = max(m + f, i), a recurrence whose
// steps compose ((a, b) then (c, d) is (a + c, max(b + c, d))), so a wave finds a whole row's maxima by a prefix scan and
// leaves every token's two factors exp(f + m - m') and exp(i - m') and exp(-m') behind. With those the recurrence is
// linear in S and n with factors that do not depend on them: every piece but a row's last first runs from zero and
// leaves what it adds and the product of its factors; a small kernel walks a row's pieces in order, leaving each
// piece's true start; then every piece runs again from there and writes its outputs. Both runs are on the matrix cores,
// in chunks of tokens (`mlstm_chunk_kernel`).
#include "common.h"
#include "holon_hip.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

namespace {

template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float part_sum(float v) {      // over the eight adjacent lanes of a column, a fixed order
  v += dpp_move<0xB1>(v);        // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);        // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);       // row_half_mirror
  return v;
}

constexpr int PARTS = 8;                 // lanes a value column is spread over
constexpr int COLS = WAVE / PARTS;       // value columns a wave owns

__device__ __forceinline__ float log_sigmoid(float x) {   // -softplus(-x), without overflow on either side
  return fminf(x, 0.f) - log1pf(expf(-fabsf(x)));
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

struct MlstmPieces {
  int tokens;                  // tokens a piece
  const int32_t* base;         // [rows]: the number of row b's first piece among all pieces of the step
  const float* gates;          // [T, H, 3]: exp(f + m - m'), exp(i - m'), exp(-m') of every token
  float* sloc;                 // [pieces, H, D, V + 1]
  float* pk;                   // [pieces, H]
};

// One wave per (row, head): the row's maxima by a prefix scan over lanes that each hold a run of neighbouring tokens,
// then every token's three factors. The slot's copies of m take the row's last maximum.
template <typename T>
__global__ void __launch_bounds__(WAVE) mlstm_gates_kernel(const T* __restrict__ proj, int width, int gate_off,
                                                           const float* __restrict__ gate_bias, float cap,
                                                           float* __restrict__ m_all, float* __restrict__ gates,
                                                           const int32_t* __restrict__ slots,
                                                           const int32_t* __restrict__ starts,
                                                           const int32_t* __restrict__ query_start, int heads,
                                                           int copies) {
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int lo = query_start[b], hi = query_start[b + 1], n = hi - lo;
  if (n <= 0) return;
  const int64_t cell = ((int64_t)slots[b] * heads + h) * copies;
  const float m0 = starts[b] > 0 ? m_all[cell] : 0.f;
  const float bi = gate_bias[h], bf = gate_bias[heads + h];
  const int seg = (n + WAVE - 1) / WAVE;
  const int t0 = lo + lane * seg, t1 = min(hi, t0 + seg);
  auto gate = [&](int t, float& it, float& ft) {
    const T* row = proj + (int64_t)t * width + gate_off;
    it = cap * tanhf((Elem<T>::load(row[h]) + bi) / cap);
    ft = log_sigmoid(cap * tanhf((Elem<T>::load(row[heads + h]) + bf) / cap));
  };
  float A = 0.f, B = -INFINITY;                       // this lane's run as one step: m -> max(m + A, B)
  for (int t = t0; t < t1; ++t) {
    float it, ft;
    gate(t, it, ft);
    B = fmaxf(B + ft, it);
    A += ft;
  }
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {           // inclusive scan: the runs of lanes 0 .. lane as one step
    const float Ao = __shfl_up(A, off, WAVE), Bo = __shfl_up(B, off, WAVE);
    if (lane >= off) {
      B = fmaxf(Bo + A, B);
      A = Ao + A;
    }
  }
  const float Ae = __shfl_up(A, 1, WAVE), Be = __shfl_up(B, 1, WAVE);
  float m = lane == 0 ? m0 : fmaxf(m0 + Ae, Be);
  for (int t = t0; t < t1; ++t) {
    float it, ft;
    gate(t, it, ft);
    const float m_new = fmaxf(ft + m, it);
    float* g = gates + ((int64_t)t * heads + h) * 3;
    g[0] = expf(ft + m - m_new);
    g[1] = expf(it - m_new);
    g[2] = expf(-m_new);
    m = m_new;
  }
  if (t0 < hi && t1 == hi)
    for (int c = 0; c < copies; ++c) m_all[cell + c] = m;
}

// A row's pieces in order: S <- pk S + sloc; sloc[p] becomes the state piece p + 1 starts from. The last piece adds nothing
// here: its place takes the state the row starts from, which the slot may no longer hold when piece 0 comes to read it.
__global__ void __launch_bounds__(256) mlstm_pieces_kernel(const float* __restrict__ S_all,
                                                           const int32_t* __restrict__ slots,
                                                           const int32_t* __restrict__ starts,
                                                           const int32_t* __restrict__ query_start, int heads, int cells,
                                                           MlstmPieces pc) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int n = query_start[b + 1] - query_start[b];
  const int pieces = (n + pc.tokens - 1) / pc.tokens;
  if (pieces < 2) return;
  const int64_t cell = (int64_t)slots[b] * heads + h;
  const bool carried = starts[b] > 0;
  const int64_t first = pc.base[b];
  for (int e = blockIdx.z * 256 + threadIdx.x; e < cells; e += gridDim.z * 256) {
    float x = carried ? S_all[cell * cells + e] : 0.f;
    pc.sloc[((first + pieces - 1) * heads + h) * cells + e] = x;
    for (int p = 0; p < pieces - 1; ++p) {
      const int64_t at = (first + p) * heads + h;
      float* add = pc.sloc + at * cells + e;
      x = pc.pk[at] * x + *add;
      *add = x;
    }
  }
}

template <int KD, typename T>
__global__ void __launch_bounds__(WAVE) mlstm_scan_kernel(const T* __restrict__ proj, int width, int q_off, int k_off,
                                                          int v_off, int gate_off, const float* __restrict__ gate_bias,
                                                          float cap, float* __restrict__ S_all, float* __restrict__ m_all,
                                                          float* __restrict__ out, float* __restrict__ den_out,
                                                          const int32_t* __restrict__ slots,
                                                          const int32_t* __restrict__ starts,
                                                          const int32_t* __restrict__ query_start, int heads, int dim,
                                                          int vdim, int col_blocks) {
  constexpr int KQ = KD / PARTS, TC = KD <= 64 ? 16 : KD <= 128 ? 8 : 4, N = TC * KD, PER = (N + WAVE - 1) / WAVE;
  __shared__ float qs[2][N], ks[2][N];
  __shared__ float vs[2][TC * COLS], gi[2][TC], gf[2][TC];
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int col_block = blockIdx.z;
  const int part = lane % PARTS, col = lane / PARTS, j = col_block * COLS + col;
  const int cols = vdim + 1;                           // S's columns: the values', then n's
  const bool active = j < cols, of_n = j == vdim;
  const int lo = query_start[b], hi = query_start[b + 1];
  const int64_t cell = (int64_t)slots[b] * heads + h;
  const int64_t mine = cell * col_blocks + col_block;        // this block's own copy of m
  float* S_held = S_all + cell * dim * cols;
  const bool carried = starts[b] > 0;
  float S[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    S[i] = (carried && active && row < dim) ? S_held[(int64_t)row * cols + j] : 0.f;
  }
  float m = carried ? m_all[mine] : 0.f;
  const float q_scale = 1.0f / sqrtf((float)dim);
  const float bi = gate_bias[h], bf = gate_bias[heads + h];
  float nq[PER], nk[PER], ngi = 0.f, ngf = 0.f;
  auto ask = [&](int t0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE, tt = idx / KD, i = idx - tt * KD;
      const bool ok = idx < N && t0 + tt < hi && i < dim;
      const T* row = proj + (int64_t)(t0 + tt) * width;
      nq[e] = ok ? Elem<T>::load(row[q_off + h * dim + i]) * q_scale : 0.f;
      nk[e] = ok ? Elem<T>::load(row[k_off + h * dim + i]) : 0.f;
    }
    static_assert(TC * COLS <= 2 * WAVE, "a lane stages at most two values of v");
    if (lane < TC && t0 + lane < hi) {
      const T* row = proj + (int64_t)(t0 + lane) * width;
      const float ai = Elem<T>::load(row[gate_off + h]) + bi, af = Elem<T>::load(row[gate_off + heads + h]) + bf;
      ngi = cap * tanhf(ai / cap);
      ngf = log_sigmoid(cap * tanhf(af / cap));
    }
  };
  float nv2[2];
  auto ask_v = [&](int t0) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int idx = lane + e * WAVE, tt = idx / COLS, jj = col_block * COLS + idx % COLS;
      const bool ok = idx < TC * COLS && t0 + tt < hi && jj < vdim;
      nv2[e] = ok ? Elem<T>::load(proj[(int64_t)(t0 + tt) * width + v_off + h * vdim + jj]) : (jj == vdim ? 1.f : 0.f);
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < N) { qs[buf][idx] = nq[e]; ks[buf][idx] = nk[e]; }
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < TC * COLS) vs[buf][idx] = nv2[e];
    }
    if (lane < TC) { gi[buf][lane] = ngi; gf[buf][lane] = ngf; }
  };
  if (lo < hi) {
    ask(lo);
    ask_v(lo);
    put(0);
  }
  __syncthreads();
  for (int t0 = lo, buf = 0; t0 < hi; t0 += TC, buf ^= 1) {
    if (t0 + TC < hi) {
      ask(t0 + TC);
      ask_v(t0 + TC);
    }
    const int nt = min(TC, hi - t0);
    for (int tt = 0; tt < nt; ++tt) {
      const float it = gi[buf][tt], ft = gf[buf][tt];
      const float m_new = fmaxf(ft + m, it);
      const float keep = expf(ft + m - m_new), take = expf(it - m_new);
      m = m_new;
      const float vt = vs[buf][tt * COLS + col] * take;
      const float* qt = &qs[buf][tt * KD + part * KQ];
      const float* kt = &ks[buf][tt * KD + part * KQ];
      float os[4] = {0.f, 0.f, 0.f, 0.f};              // four short chains of sums, not one long one
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        S[i] = keep * S[i] + kt[i] * vt;
        os[i % 4] += S[i] * qt[i];
      }
      const float o = part_sum((os[0] + os[1]) + (os[2] + os[3]));
      if (active && part == 0) {
        if (of_n) den_out[(int64_t)(t0 + tt) * heads + h] = fmaxf(fabsf(o), expf(-m)) + 1e-6f;
        else out[((int64_t)(t0 + tt) * heads + h) * vdim + j] = o;
      }
    }
    if (t0 + TC < hi) put(buf ^ 1);
    __syncthreads();
  }
  if (lo >= hi) return;
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    if (row >= dim) continue;
    if (active) S_held[(int64_t)row * cols + j] = S[i];
  }
  if (lane == 0) m_all[mine] = m;
}

// Rows in pieces, on the float32 matrix cores (v_mfma_f32_16x16x4_f32): a block of eight waves takes one (row's piece, head)
// and 128 value columns, wave w columns 16 w .. 16 w + 15 with S's KD x 16 part in its accumulators. Tokens go in chunks of
// C. With the factors k_t (keep) and i_t (take) of a chunk's tokens,
//   p_t = k_1 .. k_t,  M_tj = i_j k_(j+1) .. k_t (j <= t),  e_j = M_(last)j:
//   o_t = p_t S^T q_t + sum_j M_tj (q_t . k_j) v_j;  S <- p_(last) S + sum_j k_j (e_j v_j)^T
// and the same for n with 1 in place of v_j. Every factor is a product of factors of at most 1: nothing is divided, no
// difference of logarithms is taken. The chunk's scores q k^T and the M are formed once by the block's waves together, the
// scores in float64: a score's rounding is shared by all of the token's columns, and made results lie 1.2 times as far from 64 bits as
// the token-by-token scan's (16 heads of 128 by 128 over 2,048 tokens: 1.56e-7 against 1.31e-7; so 1.14e-7, for 5 % of the time).
// Bound by the float32 matrix cores (two products with S a token), by the barriers around a chunk, and in the second pass by its
// registers: keys of 128 need all 256 and spill 42 of them (172 bytes a lane; 13 with bfloat16 keys and queries in pieces of 16 bytes,
// PIECES, four prompts of 700 to 1,500 tokens of 16 heads 103 us and 95), keys of 256 138, with the LDS for two waves a SIMD (one
// block a unit) to hide that; the first pass spills at keys of 256 alone (36; pieces would make it 83, so they go value by value). Two layers of 16 heads of 128 by 128 over steps of 4,096
// and 304 tokens: 150 us for the first passes and 400 for the second ones (368 without the scores in float64 and the branch for
// values that are not finite); token by token, a wave 8 columns with S in registers, 3,400 in all.
// Operands: lane (g4, c) of A holds row c, of B column c, and product i of a group of 16 takes inner index 4 g4 + i, so that
// a result's registers are the B operands of the products over its rows.
template <int KD, int PASS, bool PIECES, typename T>
__global__ void __launch_bounds__(512) mlstm_chunk_kernel(const T* __restrict__ proj, int width, int q_off, int k_off,
                                                          int v_off, float* __restrict__ S_all, float* __restrict__ out,
                                                          float* __restrict__ den_out, const int32_t* __restrict__ slots,
                                                          const int32_t* __restrict__ starts,
                                                          const int32_t* __restrict__ query_start, int heads, int dim,
                                                          int vdim, int col_blocks, MlstmPieces pc) {
  constexpr bool OUT = PASS == 2;
  constexpr int C = KD <= 128 ? 64 : 32, CT = C / 16, DT = KD / 16, QS = KD + 4, MS = C + 4, THREADS = 512;
  constexpr int VEC = PIECES ? 16 / (int)sizeof(T) : 1;      // values of a load
  constexpr int PER = C * KD / THREADS / VEC, TPT = THREADS / C;            // staged pieces a thread; threads a token
  static_assert(!PIECES || PER >= 1, "a piece a thread");
  struct alignas(VEC * sizeof(T)) Piece { T v[VEC]; };
  __shared__ __attribute__((aligned(16))) float qs[OUT ? C * QS : 4], ks[C * QS];
  __shared__ __attribute__((aligned(16))) float score[OUT ? C * MS : 4], fade[OUT ? C * MS : 4];
  __shared__ __attribute__((aligned(16))) float p_s[C], e_s[C];      // (read 16 bytes at a time, as those above)
  __shared__ float n_s[KD], keep_s[C], take_s[C], low_s[C];
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int g4 = lane / 16, c = lane % 16;
  const int piece = blockIdx.z / col_blocks, col0 = (blockIdx.z % col_blocks) * 128;
  const int cols = vdim + 1;                               // S's columns: the values', then n's
  int lo = query_start[b], hi = query_start[b + 1];
  const int pieces = (hi - lo + pc.tokens - 1) / pc.tokens;  // (everything here is the same in all of the block's lanes)
  if (piece >= pieces || (!OUT && piece == pieces - 1)) return;
  lo += piece * pc.tokens;
  hi = min(hi, lo + pc.tokens);
  const bool from_slot = piece == 0, to_slot = OUT && piece == pieces - 1;
  const int64_t piece_no = pc.base[b] + piece;
  float* held = S_all + ((int64_t)slots[b] * heads + h) * dim * cols;
  const bool carried = starts[b] > 0;
  const float* before = from_slot && to_slot ? held
                                             : pc.sloc + ((piece_no + (from_slot ? pieces : 0) - 1) * heads + h) * dim * cols;
  const bool some = OUT && (!from_slot || carried);        // whether there is a state to start from
  const int j = col0 + 16 * wave + c;                      // this lane's value column
  const bool col = j < vdim;
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * dt + 4 * g4 + i;
      S[dt][i] = some && col && d < dim ? before[(int64_t)d * cols + j] : 0.f;
    }
  float n = some && tid < dim ? before[(int64_t)tid * cols + vdim] : 0.f;     // thread d < KD: n's element d
  if (tid < KD) n_s[tid] = n;
  float run = 1.f;                                         // the product of the piece's factors so far
  const float q_scale = 1.0f / sqrtf((float)dim);
  // what a chunk needs, on its way to registers: places that do not exist are read from ones that do and made harmless
  // when the values are used, so that nothing here waits for a load
  Piece nq[OUT ? PER : 1], nk[PER];
  T nv[CT][4];
  float ng[3];
  auto ask = [&](int t0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = (tid + e * THREADS) * VEC, t = min(t0 + idx / KD, hi - 1), d = PIECES ? idx % KD : min(idx % KD, dim - 1);
      const T* row = proj + (int64_t)t * width + h * dim + d;
      nk[e] = *reinterpret_cast<const Piece*>(row + k_off);
      if constexpr (OUT) nq[e] = *reinterpret_cast<const Piece*>(row + q_off);
    }
#pragma unroll
    for (int tt = 0; tt < CT; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        nv[tt][i] = proj[(int64_t)min(t0 + 16 * tt + 4 * g4 + i, hi - 1) * width + v_off + h * vdim + min(j, vdim - 1)];
    const float* g = pc.gates + ((int64_t)min(t0 + tid % C, hi - 1) * heads + h) * 3;
    ng[0] = g[0]; ng[1] = g[1]; ng[2] = g[2];
  };
  if (lo < hi) ask(lo);
  for (int t0 = lo; t0 < hi; t0 += C) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = (tid + e * THREADS) * VEC, at = idx / KD * QS + idx % KD;
      const bool ok = t0 + idx / KD < hi && (PIECES || idx % KD < dim);
#pragma unroll
      for (int x = 0; x < VEC; ++x) {
        ks[at + x] = ok ? Elem<T>::load(nk[e].v[x]) : 0.f;
        if constexpr (OUT) qs[at + x] = ok ? Elem<T>::load(nq[e].v[x]) * q_scale : 0.f;
      }
    }
    if (tid < C) {
      const bool ok = t0 + tid < hi;                       // (a token that is not there keeps everything and adds nothing)
      keep_s[tid] = ok ? ng[0] : 1.f;
      take_s[tid] = ok ? ng[1] : 0.f;
      low_s[tid] = ng[2];
    }
    f32x4 vv[CT];
#pragma unroll
    for (int tt = 0; tt < CT; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) vv[tt][i] = t0 + 16 * tt + 4 * g4 + i < hi && col ? Elem<T>::load(nv[tt][i]) : 0.f;
    lds_barrier();
    if (t0 + C < hi) ask(t0 + C);
    if (wave == 0) {                                       // p: products from the chunk's start; e: to its end
      float p = lane < C ? keep_s[lane] : 1.f, e = lane + 1 < C ? keep_s[lane + 1] : 1.f;
#pragma unroll
      for (int off = 1; off < C; off <<= 1) {
        const float pu = __shfl_up(p, off, WAVE), ed = __shfl_down(e, off, WAVE);
        if (lane >= off) p *= pu;
        if (lane + off < C) e *= ed;
      }
      if (lane < C) {
        p_s[lane] = p;
        e_s[lane] = take_s[lane] * e;
      }
    }
    if constexpr (OUT) {
      // fade[t][j] = M_tj: thread (j, seg) takes C / TPT neighbouring t
      constexpr int SEG = C / TPT;
      const int jj = tid % C, s0 = tid / C * SEG;
      float f = take_s[jj];
      for (int t = jj + 1; t < s0; ++t) f *= keep_s[t];
#pragma unroll
      for (int i = 0; i < SEG; ++i) {
        const int t = s0 + i;
        if (t > jj) f *= keep_s[t];
        fade[t * MS + jj] = t >= jj ? f : 0.f;
      }
      // scores: the tiles on and below the diagonal, a wave one or two
      for (int tile = wave; tile < CT * (CT + 1) / 2; tile += THREADS / WAVE) {
        int ti = 0, first = 0;
        while (first + ti + 1 <= tile) first += ++ti;
        const int tj = tile - first;
        // in float64 (v_mfma_f64_16x16x4_f64; lane (g4, c): rows 4 i + g4 of column c)
        f64x4 sum = {0., 0., 0., 0.};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const f32x4 qa = *reinterpret_cast<const f32x4*>(&qs[(16 * ti + c) * QS + 16 * dt + 4 * g4]);
          const f32x4 kb = *reinterpret_cast<const f32x4*>(&ks[(16 * tj + c) * QS + 16 * dt + 4 * g4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_mfma_f64_16x16x4f64((double)qa[i], (double)kb[i], sum, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)                        // (above the diagonal: 0, whatever a later token's key holds)
          score[(16 * ti + 4 * i + g4) * MS + 16 * tj + c] = tj < ti || 4 * i + g4 >= c ? (float)sum[i] : 0.f;
      }
    }
    lds_barrier();
    if constexpr (OUT) {
#pragma unroll
      for (int ti = 0; ti < CT; ++ti) {
        f32x4 o[4];                                        // four short chains of sums, not one long one
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const f32x4 qa = *reinterpret_cast<const f32x4*>(&qs[(16 * ti + c) * QS + 16 * dt + 4 * g4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i], S[dt][i], o[i], 0, 0, 0);
        }
        const f32x4 pt = *reinterpret_cast<const f32x4*>(&p_s[16 * ti + 4 * g4]);
        const f32x4 old = ((o[0] + o[1]) + (o[2] + o[3])) * pt;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tj = 0; tj <= ti; ++tj) {
          const int at = (16 * ti + c) * MS + 16 * tj + 4 * g4;
          const f32x4 sa = *reinterpret_cast<const f32x4*>(&score[at]) * *reinterpret_cast<const f32x4*>(&fade[at]);
#pragma unroll
          for (int i = 0; i < 4; ++i)                      // (a value times the 0 above the diagonal: see below)
            o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(sa[i], tj < ti || finite(vv[tj][i]) ? vv[tj][i] : 0.f, o[i], 0, 0, 0);
        }
        const f32x4 sum = old + ((o[0] + o[1]) + (o[2] + o[3]));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = t0 + 16 * ti + 4 * g4 + i;
          if (t < hi && col) out[((int64_t)t * heads + h) * vdim + j] = sum[i];
        }
      }
      // A value that is not finite belongs into its own token's result and the later ones', and the products on the diagonal,
      // where it would meet the earlier ones' zeros, went without it: those of its 16 tokens get it here, the lane that stored
      // a result adding to it.
      bool odd = false;
#pragma unroll
      for (int tt = 0; tt < CT; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) odd |= !finite(vv[tt][i]);
      if (__ballot(odd) != 0) {
#pragma nounroll
        for (int q = 0; q < min(C, hi - t0); ++q) {
          const float v = Elem<T>::load(proj[(int64_t)(t0 + q) * width + v_off + h * vdim + min(j, vdim - 1)]);
          if (finite(v) || !col) continue;
#pragma nounroll
          for (int t = max(q, q / 16 * 16 + 4 * g4); t < q / 16 * 16 + 4 * g4 + 4; ++t)
            if (t0 + t < hi) out[((int64_t)(t0 + t) * heads + h) * vdim + j] += score[t * MS + q] * fade[t * MS + q] * v;
        }
      }
      if (col0 == 0) {                                     // the denominators: TPT neighbouring lanes a token
        const int t = tid / TPT, part = tid % TPT;
        float dot = 0.f, sum = 0.f;
        for (int d = part; d < KD; d += TPT) dot += qs[t * QS + d] * n_s[d];
        for (int q = part; q <= t; q += TPT) sum += score[t * MS + q] * fade[t * MS + q];
        float under = dot * p_s[t] + sum;
#pragma unroll
        for (int off = 1; off < TPT; off <<= 1) under += __shfl_xor(under, off, WAVE);
        if (part == 0 && t0 + t < hi) den_out[(int64_t)(t0 + t) * heads + h] = fmaxf(fabsf(under), low_s[t]) + 1e-6f;
      }
    }
    const float all = p_s[C - 1];
    run *= all;
    if (!OUT || t0 + C < hi || to_slot) {
#pragma unroll
      for (int tt = 0; tt < CT; ++tt) vv[tt] *= *reinterpret_cast<const f32x4*>(&e_s[16 * tt + 4 * g4]);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        f32x4 add[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};         // the chunk's part: S is rounded once a chunk
#pragma unroll
        for (int tt = 0; tt < CT; ++tt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            add[i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[(16 * tt + 4 * g4 + i) * QS + 16 * dt + c], vv[tt][i],
                                                              add[i % 2], 0, 0, 0);
        S[dt] = S[dt] * all + (add[0] + add[1]);
      }
      if (tid < KD) {
        float add[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int t = 0; t < C; ++t) add[t % 4] += e_s[t] * ks[t * QS + tid];
        n = all * n + ((add[0] + add[1]) + (add[2] + add[3]));
      }
    }
    lds_barrier();                                         // all have read what the next chunk overwrites
    if (tid < KD) n_s[tid] = n;
  }
  if (OUT && !to_slot) return;
  float* left = OUT ? held : pc.sloc + (piece_no * heads + h) * dim * cols;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * dt + 4 * g4 + i;
      if (col && d < dim) left[(int64_t)d * cols + j] = S[dt][i];
    }
  if (col0 == 0 && tid < dim) left[(int64_t)tid * cols + vdim] = n;
  if (!OUT && col0 == 0 && tid == 0) pc.pk[piece_no * heads + h] = run;
}

template <typename T, int KD>
void launch_mlstm(dim3 grid, hipStream_t s, const void* proj, int width, int q_off, int k_off, int v_off, int gate_off,
                  const float* gate_bias, float cap, float* S, float* m, float* out, float* den, const int32_t* slots,
                  const int32_t* starts, const int32_t* qs, int heads, int dim, int vdim, int col_blocks) {
  mlstm_scan_kernel<KD, T><<<grid, WAVE, 0, s>>>((const T*)proj, width, q_off, k_off, v_off, gate_off, gate_bias, cap, S, m,
                                                  out, den, slots, starts, qs, heads, dim, vdim, col_blocks);
}

template <typename T, int KD>
void launch_chunks(int pass, dim3 grid, hipStream_t s, const void* proj, int width, int q_off, int k_off, int v_off, float* S,
                   float* out, float* den, const int32_t* slots, const int32_t* starts, const int32_t* qs, int heads,
                   int dim, int vdim, int col_blocks, MlstmPieces pc) {
  // keys and queries in pieces of 16 bytes, where all of a head's values are there and lie on such borders
  constexpr int V = 16 / (int)sizeof(T);
  const bool pieces = dim == KD && width % V == 0 && q_off % V == 0 && k_off % V == 0 && (uintptr_t)proj % 16 == 0;
#define CHUNKS(PASS, PIECES)                                                                                                       \
  mlstm_chunk_kernel<KD, PASS, PIECES, T><<<grid, 512, 0, s>>>((const T*)proj, width, q_off, k_off, v_off, S, out, den, slots, starts, \
                                                               qs, heads, dim, vdim, col_blocks, pc)
  if constexpr (KD == 64 || KD == 128) {
    if (pieces) {
      if (pass == 1) CHUNKS(1, true);
      else CHUNKS(2, true);
      return;
    }
  }
  if (pass == 1) CHUNKS(1, false);
  else CHUNKS(2, false);
#undef CHUNKS
}
}  // namespace

#define MLSTM_BY_KEY(dim, CALL)                               \
  do {                                                        \
    if ((dim) <= 16) { constexpr int KD = 16; CALL; }         \
    else if ((dim) <= 32) { constexpr int KD = 32; CALL; }    \
    else if ((dim) <= 64) { constexpr int KD = 64; CALL; }    \
    else if ((dim) <= 128) { constexpr int KD = 128; CALL; }  \
    else { constexpr int KD = 256; CALL; }                    \
  } while (0)

extern "C" int holon_mlstm_scan(const void* proj, int width, int q_off, int k_off, int v_off, int gate_off,
                                const float* gate_bias, float cap, float* S, float* m, float* out, float* den,
                                const int32_t* slots, const int32_t* starts, const int32_t* query_start, int rows,
                                int heads, int dim, int vdim, int state_slots, int dtype, int tokens, int piece_tokens,
                                int max_pieces, const int32_t* piece_base, float* gates, float* sloc, float* pk,
                                void* stream) {
  HOLON_CHECK(rows >= 0 && heads > 0 && heads <= 65535 && dim > 0 && dim <= 256 && vdim > 0 && state_slots > 0,
              "mlstm_scan: %d heads of %d/%d (keys of at most 256)", heads, dim, vdim);
  HOLON_CHECK(cap > 0.f && width > 0 && q_off >= 0 && k_off >= 0 && v_off >= 0 && gate_off >= 0 &&
                  q_off + heads * dim <= width && k_off + heads * dim <= width && v_off + heads * vdim <= width &&
                  gate_off + 2 * heads <= width,
              "mlstm_scan: columns do not lie within rows of %d", width);
  HOLON_CHECK(piece_tokens == 0 || (piece_tokens > 0 && max_pieces > 0 && piece_base && gates && sloc && pk),
              "mlstm_scan: rows in pieces of %d tokens need the pieces' table and workspaces", piece_tokens);
  if (rows == 0) return 0;
  const int col_blocks = (vdim + 1 + COLS - 1) / COLS;     // the values' columns and n's
  hipStream_t s = (hipStream_t)stream;
#define MLSTM_BY_TYPE(CALL)                                               \
  do {                                                                    \
    if (dtype == HOLON_F32) { using T = float; MLSTM_BY_KEY(dim, CALL); }  \
    else { using T = bf16_t; MLSTM_BY_KEY(dim, CALL); }                    \
  } while (0)
  if (piece_tokens == 0) {
    HOLON_CHECK(col_blocks <= 65535, "mlstm_scan: values of %d exceed one launch", vdim);
    MLSTM_BY_TYPE((launch_mlstm<T, KD>(dim3(rows, heads, col_blocks), s, proj, width, q_off, k_off, v_off, gate_off, gate_bias,
                                       cap, S, m, out, den, slots, starts, query_start, heads, dim, vdim, col_blocks)));
    HOLON_LAUNCH_OK();
    return 0;
  }
  (void)tokens;
  const MlstmPieces pc{piece_tokens, piece_base, gates, sloc, pk};
  const int wide = (vdim + 127) / 128;                     // blocks of 128 value columns
  HOLON_CHECK((int64_t)wide * max_pieces <= 65535, "mlstm_scan: %d pieces a row exceed one launch", max_pieces);
  if (dtype == HOLON_F32)
    mlstm_gates_kernel<float><<<dim3(rows, heads), WAVE, 0, s>>>((const float*)proj, width, gate_off, gate_bias, cap, m,
                                                                 gates, slots, starts, query_start, heads, col_blocks);
  else
    mlstm_gates_kernel<bf16_t><<<dim3(rows, heads), WAVE, 0, s>>>((const bf16_t*)proj, width, gate_off, gate_bias, cap, m,
                                                                  gates, slots, starts, query_start, heads, col_blocks);
  HOLON_LAUNCH_OK();
  const dim3 grid(rows, heads, wide * max_pieces);
  MLSTM_BY_TYPE((launch_chunks<T, KD>(1, grid, s, proj, width, q_off, k_off, v_off, S, out, den, slots, starts, query_start,
                                      heads, dim, vdim, wide, pc)));
  HOLON_LAUNCH_OK();
  const int cells = dim * (vdim + 1);
  const int walkers = (cells + 1023) / 1024;                // blocks a (row, head): four of its values a thread
  mlstm_pieces_kernel<<<dim3(rows, heads, walkers), 256, 0, s>>>(S, slots, starts, query_start, heads, cells, pc);
  HOLON_LAUNCH_OK();
  MLSTM_BY_TYPE((launch_chunks<T, KD>(2, grid, s, proj, width, q_off, k_off, v_off, S, out, den, slots, starts, query_start,
                                      heads, dim, vdim, wide, pc)));
  HOLON_LAUNCH_OK();
#undef MLSTM_BY_TYPE
  return 0;
}
