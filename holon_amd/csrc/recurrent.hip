// Recurrent mixers: a short causal filter with carried inputs, the gated delta rule, a decayed key-value memory with
// token shift, and the small float32 steps around them. A step's rows are ranges of its flat tokens
// (query_start[b] .. query_start[b + 1]), each continuing the state in its request's slot; a row that starts at
// position 0 starts from zeros whatever the slot holds.
//
// The two scans keep a head's matrix S [D, V] in registers through a row's tokens. Its columns never meet, so a wave
// owns 8 of them, eight lanes a column with an eighth of the key rows each; what a token needs of a whole column (a dot
// product with the key, the read-out) is summed over a lane's rows in ascending order and then over the eight lanes in a
// fixed order. Each token's key and query reach the lanes through LDS. The key size is padded to the next instantiated
// one with zeros (a zero key writes nothing).
#include "common.h"
#include "head_rows.h"
#include "holon_hip.h"

namespace {

// The rows of x may be columns of wider rows (x_stride values apart); `bias` is nullable. ring: the slot holds `taps`
// inputs, that of position p at place p % taps; else the last taps - 1, oldest first.
template <typename T>
__global__ void causal_conv_kernel(const T* __restrict__ x, int64_t x_stride, const T* __restrict__ w,
                                   const T* __restrict__ bias, T* __restrict__ state,
                                   T* __restrict__ y, const int32_t* __restrict__ slots,
                                   const int32_t* __restrict__ starts, const int32_t* __restrict__ query_start,
                                   const int32_t* __restrict__ token_row, int channels, int taps, int add_input,
                                   int act, int keep, int ring) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = blockIdx.y;
  if (c >= channels) return;
  const int b = keep ? t : token_row[t];               // keep: every row has one token, token t is row t
  const int q0 = keep ? t : query_start[b];
  const int i = t - q0;
  const int start = starts[b];
  const bool carried = start > 0;
  T* held = state + (int64_t)slots[b] * (ring ? taps : taps - 1) * channels;
  float acc = 0.f;
  for (int j = 0; j < taps; ++j) {
    const int l = i - (taps - 1) + j;
    float v = 0.f;
    if (l >= 0) v = Elem<T>::load(x[(q0 + l) * x_stride + c]);
    else if (carried && (!ring || start + l >= 0))
      v = Elem<T>::load(held[(int64_t)(ring ? (start + l) % taps : taps - 1 + l) * channels + c]);
    acc += Elem<T>::load(w[(int64_t)c * taps + j]) * v;
  }
  if (bias) acc += Elem<T>::load(bias[c]);
  if (add_input) acc += Elem<T>::load(x[t * x_stride + c]);
  if (act) acc = silu<T>(acc);
  y[(int64_t)t * channels + c] = Elem<T>::store(acc);
  if (keep && ring) {
    held[(int64_t)(start % taps) * channels + c] = x[t * x_stride + c];
  } else if (keep) {           // the row's one token: this thread alone reads and writes its channel of the slot
    for (int e = 0; e + 2 < taps; ++e)
      held[(int64_t)e * channels + c] = carried ? held[(int64_t)(e + 1) * channels + c] : Elem<T>::store(0.f);
    if (taps > 1) held[(int64_t)(taps - 2) * channels + c] = x[t * x_stride + c];
  }
}

// The same for prompt portions with a thread taking 16 bytes of channels at a time (channels a multiple of that; rows
// of x, y and the slots then start on 16-byte borders): the same products in the same order.
template <typename T>
__global__ void __launch_bounds__(256) causal_conv_wide_kernel(const T* __restrict__ x, int64_t x_stride,
                                                               const T* __restrict__ w, const T* __restrict__ bias,
                                                               const T* __restrict__ state, T* __restrict__ y,
                                                               const int32_t* __restrict__ slots,
                                                               const int32_t* __restrict__ starts,
                                                               const int32_t* __restrict__ query_start,
                                                               const int32_t* __restrict__ token_row, int channels,
                                                               int taps, int add_input, int act, int ring) {
  constexpr int N = Elem<T>::kVec;
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * N;
  const int t = blockIdx.y;
  if (c >= channels) return;
  const int b = token_row[t];
  const int q0 = query_start[b];
  const int i = t - q0;
  const int start = starts[b];
  const bool carried = start > 0;
  const T* held = state + (int64_t)slots[b] * (ring ? taps : taps - 1) * channels;
  float acc[N];
#pragma unroll
  for (int u = 0; u < N; ++u) acc[u] = 0.f;
  uint4 last = make_uint4(0u, 0u, 0u, 0u);
  for (int j = 0; j < taps; ++j) {
    const int l = i - (taps - 1) + j;
    uint4 raw = make_uint4(0u, 0u, 0u, 0u);
    if (l >= 0) raw = *reinterpret_cast<const uint4*>(x + (q0 + l) * x_stride + c);
    else if (carried && (!ring || start + l >= 0))
      raw = *reinterpret_cast<const uint4*>(held + (int64_t)(ring ? (start + l) % taps : taps - 1 + l) * channels + c);
    const T* v = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int u = 0; u < N; ++u) acc[u] += Elem<T>::load(w[(int64_t)(c + u) * taps + j]) * Elem<T>::load(v[u]);
    last = raw;
  }
  const T* own = reinterpret_cast<const T*>(&last);      // the last tap's input is the token itself
  uint4 out;
  T* o = reinterpret_cast<T*>(&out);
#pragma unroll
  for (int u = 0; u < N; ++u) {
    float a = acc[u];
    if (bias) a += Elem<T>::load(bias[c + u]);
    if (add_input) a += Elem<T>::load(own[u]);
    if (act) a = silu<T>(a);
    o[u] = Elem<T>::store(a);
  }
  *reinterpret_cast<uint4*>(y + (int64_t)t * channels + c) = out;
}

// The same for up to four taps with a thread taking RUN neighbouring tokens: its channels' taps are read once, as whole
// vectors, and an input serves every token of the run that it reaches. Tokens of a run may belong to different rows; an
// input in front of its row's first token comes from the row's slot.
template <typename T, int TAPS>
__global__ void __launch_bounds__(256) causal_conv_run_kernel(const T* __restrict__ x, int64_t x_stride,
                                                              const T* __restrict__ w, const T* __restrict__ bias,
                                                              const T* __restrict__ state, T* __restrict__ y,
                                                              const int32_t* __restrict__ slots,
                                                              const int32_t* __restrict__ starts,
                                                              const int32_t* __restrict__ query_start,
                                                              const int32_t* __restrict__ token_row, int tokens,
                                                              int channels, int add_input, int act, int ring) {
  constexpr int N = Elem<T>::kVec, RUN = 8;
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * N, t0 = blockIdx.y * RUN;
  if (c >= channels) return;
  uint4 win[RUN + TAPS - 1];                             // the inputs of tokens t0 - TAPS + 1 .. t0 + RUN - 1
#pragma unroll
  for (int e = 0; e < RUN + TAPS - 1; ++e) {
    const int t = t0 - (TAPS - 1) + e;
    win[e] = t >= 0 && t < tokens ? *reinterpret_cast<const uint4*>(x + t * x_stride + c) : make_uint4(0u, 0u, 0u, 0u);
  }
  float wv[N * TAPS], bv[N];
#pragma unroll
  for (int e = 0; e < TAPS; ++e) {                       // (N TAPS values are TAPS whole vectors)
    const uint4 raw = *reinterpret_cast<const uint4*>(w + (int64_t)c * TAPS + e * N);
    const T* v = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int u = 0; u < N; ++u) wv[e * N + u] = Elem<T>::load(v[u]);
  }
#pragma unroll
  for (int u = 0; u < N; ++u) bv[u] = bias ? Elem<T>::load(bias[c + u]) : 0.f;
#pragma unroll
  for (int r = 0; r < RUN; ++r) {
    const int t = t0 + r;
    if (t >= tokens) break;
    const int b = token_row[t], i = t - query_start[b];
    float acc[N];
#pragma unroll
    for (int u = 0; u < N; ++u) acc[u] = 0.f;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
      const int l = i - (TAPS - 1) + j;
      uint4 raw = win[r + j];
      if (l < 0) {
        const int start = starts[b];
        raw = make_uint4(0u, 0u, 0u, 0u);
        if (start > 0 && (!ring || start + l >= 0))
          raw = *reinterpret_cast<const uint4*>(state + ((int64_t)slots[b] * (ring ? TAPS : TAPS - 1) +
                                                         (ring ? (start + l) % TAPS : TAPS - 1 + l)) * channels + c);
      }
      const T* v = reinterpret_cast<const T*>(&raw);
#pragma unroll
      for (int u = 0; u < N; ++u) acc[u] += wv[u * TAPS + j] * Elem<T>::load(v[u]);
    }
    const T* own = reinterpret_cast<const T*>(&win[r + TAPS - 1]);
    uint4 out;
    T* o = reinterpret_cast<T*>(&out);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      float a = bias ? acc[u] + bv[u] : acc[u];
      if (add_input) a += Elem<T>::load(own[u]);
      if (act) a = silu<T>(a);
      o[u] = Elem<T>::store(a);
    }
    *reinterpret_cast<uint4*>(y + (int64_t)t * channels + c) = out;
  }
}

// After the filter has read the old inputs: the slot takes the row's last taps - 1 inputs, oldest first. A thread
// moves its channel's entries in ascending order and reads only entries at or behind the one it writes. (A ring takes the
// row's own last inputs at their places; older ones lie where they are.)
template <typename T>
__global__ void causal_conv_keep_kernel(const T* __restrict__ x, int64_t x_stride, T* __restrict__ state,
                                        const int32_t* __restrict__ slots,
                                        const int32_t* __restrict__ starts, const int32_t* __restrict__ query_start,
                                        int channels, int taps, int ring) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (c >= channels) return;
  const int q0 = query_start[b], n = query_start[b + 1] - q0;
  const bool carried = starts[b] > 0;
  T* held = state + (int64_t)slots[b] * (ring ? taps : taps - 1) * channels;
  if (ring) {
    for (int l = max(0, n - taps); l < n; ++l)
      held[(int64_t)((starts[b] + l) % taps) * channels + c] = x[(q0 + l) * x_stride + c];
    return;
  }
  for (int i = 0; i < taps - 1; ++i) {
    const int l = n - (taps - 1) + i;
    T v = Elem<T>::store(0.f);
    if (l >= 0) v = x[(q0 + l) * x_stride + c];
    else if (carried) v = held[(int64_t)(i + n) * channels + c];
    held[(int64_t)i * channels + c] = v;
  }
}

__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// One block a token. Waves take the 2 G heads of q and k in turn: unit vectors (q also times D^-0.5); then the step
// sizes and decays of the H heads.
template <typename T>
__global__ void __launch_bounds__(256) delta_prepare_kernel(const T* __restrict__ qkv, const T* __restrict__ ab,
                                                            const float* __restrict__ a_log,
                                                            const float* __restrict__ dt_bias, float* __restrict__ qn,
                                                            float* __restrict__ kn, float* __restrict__ beta,
                                                            float* __restrict__ g, int heads, int kv_heads, int dim,
                                                            int vdim) {
  const int t = blockIdx.x;
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int width = 2 * kv_heads * dim + heads * vdim;
  const T* row = qkv + (int64_t)t * width;
  for (int idx = wave; idx < 2 * kv_heads; idx += 4) {
    const bool is_q = idx < kv_heads;
    const int h = is_q ? idx : idx - kv_heads;
    const T* src = row + (int64_t)idx * dim;
    float ss = 0.f;
    for (int d = lane; d < dim; d += WAVE) {
      const float v = Elem<T>::load(src[d]);
      ss += v * v;
    }
    ss = wave_sum(ss);
    const float r = (1.0f / sqrtf(ss + 1e-6f)) * (is_q ? 1.0f / sqrtf((float)dim) : 1.0f);
    float* dst = (is_q ? qn : kn) + ((int64_t)t * kv_heads + h) * dim;
    for (int d = lane; d < dim; d += WAVE) dst[d] = Elem<T>::load(src[d]) * r;
  }
  for (int h = threadIdx.x; h < heads; h += 256) {
    const float a = Elem<T>::load(ab[(int64_t)t * 2 * heads + h]);
    const float b = Elem<T>::load(ab[(int64_t)t * 2 * heads + heads + h]);
    beta[(int64_t)t * heads + h] = 1.0f / (1.0f + expf(-b));
    g[(int64_t)t * heads + h] = expf(-expf(a_log[h]) * softplus_f(a + dt_bias[h]));
  }
}

// Sum over the eight adjacent lanes that share a column, by data-parallel moves inside the vector unit (no trip through
// LDS): lane ^ 1, lane ^ 2, then the mirror image inside the eight, which lies in the other four. A fixed order.
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float part_sum(float v) {
  v += dpp_move<0xB1>(v);        // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);        // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);       // row_half_mirror
  return v;
}

constexpr int SCAN_PARTS = 8;      // lanes a value column is spread over, each with an eighth of the key rows
constexpr int SCAN_COLS = WAVE / SCAN_PARTS;      // value columns a wave owns

// Tokens a wave stages at a time: their operands travel from memory to LDS as one batch of loads while the batch before
// is worked through, so that a token's arithmetic never waits for memory (one token at a time, a step took as long as
// a load: 0.9 us). About a thousand values per operand and batch.
// ARRAYS: operands of D values a token that the scan stages (they decide the block's LDS, and with it how many waves a
// compute unit holds: the scans wait on latencies, so more waves are more throughput).
template <int KD, int ARRAYS> struct ScanChunk {
  static constexpr int kTokens = ARRAYS <= 2 ? (KD <= 64 ? 16 : KD <= 128 ? 8 : 4) : (KD <= 64 ? 8 : KD <= 128 ? 4 : 2);
};

// Per (row, head): S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q. Lane 8 c + p owns rows
// p KD/8 .. (p + 1) KD/8 - 1 of column c of S. (Longer rows go in blocks of tokens on the matrix cores: delta_rule.hip; `piece_of`, nullable,
// says which rows do.)
template <int KD, typename T>
__global__ void __launch_bounds__(WAVE) delta_scan_kernel(const float* __restrict__ qn, const float* __restrict__ kn,
                                                          const T* __restrict__ qkv, int qkv_stride, int v_offset,
                                                          const float* __restrict__ beta, const float* __restrict__ g,
                                                          float* __restrict__ state, float* __restrict__ out,
                                                          const int32_t* __restrict__ slots,
                                                          const int32_t* __restrict__ starts,
                                                          const int32_t* __restrict__ query_start,
                                                          const int32_t* __restrict__ piece_of, int heads, int kv_heads, int dim,
                                                          int vdim) {
  constexpr int KQ = KD / SCAN_PARTS, TC = ScanChunk<KD, 2>::kTokens, N = TC * KD, PER = (N + WAVE - 1) / WAVE;
  constexpr int VPER = (TC * SCAN_COLS + WAVE - 1) / WAVE;
  __shared__ __attribute__((aligned(16))) float ks[2][N], qs[2][N];
  __shared__ float vs[2][TC * SCAN_COLS], gs[2][TC], bs[2][TC];
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  if (piece_of && piece_of[b] > 0) return;               // (uniform over the block)
  const int col_block = blockIdx.z;
  const int part = lane % SCAN_PARTS, col = lane / SCAN_PARTS, j = col_block * SCAN_COLS + col;
  const int hk = h / (heads / kv_heads);
  const bool active = j < vdim;
  const int lo = query_start[b], hi = query_start[b + 1];
  float* held = state + ((int64_t)slots[b] * heads + h) * dim * vdim;
  const bool some = starts[b] > 0;                       // whether there is a state to start from
  float S[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    const bool in = active && row < dim;
    S[i] = some && in ? held[(int64_t)row * vdim + j] : 0.f;
  }
  float nk[PER], nq[PER], nv[VPER], ng = 1.f, nb = 0.f;
  auto ask = [&](int t0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE, tt = idx / KD, i = idx - tt * KD;
      const bool ok = idx < N && t0 + tt < hi && i < dim;
      const int64_t at = ((int64_t)(t0 + tt) * kv_heads + hk) * dim + i;
      nk[e] = ok ? kn[at] : 0.f;
      nq[e] = ok ? qn[at] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < VPER; ++e) {
      const int idx = lane + e * WAVE, tt = idx / SCAN_COLS, jj = col_block * SCAN_COLS + idx % SCAN_COLS;
      const bool ok = idx < TC * SCAN_COLS && t0 + tt < hi && jj < vdim;
      nv[e] = ok ? Elem<T>::load(qkv[(int64_t)(t0 + tt) * qkv_stride + v_offset + h * vdim + jj]) : 0.f;
    }
    const bool ok = lane < TC && t0 + lane < hi;
    ng = ok ? g[(int64_t)(t0 + lane) * heads + h] : 1.f;
    nb = ok ? beta[(int64_t)(t0 + lane) * heads + h] : 0.f;
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < N) { ks[buf][idx] = nk[e]; qs[buf][idx] = nq[e]; }
    }
#pragma unroll
    for (int e = 0; e < VPER; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < TC * SCAN_COLS) vs[buf][idx] = nv[e];
    }
    if (lane < TC) { gs[buf][lane] = ng; bs[buf][lane] = nb; }
  };
  if (lo < hi) {
    ask(lo);
    put(0);
  }
  __syncthreads();
  for (int t0 = lo, buf = 0; t0 < hi; t0 += TC, buf ^= 1) {
    if (t0 + TC < hi) ask(t0 + TC);
    const int nt = min(TC, hi - t0);
    for (int tt = 0; tt < nt; ++tt) {
      const float gt = gs[buf][tt], bt = bs[buf][tt], vt = vs[buf][tt * SCAN_COLS + col];
      const float* kt = &ks[buf][tt * KD + part * KQ];
      const float* qt = &qs[buf][tt * KD + part * KQ];
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        S[i] *= gt;
        dot += S[i] * kt[i];
      }
      const float u = bt * (vt - part_sum(dot));
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        S[i] += kt[i] * u;
        o += S[i] * qt[i];
      }
      o = part_sum(o);
      if (active && part == 0) out[((int64_t)(t0 + tt) * heads + h) * vdim + j] = o;
    }
    if (t0 + TC < hi) put(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    if (active && row < dim) held[(int64_t)row * vdim + j] = S[i];
  }
}

// Per (row, head): o = (S + diag(u) k v^T)^T r; S <- diag(w) S + k v^T. The same split of S [D, D] over lanes. (Rows in
// pieces go on the matrix cores: `holon_memory_scan_pieces`. Short rows stay here, where every sum's order is the token's
// alone.)
template <int KD, typename T>
__global__ void __launch_bounds__(WAVE) memory_scan_kernel(const T* __restrict__ r, const T* __restrict__ k,
                                                           const T* __restrict__ v, const float* __restrict__ w,
                                                           const float* __restrict__ u, float* __restrict__ state,
                                                           float* __restrict__ out, const int32_t* __restrict__ slots,
                                                           const int32_t* __restrict__ starts,
                                                           const int32_t* __restrict__ query_start, int heads, int dim) {
  constexpr int KQ = KD / SCAN_PARTS, TC = ScanChunk<KD, 3>::kTokens, N = TC * KD, PER = (N + WAVE - 1) / WAVE;
  constexpr int VPER = (TC * SCAN_COLS + WAVE - 1) / WAVE;
  __shared__ __attribute__((aligned(16))) float rs[2][N], ks[2][N], ws[2][N], us[KD];
  __shared__ float vs[2][TC * SCAN_COLS];
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int col_block = blockIdx.z;
  const int part = lane % SCAN_PARTS, col = lane / SCAN_PARTS, j = col_block * SCAN_COLS + col;
  const bool active = j < dim;
  const int lo = query_start[b], hi = query_start[b + 1];
  float* held = state + ((int64_t)slots[b] * heads + h) * dim * dim;
  const bool carried = starts[b] > 0;
  float S[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    S[i] = carried && active && row < dim ? held[(int64_t)row * dim + j] : 0.f;
  }
  for (int i = lane; i < KD; i += WAVE) us[i] = i < dim ? u[h * dim + i] : 0.f;
  const int64_t width = (int64_t)heads * dim;
  float nr[PER], nk[PER], nw[PER], nv[VPER];
  auto ask = [&](int t0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE, tt = idx / KD, i = idx - tt * KD;
      const bool ok = idx < N && t0 + tt < hi && i < dim;
      const int64_t at = (int64_t)(t0 + tt) * width + h * dim + i;
      nr[e] = ok ? Elem<T>::load(r[at]) : 0.f;
      nk[e] = ok ? Elem<T>::load(k[at]) : 0.f;
      nw[e] = ok ? w[at] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < VPER; ++e) {
      const int idx = lane + e * WAVE, tt = idx / SCAN_COLS, jj = col_block * SCAN_COLS + idx % SCAN_COLS;
      const bool ok = idx < TC * SCAN_COLS && t0 + tt < hi && jj < dim;
      nv[e] = ok ? Elem<T>::load(v[(int64_t)(t0 + tt) * width + h * dim + jj]) : 0.f;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < N) { rs[buf][idx] = nr[e]; ks[buf][idx] = nk[e]; ws[buf][idx] = nw[e]; }
    }
#pragma unroll
    for (int e = 0; e < VPER; ++e) {
      const int idx = lane + e * WAVE;
      if (idx < TC * SCAN_COLS) vs[buf][idx] = nv[e];
    }
  };
  if (lo < hi) {
    ask(lo);
    put(0);
  }
  __syncthreads();
  for (int t0 = lo, buf = 0; t0 < hi; t0 += TC, buf ^= 1) {
    if (t0 + TC < hi) ask(t0 + TC);
    const int nt = min(TC, hi - t0);
    for (int tt = 0; tt < nt; ++tt) {
      const float vt = vs[buf][tt * SCAN_COLS + col];
      const float* rt = &rs[buf][tt * KD + part * KQ];
      const float* kt = &ks[buf][tt * KD + part * KQ];
      const float* wt = &ws[buf][tt * KD + part * KQ];
      const float* ut = &us[part * KQ];
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        const float kv = kt[i] * vt;
        o += rt[i] * (S[i] + ut[i] * kv);
        S[i] = wt[i] * S[i] + kv;
      }
      o = part_sum(o);
      if (active && part == 0) out[(int64_t)(t0 + tt) * width + h * dim + j] = o;
    }
    if (t0 + TC < hi) put(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int row = part * KQ + i;
    if (!active || row >= dim) continue;
    held[(int64_t)row * dim + j] = S[i];
  }
}

// One wave per (token, head): o / sqrt(mean(o^2) + eps) * weight * act(gate), act = silu, or the sigmoid alone
// (`plain_sigmoid`). A token's gates are `gate_stride` values apart (columns of a wider projection). With `den`
// (one value a token and head) o is divided by it first.
template <typename T>
__global__ void __launch_bounds__(256) gated_out_kernel(const float* __restrict__ o, const T* __restrict__ gate,
                                                        const T* __restrict__ weight, T* __restrict__ y, int64_t cells,
                                                        int heads, int vdim, int per_head, float eps,
                                                        int64_t gate_stride, int plain_sigmoid,
                                                        const float* __restrict__ den) {
  const int64_t cell = (int64_t)blockIdx.x * 4 + threadIdx.x / WAVE;
  const int lane = threadIdx.x % WAVE;
  if (cell >= cells) return;
  const int h = (int)(cell % heads);
  const float* src = o + cell * vdim;
  const float under = den ? den[cell] : 1.f;
  float ss = 0.f;
  for (int d = lane; d < vdim; d += WAVE) {
    const float v = den ? src[d] / under : src[d];
    ss += v * v;
  }
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)vdim + eps);
  for (int d = lane; d < vdim; d += WAVE) {
    const float wv = Elem<T>::load(weight[per_head ? h * vdim + d : d]);
    const float gv = Elem<T>::load(gate[(cell / heads) * gate_stride + (int64_t)h * vdim + d]);
    const float act = plain_sigmoid ? 1.0f / (1.0f + expf(-gv)) : silu<T>(gv);
    y[cell * vdim + d] = Elem<T>::store((den ? src[d] / under : src[d]) * r * wv * act);
  }
}

// The same for heads of 64, 128 and 256 (LANES 8, 16, 32) on borders of 16 bytes: eight neighbouring values a lane, 64 / LANES cells a wave, every
// load under way before a sum is taken. The same bits. 2,048 tokens of 32 heads of 64 7.6 us, a value a lane at a time 20.8 (33 MB: 6.8
// at a copy's rate).
template <typename T, int LANES>
__global__ void __launch_bounds__(256) gated_out_rows_kernel(const float* __restrict__ o, const T* __restrict__ gate,
                                                             const T* __restrict__ weight, T* __restrict__ y, int64_t cells, int heads,
                                                             int per_head, float eps, int64_t gate_stride, int plain_sigmoid,
                                                             const float* __restrict__ den) {
  constexpr int D = LANES * 8, PER = WAVE / LANES;
  const int lane = threadIdx.x % WAVE, d0 = lane % LANES * 8;
  const int64_t cell = ((int64_t)blockIdx.x * 4 + threadIdx.x / WAVE) * PER + lane / LANES, at = min(cell, cells - 1);
  const int h = (int)(at % heads);
  float v[8], wv[8], gv[8];
  head_rows::load8(o + at * D + d0, v);
  head_rows::load8(weight + (per_head ? h * D : 0) + d0, wv);
  head_rows::load8(gate + (at / heads) * gate_stride + (int64_t)h * D + d0, gv);
  if (den) {
    const float under = den[at];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = v[j] / under;
  }
  const float r = 1.0f / sqrtf(head_rows::sum_of_squares<LANES>(v, lane) / (float)D + eps);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = v[j] * r * wv[j] * (plain_sigmoid ? 1.0f / (1.0f + expf(-gv[j])) : silu<T>(gv[j]));
  if (cell < cells) head_rows::store8(y + cell * D + d0, v);
}

template <typename T>
__global__ void shift_mix_kernel(const T* __restrict__ x, const T* __restrict__ mu, T* __restrict__ state,
                                 T* __restrict__ y, const int32_t* __restrict__ slots, const int32_t* __restrict__ starts,
                                 const int32_t* __restrict__ query_start, const int32_t* __restrict__ token_row,
                                 int tokens, int width, int mixes, int keep) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = blockIdx.y;
  if (c >= width) return;
  const int b = keep ? t : token_row[t];               // keep: every row has one token, token t is row t
  float prev = 0.f;
  if (!keep && t > query_start[b]) prev = Elem<T>::load(x[(int64_t)(t - 1) * width + c]);
  else if (starts[b] > 0) prev = Elem<T>::load(state[(int64_t)slots[b] * width + c]);
  const float cur = Elem<T>::load(x[(int64_t)t * width + c]);
  for (int s = 0; s < mixes; ++s)
    y[((int64_t)s * tokens + t) * width + c] = Elem<T>::store(cur + (prev - cur) * Elem<T>::load(mu[(int64_t)s * width + c]));
  if (keep) state[(int64_t)slots[b] * width + c] = x[(int64_t)t * width + c];
}

// The same, 16 bytes of neighbouring channels a thread and load, for steps of SHIFT_PIECES_FROM values (tokens times channels) and more: below, a
// block's round of latency is what a step takes, and a thread with more to do makes it longer. A row's blocks are as many as 256 threads each need,
// of as many waves as an even share takes. Over 10,560 steps the choice is 0.3 % from the better form on average and up to 14 % (3,136 float32 channels, six
// mixes). In us, pieces against a channel a thread: 2,058 tokens of 2,048 mixed five times 14.2 / 23.7 (bfloat16), 1,913 20.2 / 21.9 (float32), 196 of
// 1,920 5.4 / 5.9 and 209 of 2,048 5.8 / 6.0; 383 of 1,024 5.5 / 5.8 and 350 of 1,088 5.8 / 5.9; 69 of 2,048 5.1 / 4.7 and 67 5.1 / 4.6. (Eight
// float32 channels a thread, 32 bytes apart from the next thread's, took up to 1.29 times as long as one.)
constexpr int64_t SHIFT_PIECES_FROM = 196608, SHIFT_PIECES_FROM_F32 = 262144;
template <typename T>
__global__ void __launch_bounds__(256) shift_mix_rows_kernel(const T* __restrict__ x, const T* __restrict__ mu, T* __restrict__ state,
                                                             T* __restrict__ y, const int32_t* __restrict__ slots,
                                                             const int32_t* __restrict__ starts, const int32_t* __restrict__ query_start,
                                                             const int32_t* __restrict__ token_row, int tokens, int width, int mixes,
                                                             int keep) {
  constexpr int N = Elem<T>::kVec;
  struct alignas(16) Piece { T v[N]; };
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * N;
  const int t = blockIdx.y;
  if (c >= width) return;
  const int b = keep ? t : token_row[t];
  Piece prev{}, cur = *reinterpret_cast<const Piece*>(x + (int64_t)t * width + c);
  if (!keep && t > query_start[b]) prev = *reinterpret_cast<const Piece*>(x + (int64_t)(t - 1) * width + c);
  else if (starts[b] > 0) prev = *reinterpret_cast<const Piece*>(state + (int64_t)slots[b] * width + c);
  for (int s = 0; s < mixes; ++s) {
    Piece m = *reinterpret_cast<const Piece*>(mu + (int64_t)s * width + c);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float now = Elem<T>::load(cur.v[j]), before = Elem<T>::load(prev.v[j]);
      m.v[j] = Elem<T>::store(now + (before - now) * Elem<T>::load(m.v[j]));
    }
    *reinterpret_cast<Piece*>(y + ((int64_t)s * tokens + t) * width + c) = m;
  }
  if (keep) *reinterpret_cast<Piece*>(state + (int64_t)slots[b] * width + c) = cur;
}

template <typename T>
__global__ void shift_keep_kernel(const T* __restrict__ x, T* __restrict__ state, const int32_t* __restrict__ slots,
                                  const int32_t* __restrict__ query_start, int width) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (c >= width) return;
  state[(int64_t)slots[b] * width + c] = x[(int64_t)(query_start[b + 1] - 1) * width + c];
}

// exp(-exp(tanh(a) w2^T + w0)) on the float32 matrix cores, whose sums are the chain of multiply-adds in ascending order. A block takes 16
// tokens and 256 channels, a wave 64 of them: lane l's four neighbouring channels are column l % 16 of four tiles, so that one load of w2
// (transposed, [rank, channels]) serves them all. The tokens' tanh values lie in LDS. FOURS: there are four channels; a lane whose four would
// end behind the last channel takes the last four, which a neighbour has as well: the same sums, stored twice. (Loads and stores of four
// are aligned as one value is, so that any number of channels takes them; value by value 17 tokens of 1,030 channels of rank 30 took 7.6 us, so 5.2.)
// A lane's four results of a tile are tokens g, 4 + g, 8 + g and 12 + g, so that a step of up to four tokens has one for every lane.
// 2,048 tokens by 2,048 channels of rank 64 17 us and one token 4.9 (on the vector unit, a token's value read from LDS for every
// multiply-add, 27 and 8.4).
__host__ __device__ constexpr int lora_pitch(int rank) { return (rank + 3) / 4 * 4 + (rank < 1000 ? 1 : 0); }      // (at most 64 KB of LDS)
constexpr int LORA_TOKENS = 16, LORA_MAX_RANK = 1024, LORA_AHEAD = 8;      // LORA_AHEAD: steps of four ranks whose weights are asked for at a time
template <bool FOURS, typename T>
__global__ void __launch_bounds__(256) decay_lora_kernel(const float* __restrict__ a, const T* __restrict__ w2t,
                                                         const float* __restrict__ w0, float* __restrict__ y, int tokens,
                                                         int channels, int rank) {
  extern __shared__ float th[];                            // [16][pitch], zeros behind the rank
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int steps = (rank + 3) / 4, pitch = lora_pitch(rank);
  const int t0 = blockIdx.x * LORA_TOKENS, lane = threadIdx.x % WAVE, g = lane / 16, c = lane % 16;
  const int first = blockIdx.y * 256 + threadIdx.x / WAVE * 64 + 4 * c, c0 = FOURS ? min(first, channels - 4) : first;
  T next[LORA_AHEAD][4];
  const auto ask = [&](int s0) {
#pragma unroll
    for (int u = 0; u < LORA_AHEAD; ++u) {
      const int64_t row = (int64_t)min(4 * (s0 + u) + g, rank - 1) * channels;
      if constexpr (FOURS) {
        struct Four { T v[4]; };
        const Four v = *reinterpret_cast<const Four*>(w2t + row + c0);
#pragma unroll
        for (int n = 0; n < 4; ++n) next[u][n] = v.v[n];
      } else {
#pragma unroll
        for (int n = 0; n < 4; ++n) next[u][n] = w2t[row + min(c0 + n, channels - 1)];
      }
    }
  };
  ask(0);
  for (int e = threadIdx.x; e < LORA_TOKENS * 4 * steps; e += 256) {
    const int tt = e / (4 * steps), r = e - tt * 4 * steps;
    th[tt * pitch + r] = t0 + tt < tokens && r < rank ? tanhf(a[(int64_t)(t0 + tt) * rank + r]) : 0.f;
  }
  __syncthreads();
  f32x4 acc[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < steps; s0 += LORA_AHEAD) {
    float w[LORA_AHEAD][4];
#pragma unroll
    for (int u = 0; u < LORA_AHEAD; ++u)
#pragma unroll
      for (int n = 0; n < 4; ++n) w[u][n] = 4 * (s0 + u) + g < rank ? Elem<T>::load(next[u][n]) : 0.f;
    if (s0 + LORA_AHEAD < steps) ask(s0 + LORA_AHEAD);
#pragma unroll
    for (int u = 0; u < LORA_AHEAD; ++u) {
      if (s0 + u >= steps) break;
      const float x = th[(c % 4 * 4 + c / 4) * pitch + 4 * (s0 + u) + g];
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, w[u][n], acc[n], 0, 0, 0);
    }
  }
  float off[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) off[n] = w0[min(c0 + n, channels - 1)];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                            // lane: tokens 4 i + g of its four channels
    const int t = t0 + 4 * i + g;
    if (t >= tokens) continue;
    struct Four { float v[4]; } o;
#pragma unroll
    for (int n = 0; n < 4; ++n) o.v[n] = expf(-expf(acc[n][i] + off[n]));
    if constexpr (FOURS) {
      if (first < channels) *reinterpret_cast<Four*>(y + (int64_t)t * channels + c0) = o;
    } else {
#pragma unroll
      for (int n = 0; n < 4; ++n)
        if (c0 + n < channels) y[(int64_t)t * channels + c0 + n] = o.v[n];
    }
  }
}

}  // namespace

#define BY_DTYPE(dtype, CALL)                    \
  do {                                           \
    if ((dtype) == HOLON_F32) { using T = float; CALL; } \
    else { using T = bf16_t; CALL; }             \
  } while (0)

extern "C" int holon_causal_conv(const void* x, int64_t x_stride, const void* w, const void* bias, void* state, void* y,
                                 const int32_t* slots,
                                 const int32_t* starts, const int32_t* query_start, const int32_t* token_row,
                                 int tokens, int rows, int channels, int taps, int state_slots, int add_input, int act,
                                 int dtype, int rows_in_order, int ring, void* stream) {
  HOLON_CHECK(tokens >= 0 && rows >= 0 && channels > 0 && taps >= 1 && taps <= 16 && state_slots > 0,
              "causal_conv: tokens=%d rows=%d channels=%d taps=%d", tokens, rows, channels, taps);
  HOLON_CHECK(tokens <= 65535 && rows <= 65535, "causal_conv: %d tokens in %d rows exceed one launch", tokens, rows);
  HOLON_CHECK(x_stride >= channels, "causal_conv: rows of %d channels %lld apart", channels, (long long)x_stride);
  if (tokens == 0 || rows == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const dim3 block(256), grid_t((channels + 255) / 256, tokens), grid_b((channels + 255) / 256, rows);
  HOLON_CHECK(!rows_in_order || tokens == rows, "causal_conv: rows in order means one token a row, got %d in %d", tokens,
              rows);
  const int vec = dtype == HOLON_F32 ? 4 : 8;
  if (!rows_in_order && channels % vec == 0 && x_stride % vec == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)y % 16 == 0 &&
      (uintptr_t)state % 16 == 0) {
    const dim3 grid_w((channels / vec + 255) / 256, tokens), grid_r((channels / vec + 255) / 256, (tokens + 7) / 8);
#define CONV_RUN(K)                                                                                                    \
  BY_DTYPE(dtype, (causal_conv_run_kernel<T, K><<<grid_r, block, 0, s>>>((const T*)x, x_stride, (const T*)w,           \
                                                                         (const T*)bias, (const T*)state, (T*)y, slots, \
                                                                         starts, query_start, token_row, tokens,       \
                                                                         channels, add_input, act, ring)))
    const bool whole_taps = (uintptr_t)w % 16 == 0;
    if (whole_taps && taps == 2) CONV_RUN(2);
    else if (whole_taps && taps == 3) CONV_RUN(3);
    else if (whole_taps && taps == 4) CONV_RUN(4);
    else BY_DTYPE(dtype, (causal_conv_wide_kernel<T><<<grid_w, block, 0, s>>>((const T*)x, x_stride, (const T*)w,
                                                                         (const T*)bias, (const T*)state, (T*)y,
                                                                         slots, starts, query_start, token_row,
                                                                         channels, taps, add_input, act, ring)));
  } else {
    BY_DTYPE(dtype, (causal_conv_kernel<T><<<grid_t, block, 0, s>>>((const T*)x, x_stride, (const T*)w, (const T*)bias,
                                                                    (T*)state, (T*)y, slots, starts, query_start,
                                                                    token_row, channels, taps, add_input, act,
                                                                    rows_in_order, ring)));
  }
  HOLON_LAUNCH_OK();
  if ((taps > 1 || ring) && !rows_in_order) {
    BY_DTYPE(dtype, (causal_conv_keep_kernel<T><<<grid_b, block, 0, s>>>((const T*)x, x_stride, (T*)state, slots, starts,
                                                                         query_start, channels, taps, ring)));
    HOLON_LAUNCH_OK();
  }
  return 0;
}

extern "C" int holon_delta_prepare(const void* qkv, const void* ab, const float* a_log, const float* dt_bias, float* qn,
                                   float* kn, float* beta, float* g, int tokens, int heads, int kv_heads, int dim,
                                   int vdim, int dtype, void* stream) {
  HOLON_CHECK(tokens >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0,
              "delta_prepare: %d/%d heads of %d/%d", heads, kv_heads, dim, vdim);
  if (tokens == 0) return 0;
  BY_DTYPE(dtype, (delta_prepare_kernel<T><<<tokens, 256, 0, (hipStream_t)stream>>>(
                      (const T*)qkv, (const T*)ab, a_log, dt_bias, qn, kn, beta, g, heads, kv_heads, dim, vdim)));
  HOLON_LAUNCH_OK();
  return 0;
}

template <typename T, int KD>
static void launch_delta(dim3 grid, hipStream_t s, const float* qn, const float* kn, const void* qkv,
                         int stride, int voff, const float* beta, const float* g, float* state, float* out,
                         const int32_t* slots, const int32_t* starts, const int32_t* qs, const int32_t* piece_of, int heads,
                         int kv_heads, int dim, int vdim) {
  delta_scan_kernel<KD, T><<<grid, WAVE, 0, s>>>(qn, kn, (const T*)qkv, stride, voff, beta, g, state, out, slots,
                                                    starts, qs, piece_of, heads, kv_heads, dim, vdim);
}

#define BY_KEY_SIZE(dim, CALL)                                  \
  do {                                                          \
    if ((dim) <= 16) { constexpr int KD = 16; CALL; }           \
    else if ((dim) <= 32) { constexpr int KD = 32; CALL; }      \
    else if ((dim) <= 48) { constexpr int KD = 48; CALL; }      \
    else if ((dim) <= 64) { constexpr int KD = 64; CALL; }      \
    else if ((dim) <= 96) { constexpr int KD = 96; CALL; }      \
    else if ((dim) <= 128) { constexpr int KD = 128; CALL; }    \
    else if ((dim) <= 192) { constexpr int KD = 192; CALL; }    \
    else { constexpr int KD = 256; CALL; }                      \
  } while (0)

int holon_delta_scan_pieces(const float* qn, const float* kn, const void* qkv, int qkv_stride, int v_offset, const float* beta,
                            const float* g, float* state, float* out, const int32_t* slots, const int32_t* starts,
                            const int32_t* query_start, int rows, int heads, int kv_heads, int dim, int vdim, int dtype,
                            int piece_tokens, int max_pieces, const int32_t* piece_base, const int32_t* piece_of, float* blocks,
                            float* a, float* sin, void* stream);

extern "C" int holon_delta_scan(const float* qn, const float* kn, const void* qkv, int qkv_stride, int v_offset,
                                const float* beta, const float* g, float* state, float* out, const int32_t* slots,
                                const int32_t* starts, const int32_t* query_start, int rows, int heads, int kv_heads,
                                int dim, int vdim, int state_slots, int dtype, int piece_tokens, int max_pieces,
                                const int32_t* piece_base, const int32_t* piece_of, float* blocks, float* a, float* sin, void* stream) {
  HOLON_CHECK(rows >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "delta_scan: %d/%d heads", heads, kv_heads);
  HOLON_CHECK(dim > 0 && dim <= 256 && vdim > 0 && vdim <= 1024, "delta_scan: key size %d (at most 256), value size %d "
              "(at most 1024)", dim, vdim);
  HOLON_CHECK(rows <= 0x7fffffff / 2 && heads <= 65535 && state_slots > 0 && v_offset >= 0 &&
              v_offset + heads * vdim <= qkv_stride, "delta_scan: launch or row layout out of range");
  HOLON_CHECK(piece_tokens == 0 || (piece_tokens > 0 && piece_tokens % 16 == 0 && max_pieces > 0 && piece_base && blocks &&
                                    (max_pieces == 1 || (a && sin)) && (((uintptr_t)blocks | (uintptr_t)a) & 15) == 0),
              "delta_scan: rows in pieces of %d tokens (a multiple of 16) need the pieces' table and workspace", piece_tokens);
  if (rows == 0) return 0;
  if (piece_tokens > 0) {
    const int failed = holon_delta_scan_pieces(qn, kn, qkv, qkv_stride, v_offset, beta, g, state, out, slots, starts, query_start, rows,
                                               heads, kv_heads, dim, vdim, dtype, piece_tokens, max_pieces, piece_base, piece_of, blocks,
                                               a, sin, stream);
    if (failed || !piece_of) return failed;
  }
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid(rows, heads, (vdim + SCAN_COLS - 1) / SCAN_COLS);      // a wave for every 8 value columns
  BY_DTYPE(dtype, BY_KEY_SIZE(dim, (launch_delta<T, KD>(grid, s, qn, kn, qkv, qkv_stride, v_offset, beta, g, state, out, slots,
                                                         starts, query_start, piece_tokens > 0 ? piece_of : nullptr, heads, kv_heads,
                                                         dim, vdim))));
  HOLON_LAUNCH_OK();
  return 0;
}

template <typename T, int KD>
static void launch_memory(dim3 grid, hipStream_t s, const void* r, const void* k, const void* v,
                          const float* w, const float* u, float* state, float* out, const int32_t* slots,
                          const int32_t* starts, const int32_t* qs, int heads, int dim) {
  memory_scan_kernel<KD, T><<<grid, WAVE, 0, s>>>((const T*)r, (const T*)k, (const T*)v, w, u, state, out, slots,
                                                     starts, qs, heads, dim);
}

int holon_memory_scan_pieces(const void* q, const void* k, const void* v, const float* w, const float* u, float* state,
                             float* out, const int32_t* slots, const int32_t* starts, const int32_t* query_start, int rows,
                             int heads, int dim, int dtype, int piece_tokens, int max_pieces, const int32_t* piece_base,
                             float* sloc, float* pw, void* stream);

// Rows in pieces (the recurrence is linear in S and its decays do not depend on S): every piece but a row's last first runs
// from S = 0 and leaves what it adds and the product of its decays per key row; a walk over a row's pieces in order leaves
// each piece's true start; then every piece runs from there and writes its outputs. A layer of 32 heads of 64 over one row
// of 2,048 tokens: 17 + 7 + 38 us in blocks of 16 tokens on the float32 matrix cores, 153 + 65 + 153 token by token with S
// in registers.
extern "C" int holon_memory_scan(const void* r, const void* k, const void* v, const float* w, const float* u,
                                 float* state, float* out, const int32_t* slots, const int32_t* starts,
                                 const int32_t* query_start, int rows, int heads, int dim, int state_slots, int dtype,
                                 int piece_tokens, int max_pieces, const int32_t* piece_base, float* sloc, float* pw,
                                 void* stream) {
  HOLON_CHECK(rows >= 0 && heads > 0 && heads <= 65535 && dim > 0 && dim <= 256 && state_slots > 0,
              "memory_scan: %d heads of %d (at most 256)", heads, dim);
  HOLON_CHECK(piece_tokens == 0 || (piece_tokens > 0 && max_pieces > 0 && piece_base && sloc && pw),
              "memory_scan: rows in pieces of %d tokens need the pieces' table and workspace", piece_tokens);
  if (rows == 0) return 0;
  if (piece_tokens)
    return holon_memory_scan_pieces(r, k, v, w, u, state, out, slots, starts, query_start, rows, heads, dim, dtype, piece_tokens,
                                    max_pieces, piece_base, sloc, pw, stream);
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid(rows, heads, (dim + SCAN_COLS - 1) / SCAN_COLS);
  BY_DTYPE(dtype, BY_KEY_SIZE(dim, (launch_memory<T, KD>(grid, s, r, k, v, w, u, state, out, slots, starts,
                                                          query_start, heads, dim))));
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_gated_out(const float* o, const void* gate, const void* weight, void* y, int tokens, int heads,
                               int vdim, int per_head, float eps, int dtype, int64_t gate_stride, int plain_sigmoid,
                               const float* den, void* stream) {
  HOLON_CHECK(tokens >= 0 && heads > 0 && vdim > 0 && gate_stride >= (int64_t)heads * vdim,
              "gated_out: %d heads of %d, gates %lld apart", heads, vdim, (long long)gate_stride);
  const int64_t cells = (int64_t)tokens * heads;
  if (cells == 0) return 0;
  HOLON_CHECK((cells + 3) / 4 <= 0x7fffffff, "gated_out: %lld cells exceed one launch", (long long)cells);
  hipStream_t s = (hipStream_t)stream;
#define GATED_ROWS(LANES)                                                                                                         \
  BY_DTYPE(dtype, (gated_out_rows_kernel<T, LANES><<<(unsigned)((cells * LANES + 255) / 256), 256, 0, s>>>(                         \
                      o, (const T*)gate, (const T*)weight, (T*)y, cells, heads, per_head, eps, gate_stride, plain_sigmoid, den)))
  const bool pieces = gate_stride % 8 == 0 && head_rows::on16(o) && head_rows::on16(gate) && head_rows::on16(weight) && head_rows::on16(y);
  if (pieces && vdim == 64) GATED_ROWS(8);
  else if (pieces && vdim == 128) GATED_ROWS(16);
  else if (pieces && vdim == 256) GATED_ROWS(32);
  else
    BY_DTYPE(dtype, (gated_out_kernel<T><<<(unsigned)((cells + 3) / 4), 256, 0, s>>>(
                        o, (const T*)gate, (const T*)weight, (T*)y, cells, heads, vdim, per_head, eps, gate_stride,
                        plain_sigmoid, den)));
#undef GATED_ROWS
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_shift_mix(const void* x, const void* mu, void* state, void* y, const int32_t* slots,
                               const int32_t* starts, const int32_t* query_start, const int32_t* token_row, int tokens,
                               int rows, int width, int mixes, int state_slots, int dtype, int rows_in_order,
                               void* stream) {
  HOLON_CHECK(tokens >= 0 && rows >= 0 && width > 0 && mixes > 0 && state_slots > 0, "shift_mix: tokens=%d width=%d",
              tokens, width);
  HOLON_CHECK(tokens <= 65535 && rows <= 65535, "shift_mix: %d tokens in %d rows exceed one launch", tokens, rows);
  if (tokens == 0 || rows == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const dim3 block(256), grid_t((width + 255) / 256, tokens), grid_b((width + 255) / 256, rows);
  HOLON_CHECK(!rows_in_order || tokens == rows, "shift_mix: rows in order means one token a row, got %d in %d", tokens,
              rows);
  const int piece = dtype == HOLON_F32 ? Elem<float>::kVec : Elem<bf16_t>::kVec, per = width / piece, across = (per + 255) / 256;
  if ((int64_t)tokens * width >= (dtype == HOLON_F32 ? SHIFT_PIECES_FROM_F32 : SHIFT_PIECES_FROM) && width % piece == 0 && head_rows::on16(x) &&
      head_rows::on16(mu) && head_rows::on16(state) && head_rows::on16(y))
    BY_DTYPE(dtype, (shift_mix_rows_kernel<T><<<dim3(across, tokens), ((per + across - 1) / across + 63) / 64 * 64, 0, s>>>(
                        (const T*)x, (const T*)mu, (T*)state, (T*)y, slots, starts, query_start, token_row, tokens, width, mixes,
                        rows_in_order)));
  else
    BY_DTYPE(dtype, (shift_mix_kernel<T><<<grid_t, block, 0, s>>>((const T*)x, (const T*)mu, (T*)state, (T*)y, slots, starts,
                                                                  query_start, token_row, tokens, width, mixes,
                                                                  rows_in_order)));
  HOLON_LAUNCH_OK();
  if (rows_in_order) return 0;                           // the one kernel has kept each row's token
  BY_DTYPE(dtype, (shift_keep_kernel<T><<<grid_b, block, 0, s>>>((const T*)x, (T*)state, slots, query_start, width)));
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_decay_lora(const float* a, const void* w2t, const float* w0, float* y, int tokens, int channels,
                                int rank, int dtype, void* stream) {
  HOLON_CHECK(tokens >= 0 && channels > 0 && rank > 0 && rank <= LORA_MAX_RANK,
              "decay_lora: %d channels, rank %d (at most %d)", channels, rank, LORA_MAX_RANK);
  if (tokens == 0) return 0;
  const dim3 grid((tokens + LORA_TOKENS - 1) / LORA_TOKENS, (channels + 255) / 256);
  HOLON_CHECK(grid.y <= 65535, "decay_lora: %d channels exceed one launch", channels);
  const size_t lds = (size_t)LORA_TOKENS * lora_pitch(rank) * sizeof(float);
  hipStream_t s = (hipStream_t)stream;
  if (channels >= 4)
    BY_DTYPE(dtype, (decay_lora_kernel<true, T><<<grid, 256, lds, s>>>(a, (const T*)w2t, w0, y, tokens, channels, rank)));
  else
    BY_DTYPE(dtype, (decay_lora_kernel<false, T><<<grid, 256, lds, s>>>(a, (const T*)w2t, w0, y, tokens, channels, rank)));
  HOLON_LAUNCH_OK();
  return 0;
}
