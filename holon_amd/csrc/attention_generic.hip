// Paged causal attention, the general kernel: any element type, any page size, any head_dim that is a multiple of 8.
// A block takes a query token and HG query heads that read one kv head. Keys are visited in tiles of 64 starting at the
// first visible key, wave w of the block's eight taking tiles w, w + 8, ..., and the waves are combined in order at the
// end: the order of every sum depends on the token's position alone, never on how the batch was cut. (Where blocks are
// many and no row has keys for eight tiles, a block has as many waves as there are: those left out would add zeros.) Scores and softmax
// are float32. For float32 operands the two long sums (a score over head_dim, the values over the keys) are accumulated
// in float64, which this GPU does at the float32 rate: a float32 running sum over 256 products of a sharp query and key
// is off by 1e-4 of the score, and that shows in the weights of the softmax.
//
// Bound by the latency of its loads. Four lanes share a key (16 keys of a tile at a time, 16 bytes a lane, so that a
// load takes whole 64-byte parts of 16 rows), a lane holds the weight of key 16 (lane % 4) + lane / 4 of the tile, and a
// value column is read in 16-byte pieces of neighbouring tokens where the pages allow. Heads of a group share what is
// read. One row in float32 over 16 heads of 128 on 4 at some 400 keys (and the prompts of 150, averaged): 47 us;
// with a wave a head, a lane a key and a value column read token by token 175.
//
// Steps of a few decode rows have fewer blocks than compute units, each reading all of a row's keys through one of them. There every wave is
// a block (SPLIT) with the registers of a whole unit to itself, so that a tile's loads are all under way at once, and a second kernel does
// what the waves did together, bit for bit. Three rows over 160 to 410 keys, float32, 16 heads of 128 on 4: 31.2 us as blocks of eight waves,
// 24.9 + 4.6 split, 16.3 + 4.7 with the loads asked for at once.
#include <type_traits>

#include "common.h"
#include "holon_hip.h"

#define GEN_MAX_D 512

namespace {
constexpr int GEN_WAVES = 8;            // (at most: see by_keys)
template <typename T> using Sums = std::conditional_t<std::is_same<T, float>::value, double, float>;      // what the long sums are formed in

// DB: blocks of 64 dimensions (head_dim at most 64 DB). VVEC: a page's tokens of one value dimension are whole 16-byte
// pieces on 16-byte borders.
// SPLIT: the block is one wave of a token's (blockIdx.x: token, wave), and what the waves exchange at the end goes to memory, `part_o`
// [tokens, heads, WAVES, head_dim] and `part_ml` [.., 2], for `attention_generic_merge_kernel`.
template <typename T, int DB, int HG, bool VVEC, int WAVES, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? WAVE : WAVES * WAVE) attention_generic_kernel(
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ pages, const int32_t* __restrict__ table,
    int table_stride, const int32_t* __restrict__ slots, const int32_t* __restrict__ lens,
    const int32_t* __restrict__ query_start, int rows, int heads, int kv_heads, int head_dim, int page_size, float scale,
    int window, Sums<T>* __restrict__ part_o, float* __restrict__ part_ml) {
  using Acc = Sums<T>;
  constexpr int HERE = SPLIT ? 1 : WAVES, THREADS = HERE * WAVE;
  __shared__ Acc q_s[HG][DB * 64];
  __shared__ Acc sum_s[HERE][HG][SPLIT ? 1 : DB * 64];
  __shared__ Acc p_s[HERE][HG][WAVE];
  __shared__ float ml_s[HERE][HG][2];
  const int local = threadIdx.x / WAVE, w = SPLIT ? blockIdx.x % WAVES : local, lane = threadIdx.x % WAVE;
  const int t = SPLIT ? blockIdx.x / WAVES : blockIdx.x, h0 = (blockIdx.z * gridDim.y + blockIdx.y) * HG;
  if (h0 >= heads) return;                                // (uniform over the block: the last of a second round of heads)
  // the row of token t: the last b with query_start[b] <= t
  int lo_b = 0, hi_b = rows - 1;
  while (lo_b < hi_b) {
    const int mid = (lo_b + hi_b + 1) / 2;
    if (query_start[mid] <= t) lo_b = mid; else hi_b = mid - 1;
  }
  const int b = lo_b;
  const int n = lens[b];
  const int nq = query_start[b + 1] - query_start[b];
  const int pos = n - nq + (t - query_start[b]);
  T* o = out + ((int64_t)t * heads + h0) * head_dim;      // (HG heads side by side)
  if (n <= 0 || pos < 0) {   // uniform over the block (one token per block)
    if constexpr (SPLIT) {   // (a largest score of +inf over no weights, which no sum leaves: zeros)
      if (lane < HG) {
        float* ml = part_ml + (((int64_t)t * heads + h0 + lane) * WAVES + w) * 2;
        ml[0] = INFINITY;
        ml[1] = 0.f;
      }
      return;
    }
    for (int d = threadIdx.x; d < HG * head_dim; d += THREADS) o[d] = Elem<T>::store(0.f);
    return;
  }
  const int hk = h0 / (heads / kv_heads);
  const int32_t* trow = table + (int64_t)slots[b] * table_stride;
  const int64_t plane = (int64_t)page_size * head_dim;
  const T* qp = q + ((int64_t)t * heads + h0) * head_dim;
  for (int d = threadIdx.x; d < HG * head_dim; d += THREADS) q_s[d / head_dim][d % head_dim] = (Acc)Elem<T>::load(qp[d]);
  __syncthreads();

  const int first = max(0, first_seen(pos, window));
  float m[HG], l[HG];
  Acc acc[HG][DB];
#pragma unroll
  for (int h = 0; h < HG; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < DB; ++i) acc[h][i] = 0;
  }
  constexpr int V = Elem<T>::kVec, PIECES = DB * 16 / V, AHEAD = PIECES <= 8 ? 4 : (PIECES <= 16 ? 2 : 1);
  const int part = lane % 4, chunks = head_dim / V;
  const auto ask_values = [&](auto& raw, int j0) {          // of a tile, V neighbouring tokens a piece (j0 is a multiple of V)
#pragma unroll
    for (int u = 0; u < WAVE / V; ++u) {
      const int key = min(j0 + u * V, pos - pos % V);
      const T* vp = pages + (((int64_t)trow[key / page_size] * 2 + 1) * kv_heads + hk) * plane + key % page_size;
#pragma unroll
      for (int i = 0; i < DB; ++i) raw[u][i] = *reinterpret_cast<const uint4*>(vp + (int64_t)min(lane + i * WAVE, head_dim - 1) * page_size);
    }
  };
  for (int j0 = first + w * WAVE; j0 <= pos; j0 += WAVES * WAVE) {
    float s[HG];
#pragma unroll
    for (int h = 0; h < HG; ++h) s[h] = -INFINITY;
    // A wave by itself: nothing covers its loads, so a tile's keys are asked for at once (as many as registers hold), and its values in front
    // of the scores' arithmetic. Keys past the token's are read from its own.
    uint4 kraw[SPLIT ? AHEAD : 1][PIECES];
    constexpr bool VALUES = SPLIT && VVEC && WAVE / V * DB <= 32;
    uint4 vraw[VALUES ? WAVE / V : 1][DB];
    const bool ahead = VALUES && j0 % V == 0;               // (a value's piece of neighbouring tokens then lies inside a page)
    const auto ask_keys = [&](int r0) {
#pragma unroll
      for (int r = 0; r < AHEAD; ++r) {
        const int key = min(j0 + 16 * (r0 + r) + lane / 4, pos);
        const T* kp = pages + (((int64_t)trow[key / page_size] * 2) * kv_heads + hk) * plane + (int64_t)(key % page_size) * head_dim;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) kraw[r][i] = *reinterpret_cast<const uint4*>(kp + min(part + 4 * i, chunks - 1) * V);
      }
    };
    if constexpr (SPLIT) {
      ask_keys(0);
      if constexpr (VALUES) {
        if (ahead) ask_values(vraw, j0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = j0 + 16 * r + lane / 4;
      Acc dot[HG];
#pragma unroll
      for (int h = 0; h < HG; ++h) dot[h] = 0;
      if constexpr (SPLIT) {
        if (AHEAD < 4 && r > 0 && r % AHEAD == 0) ask_keys(r);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
          const int c = part + 4 * i;
          if (c >= chunks) break;
          const T* e = reinterpret_cast<const T*>(&kraw[r % AHEAD][i]);
#pragma unroll
          for (int x = 0; x < V; ++x) {
            const Acc k = (Acc)Elem<T>::load(e[x]);
#pragma unroll
            for (int h = 0; h < HG; ++h) dot[h] += q_s[h][c * V + x] * k;
          }
        }
      } else if (key <= pos) {
        const int page = trow[key / page_size], off = key % page_size;
        const T* kp = pages + (((int64_t)page * 2 + 0) * kv_heads + hk) * plane + (int64_t)off * head_dim;
#pragma unroll 4
        for (int c = part; c < chunks; c += 4) {
          const uint4 raw = *reinterpret_cast<const uint4*>(kp + c * V);
          const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
          for (int i = 0; i < V; ++i) {
            const Acc k = (Acc)Elem<T>::load(e[i]);
#pragma unroll
            for (int h = 0; h < HG; ++h) dot[h] += q_s[h][c * V + i] * k;
          }
        }
      }
#pragma unroll
      for (int h = 0; h < HG; ++h) {
        dot[h] += lane_xor<1>(dot[h]);
        dot[h] += lane_xor<2>(dot[h]);
        if (r == part && key <= pos) s[h] = (float)dot[h] * scale;
      }
    }
    const int mine = 16 * part + lane / 4;                // the tile's key whose weight this lane holds
#pragma unroll
    for (int h = 0; h < HG; ++h) {
      const float m_new = fmaxf(m[h], wave_max(s[h]));
      const float at = m_new == -INFINITY ? 0.f : m_new;  // (scores of -inf weigh 0, one that is NaN stays one)
      const float alpha = expf(m[h] - at);                // m = -inf on the first tile: alpha = 0
      const float p = j0 + mine <= pos ? expf(s[h] - at) : 0.f;
      l[h] = l[h] * alpha + wave_sum(p);
      m[h] = m_new;
      p_s[local][h][mine] = (Acc)p;
#pragma unroll
      for (int i = 0; i < DB; ++i) acc[h][i] *= (Acc)alpha;
    }
    const int count = min(WAVE, pos - j0 + 1);
    if constexpr (VALUES) {
      if (ahead) {
#pragma unroll
        for (int u = 0; u < WAVE / V; ++u) {
          if (u * V >= count) break;
#pragma unroll
          for (int i = 0; i < DB; ++i) {
            const T* e = reinterpret_cast<const T*>(&vraw[u][i]);
#pragma unroll
            for (int x = 0; x < V; ++x) {                    // (what lies behind the token may be anything: it weighs 0)
              const Acc v = u * V + x < count ? (Acc)Elem<T>::load(e[x]) : (Acc)0;
#pragma unroll
              for (int h = 0; h < HG; ++h) acc[h][i] += p_s[local][h][u * V + x] * v;
            }
          }
        }
        continue;
      }
    }
    // (what a wave wrote to LDS it reads back behind its own wait: no other wave touches p_s[local])
    for (int j = 0; j < count;) {
      const int key = j0 + j, off = key % page_size;
      const int run = min(count - j, page_size - off);    // keys of one page
      const T* vp = pages + (((int64_t)trow[key / page_size] * 2 + 1) * kv_heads + hk) * plane + off;
      int u = 0;
      if (VVEC && off % V == 0) {
#pragma unroll 4
        for (; u + V <= run; u += V) {
#pragma unroll
          for (int i = 0; i < DB; ++i) {
            const int d = lane + i * WAVE;
            if (d >= head_dim) break;
            const uint4 raw = *reinterpret_cast<const uint4*>(vp + (int64_t)d * page_size + u);
            const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
            for (int x = 0; x < V; ++x) {
              const Acc v = (Acc)Elem<T>::load(e[x]);
#pragma unroll
              for (int h = 0; h < HG; ++h) acc[h][i] += p_s[local][h][j + u + x] * v;
            }
          }
        }
      }
      for (; u < run; ++u) {
#pragma unroll
        for (int i = 0; i < DB; ++i) {
          const int d = lane + i * WAVE;
          if (d >= head_dim) break;
          const Acc v = (Acc)Elem<T>::load(vp[(int64_t)d * page_size + u]);
#pragma unroll
          for (int h = 0; h < HG; ++h) acc[h][i] += p_s[local][h][j + u] * v;
        }
      }
      j += run;
    }
  }
  if constexpr (SPLIT) {
#pragma unroll
    for (int h = 0; h < HG; ++h) {
      const int64_t cell = ((int64_t)t * heads + h0 + h) * WAVES + w;
#pragma unroll
      for (int i = 0; i < DB; ++i)
        if (lane + i * WAVE < head_dim) part_o[cell * head_dim + lane + i * WAVE] = acc[h][i];
      if (lane == 0) { part_ml[cell * 2] = m[h]; part_ml[cell * 2 + 1] = l[h]; }
    }
    return;
  }
#pragma unroll
  for (int h = 0; h < HG; ++h) {
#pragma unroll
    for (int i = 0; i < DB; ++i) sum_s[w][h][lane + i * WAVE] = acc[h][i];
    if (lane == 0) { ml_s[w][h][0] = m[h]; ml_s[w][h][1] = l[h]; }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < HG * head_dim; e += THREADS) {
    const int h = e / head_dim, d = e % head_dim;
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) top = fmaxf(top, ml_s[i][h][0]);
    Acc sum = 0;
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) {
      const float f = expf(ml_s[i][h][0] - top);          // (0 for a wave without keys, whose sums are 0 too)
      den = fmaf(ml_s[i][h][1], f, den);
      sum = fma(sum_s[i][h][d], (Acc)f, sum);
    }
    o[e] = Elem<T>::store((float)(sum / (Acc)den));
  }
}

// What the waves of a block do at its end, from their sums in memory: the same operations in the same order.
template <typename T, int WAVES>
__global__ void __launch_bounds__(GEN_MAX_D) attention_generic_merge_kernel(const Sums<T>* __restrict__ part, const float* __restrict__ part_ml,
                                                                            T* __restrict__ out, int heads, int head_dim) {
  const int64_t cell = ((int64_t)blockIdx.x * heads + blockIdx.y) * WAVES;
  const int d = threadIdx.x;
  float m[WAVES], l[WAVES], top = -INFINITY, den = 0.f;
  Sums<T> o[WAVES], sum = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    m[i] = part_ml[(cell + i) * 2];
    l[i] = part_ml[(cell + i) * 2 + 1];
    o[i] = part[(cell + i) * head_dim + d];
  }
  T* to = out + ((int64_t)blockIdx.x * heads + blockIdx.y) * head_dim + d;
  if (m[0] == INFINITY && l[0] == 0.f) {
    *to = Elem<T>::store(0.f);
    return;
  }
#pragma unroll
  for (int i = 0; i < WAVES; ++i) top = fmaxf(top, m[i]);
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const float f = expf(m[i] - top);
    den = fmaf(l[i], f, den);
    sum = fma(o[i], (Sums<T>)f, sum);
  }
  *to = Elem<T>::store((float)(sum / (Sums<T>)den));
}

template <typename T, int DB, int HG, int WAVES>
void launch(bool vvec, hipStream_t s, const T* q, T* out, const T* pages, const int32_t* table, int table_stride,
            const int32_t* slots, const int32_t* lens, const int32_t* query_start, int rows, int tokens, int heads,
            int kv_heads, int head_dim, int page_size, float scale, int window, Sums<T>* part, float* part_ml) {
  const int groups = heads / HG, rounds = (groups + 65534) / 65535;       // (a grid's second number has 16 bits)
  const bool split = part != nullptr;
  const dim3 grid(split ? tokens * WAVES : tokens, (groups + rounds - 1) / rounds, rounds);
#define GEN_LAUNCH(VVEC, SPLIT)                                                                                                   \
  attention_generic_kernel<T, DB, HG, VVEC, WAVES, SPLIT><<<grid, SPLIT ? WAVE : WAVES * WAVE, 0, s>>>(                           \
      q, out, pages, table, table_stride, slots, lens, query_start, rows, heads, kv_heads, head_dim, page_size, scale, window, part, part_ml)
  if constexpr (WAVES == GEN_WAVES) {
    if (split) {
      if (vvec) GEN_LAUNCH(true, true);
      else GEN_LAUNCH(false, true);
      attention_generic_merge_kernel<T, WAVES><<<dim3(tokens, heads), head_dim, 0, s>>>(part, part_ml, out, heads, head_dim);
      return;
    }
  }
  if (vvec) GEN_LAUNCH(true, false);
  else GEN_LAUNCH(false, false);
#undef GEN_LAUNCH
}

// `most`: no query sees more keys (0: not known). Waves without a tile are left out where there are more blocks than compute units:
// a block of eight waves of which one has keys holds registers and LDS that seven more blocks could use. 32 prompts of 64, float32,
// 8 heads of 128 on 8: 83 us (eight waves 291, a wave a head and a lane a key 230); 8 prompts of 200, 10 heads of 80 on 2 154 (273, 351);
// 32 prompts of 64, 6 heads of 48 on 2, bfloat16 29 (148, 79). With up to a block a unit the waves share the queries' load and the last
// sums: 64 rows of 60 keys, 4 heads of 256 on one, 21 us with eight waves and 25 with one.
// (`whole`: all eight waves, whatever the keys: a call that splits them.)
template <typename T, int DB, int HG, typename... Args>
void by_keys(bool whole, int64_t blocks, int most, Args... args) {
  if (whole || blocks <= 256 || most <= 0 || most > 4 * WAVE) launch<T, DB, HG, GEN_WAVES>(args...);
  else if (most > 2 * WAVE) launch<T, DB, HG, 4>(args...);
  else if (most > WAVE) launch<T, DB, HG, 2>(args...);
  else launch<T, DB, HG, 1>(args...);
}

template <typename T>
void by_size(hipStream_t s, const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
             const int32_t* slots, const int32_t* lens, const int32_t* query_start, int rows, int tokens, int heads,
             int kv_heads, int head_dim, int page_size, float scale, int window, int most, void* part, float* part_ml) {
  const int group = heads / kv_heads;
  const bool vvec = page_size % Elem<T>::kVec == 0 && (uintptr_t)pages % 16 == 0;
#define GEN(DB, HG)                                                                                                    \
  by_keys<T, DB, HG>(part != nullptr, (int64_t)tokens * (heads / HG), most, vvec, s, (const T*)q, (T*)out, (const T*)pages, table,       \
                     table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim, page_size, scale, \
                     window, (Sums<T>*)part, part_ml)
#define GEN_HEADS(DB)                  \
  do {                                 \
    if (group % 4 == 0) GEN(DB, 4);    \
    else if (group % 2 == 0) GEN(DB, 2); \
    else GEN(DB, 1);                   \
  } while (0)
  if (head_dim <= 64) GEN_HEADS(1);
  else if (head_dim <= 128) GEN_HEADS(2);
  else if (head_dim <= 256) GEN_HEADS(4);
  else GEN(8, 1);
#undef GEN_HEADS
#undef GEN
}
}  // namespace

static int generic_launch(const void* q, void* out, const void* pages, const int32_t* table,
                                       int table_stride, const int32_t* slots, const int32_t* lens,
                                       const int32_t* query_start, int rows, int tokens, int heads, int kv_heads,
                                       int head_dim, int page_size, int num_pages, float scale, int window, int most,
                                       int dtype, void* part, float* part_ml, void* stream) {
  HOLON_CHECK(rows >= 0 && tokens >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
              "attention: bad head counts %d/%d", heads, kv_heads);
  HOLON_CHECK(head_dim > 0 && head_dim % 8 == 0 && head_dim <= GEN_MAX_D,
              "attention: head_dim %d must be a multiple of 8, at most %d", head_dim, GEN_MAX_D);
  HOLON_CHECK(page_size > 0 && num_pages > 0 && window > -0x7fffffff, "attention: bad page size or window");
  if (tokens == 0 || rows == 0) return 0;
  const int seen = window < 0 ? -window : window;          // (a query sees no more keys than its window holds)
  if (seen > 0 && (most <= 0 || most > seen)) most = seen;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HOLON_F32)
    by_size<float>(s, q, out, pages, table, table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim,
                   page_size, scale, window, most, part, part_ml);
  else
    by_size<bf16_t>(s, q, out, pages, table, table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim,
                    page_size, scale, window, most, part, part_ml);
  HOLON_LAUNCH_OK();
  return 0;
}

extern "C" int holon_attention_generic(const void* q, void* out, const void* pages, const int32_t* table,
                                       int table_stride, const int32_t* slots, const int32_t* lens,
                                       const int32_t* query_start, int rows, int tokens, int heads, int kv_heads,
                                       int head_dim, int page_size, int num_pages, float scale, int window, int most,
                                       int dtype, void* stream) {
  return generic_launch(q, out, pages, table, table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim, page_size,
                        num_pages, scale, window, most, dtype, nullptr, nullptr, stream);
}

// The same bits with every wave of a block in a block of its own and a second kernel behind them: part [tokens, heads, 8, head_dim]
// (float64 for float32 operands, else float32), part_ml [tokens, heads, 8, 2] float32.
extern "C" int holon_attention_generic_split(const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
                                             const int32_t* slots, const int32_t* lens, const int32_t* query_start, int rows, int tokens,
                                             int heads, int kv_heads, int head_dim, int page_size, int num_pages, float scale, int window,
                                             int most, int dtype, void* part, float* part_ml, void* stream) {
  HOLON_CHECK(part != nullptr && part_ml != nullptr && heads <= 65535 && tokens <= 1 << 26, "attention: no room for the waves' sums");
  return generic_launch(q, out, pages, table, table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim, page_size,
                        num_pages, scale, window, most, dtype, part, part_ml, stream);
}
