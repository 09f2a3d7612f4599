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
#include <type_traits>

#include "common.h"
#include "holon_hip.h"

#define GEN_MAX_D 512

namespace {
constexpr int GEN_WAVES = 8;            // (at most: see by_keys)

// DB: blocks of 64 dimensions (head_dim at most 64 DB). VVEC: a page's tokens of one value dimension are whole 16-byte
// pieces on 16-byte borders.
template <typename T, int DB, int HG, bool VVEC, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE) attention_generic_kernel(
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ pages, const int32_t* __restrict__ table,
    int table_stride, const int32_t* __restrict__ slots, const int32_t* __restrict__ lens,
    const int32_t* __restrict__ query_start, int rows, int heads, int kv_heads, int head_dim, int page_size, float scale,
    int window) {
  using Acc = std::conditional_t<std::is_same<T, float>::value, double, float>;
  __shared__ Acc q_s[HG][DB * 64];
  __shared__ Acc sum_s[WAVES][HG][DB * 64];
  __shared__ Acc p_s[WAVES][HG][WAVE];
  __shared__ float ml_s[WAVES][HG][2];
  const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int t = blockIdx.x, h0 = (blockIdx.z * gridDim.y + blockIdx.y) * HG;
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
    for (int d = threadIdx.x; d < HG * head_dim; d += WAVES * WAVE) o[d] = Elem<T>::store(0.f);
    return;
  }
  const int hk = h0 / (heads / kv_heads);
  const int32_t* trow = table + (int64_t)slots[b] * table_stride;
  const int64_t plane = (int64_t)page_size * head_dim;
  const T* qp = q + ((int64_t)t * heads + h0) * head_dim;
  for (int d = threadIdx.x; d < HG * head_dim; d += WAVES * WAVE) q_s[d / head_dim][d % head_dim] = (Acc)Elem<T>::load(qp[d]);
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
  constexpr int V = Elem<T>::kVec;
  const int part = lane % 4, chunks = head_dim / V;
  for (int j0 = first + w * WAVE; j0 <= pos; j0 += WAVES * WAVE) {
    float s[HG];
#pragma unroll
    for (int h = 0; h < HG; ++h) s[h] = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = j0 + 16 * r + lane / 4;
      Acc dot[HG];
#pragma unroll
      for (int h = 0; h < HG; ++h) dot[h] = 0;
      if (key <= pos) {
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
        dot[h] += __shfl_xor(dot[h], 1, WAVE);
        dot[h] += __shfl_xor(dot[h], 2, WAVE);
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
      p_s[w][h][mine] = (Acc)p;
#pragma unroll
      for (int i = 0; i < DB; ++i) acc[h][i] *= (Acc)alpha;
    }
    const int count = min(WAVE, pos - j0 + 1);
    // (what a wave wrote to LDS it reads back behind its own wait: no other wave touches p_s[w])
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
              for (int h = 0; h < HG; ++h) acc[h][i] += p_s[w][h][j + u + x] * v;
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
          for (int h = 0; h < HG; ++h) acc[h][i] += p_s[w][h][j + u] * v;
        }
      }
      j += run;
    }
  }
#pragma unroll
  for (int h = 0; h < HG; ++h) {
#pragma unroll
    for (int i = 0; i < DB; ++i) sum_s[w][h][lane + i * WAVE] = acc[h][i];
    if (lane == 0) { ml_s[w][h][0] = m[h]; ml_s[w][h][1] = l[h]; }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < HG * head_dim; e += WAVES * WAVE) {
    const int h = e / head_dim, d = e % head_dim;
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) top = fmaxf(top, ml_s[i][h][0]);
    Acc sum = 0;
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) {
      const float f = expf(ml_s[i][h][0] - top);          // (0 for a wave without keys, whose sums are 0 too)
      den += ml_s[i][h][1] * f;
      sum += sum_s[i][h][d] * (Acc)f;
    }
    o[e] = Elem<T>::store((float)(sum / (Acc)den));
  }
}

template <typename T, int DB, int HG, int WAVES>
void launch(bool vvec, hipStream_t s, const T* q, T* out, const T* pages, const int32_t* table, int table_stride,
            const int32_t* slots, const int32_t* lens, const int32_t* query_start, int rows, int tokens, int heads,
            int kv_heads, int head_dim, int page_size, float scale, int window) {
  const int groups = heads / HG, rounds = (groups + 65534) / 65535;       // (a grid's second number has 16 bits)
  const dim3 grid(tokens, (groups + rounds - 1) / rounds, rounds);
  if (vvec)
    attention_generic_kernel<T, DB, HG, true, WAVES><<<grid, WAVES * WAVE, 0, s>>>(q, out, pages, table, table_stride, slots,
        lens, query_start, rows, heads, kv_heads, head_dim, page_size, scale, window);
  else
    attention_generic_kernel<T, DB, HG, false, WAVES><<<grid, WAVES * WAVE, 0, s>>>(q, out, pages, table, table_stride, slots,
        lens, query_start, rows, heads, kv_heads, head_dim, page_size, scale, window);
}

// `most`: no query sees more keys (0: not known). Waves without a tile are left out where there are more blocks than compute units:
// a block of eight waves of which one has keys holds registers and LDS that seven more blocks could use. 32 prompts of 64, float32,
// 8 heads of 128 on 8: 83 us (eight waves 291, a wave a head and a lane a key 230); 8 prompts of 200, 10 heads of 80 on 2 154 (273, 351);
// 32 prompts of 64, 6 heads of 48 on 2, bfloat16 29 (148, 79). With up to a block a unit the waves share the queries' load and the last
// sums: 64 rows of 60 keys, 4 heads of 256 on one, 21 us with eight waves and 25 with one.
template <typename T, int DB, int HG, typename... Args>
void by_keys(int64_t blocks, int most, Args... args) {
  if (blocks <= 256 || most <= 0 || most > 4 * WAVE) launch<T, DB, HG, GEN_WAVES>(args...);
  else if (most > 2 * WAVE) launch<T, DB, HG, 4>(args...);
  else if (most > WAVE) launch<T, DB, HG, 2>(args...);
  else launch<T, DB, HG, 1>(args...);
}

template <typename T>
void by_size(hipStream_t s, const void* q, void* out, const void* pages, const int32_t* table, int table_stride,
             const int32_t* slots, const int32_t* lens, const int32_t* query_start, int rows, int tokens, int heads,
             int kv_heads, int head_dim, int page_size, float scale, int window, int most) {
  const int group = heads / kv_heads;
  const bool vvec = page_size % Elem<T>::kVec == 0 && (uintptr_t)pages % 16 == 0;
#define GEN(DB, HG)                                                                                                    \
  by_keys<T, DB, HG>((int64_t)tokens * (heads / HG), most, vvec, s, (const T*)q, (T*)out, (const T*)pages, table,       \
                     table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim, page_size, scale, \
                     window)
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

extern "C" int holon_attention_generic(const void* q, void* out, const void* pages, const int32_t* table,
                                       int table_stride, const int32_t* slots, const int32_t* lens,
                                       const int32_t* query_start, int rows, int tokens, int heads, int kv_heads,
                                       int head_dim, int page_size, int num_pages, float scale, int window, int most,
                                       int dtype, void* stream) {
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
                   page_size, scale, window, most);
  else
    by_size<bf16_t>(s, q, out, pages, table, table_stride, slots, lens, query_start, rows, tokens, heads, kv_heads, head_dim,
                    page_size, scale, window, most);
  HOLON_LAUNCH_OK();
  return 0;
}
