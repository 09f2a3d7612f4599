// Which rows of a step chose which expert, and the adding up of what the experts made of them (moe_rows.hip, moe_f32.hip).
#pragma once
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace moe_lists {
constexpr int MAX_EXPERTS = 1024, MAX_TOP = 256;
constexpr int TOKEN_BITS = 22;                       // a list's entry: the row, and above it the place among the row's choices
constexpr int LIST_THREADS = 1024;

struct MoeRows {
  const float* weights;                              // [rows, stride]: 0 where a row did not choose an expert
  int stride, rows, hidden, experts, top, ff, shared, shared_col;   // shared_col < 0: the shared expert's weight is 1
  int* counts;                                       // [experts] rows that chose it
  int* lists;                                        // [experts, rows]
  int* slots;                                        // [rows, top] where a row's parts lie, -1: it made fewer choices
};

// Blocks of `experts`: an expert's list. The rest: what rows of fewer choices than `top` leave over. (No more than `top` of a
// row's weights are taken, so that the lists hold rows * top entries at most whatever the weights are.)
static __global__ void __launch_bounds__(LIST_THREADS) moe_lists_kernel(MoeRows p) {
  __shared__ int sums[LIST_THREADS / WAVE];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  if ((int)blockIdx.x >= p.experts) {
    const int t = (blockIdx.x - p.experts) * LIST_THREADS + threadIdx.x;
    if (t >= p.rows) return;
    int n = 0;
    for (int e = 0; e < p.experts; ++e) n += p.weights[(int64_t)t * p.stride + e] != 0.f;
    for (int j = n; j < p.top; ++j) p.slots[(int64_t)t * p.top + j] = -1;
    return;
  }
  const int e = blockIdx.x;
  int total = 0;
  for (int t0 = 0; t0 < p.rows; t0 += LIST_THREADS) {
    const int t = t0 + threadIdx.x;
    int place = 0;
    bool mine = t < p.rows && p.weights[(int64_t)t * p.stride + e] != 0.f;
    if (mine) {
      for (int before = 0; before < e; ++before) place += p.weights[(int64_t)t * p.stride + before] != 0.f;
      mine = place < p.top;
    }
    const uint64_t mask = __ballot(mine);
    if (lane == 0) sums[wave] = __popcll(mask);
    __syncthreads();
    int at = total, all = 0;
    for (int w = 0; w < LIST_THREADS / WAVE; ++w) {
      if (w < wave) at += sums[w];
      all += sums[w];
    }
    if (mine) p.lists[(int64_t)e * p.rows + at + __popcll(mask & ((1ull << lane) - 1))] = t | place << TOKEN_BITS;
    total += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) p.counts[e] = total;
}

struct RowTile {
  int expert, first, count, row0;                    // the expert's rows come from `first` on; this tile's from row0 of them
};

// Tiles of TILE rows of all experts together, and (tile >= 0) which expert's the given one is. Every lane of a wave calls it.
template <int TILE>
__device__ __forceinline__ int find_rows(const MoeRows& p, int tile, RowTile& out) {
  const int lane = threadIdx.x % WAVE;
  int tiles = 0, rows = 0;
  for (int e0 = 0; e0 < p.experts; e0 += WAVE) {
    const int count = e0 + lane < p.experts ? p.counts[e0 + lane] : 0;
    int t = (count + TILE - 1) / TILE, r = count;
#pragma unroll
    for (int o = 1; o < WAVE; o *= 2) {              // sums up to this lane's expert
      const int t_before = __shfl_up(t, o, WAVE), r_before = __shfl_up(r, o, WAVE);
      if (lane >= o) t += t_before, r += r_before;
    }
    if (tile >= 0) {
      const uint64_t past = __ballot(tiles + t > tile);
      if (past != 0) {
        const int at = __builtin_ctzll(past);
        out.expert = e0 + at;
        out.count = __builtin_amdgcn_readlane(count, at);
        out.first = rows + __builtin_amdgcn_readlane(r, at) - out.count;
        out.row0 = (tile - tiles - (__builtin_amdgcn_readlane(t, at) - (out.count + TILE - 1) / TILE)) * TILE;
        return 0;
      }
    }
    tiles += __builtin_amdgcn_readlane(t, WAVE - 1);
    rows += __builtin_amdgcn_readlane(r, WAVE - 1);
  }
  return tiles;
}

// hidden: a multiple of 8.
// y: a row's parts in the experts' order, the shared expert's last, rounded once. A thread 8 columns, as many loads under way
// as there are parts: 4,096 rows of 4,096 with three parts each are bound by the 235 MB that are read and written.
constexpr int ADD_AT_ONCE = 4;
template <typename T>
static __global__ void __launch_bounds__(256) moe_add_parts_kernel(const float* __restrict__ parts, T* __restrict__ y, MoeRows p) {
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (at >= (int64_t)p.rows * p.hidden) return;
  const int row = (int)(at / p.hidden), column = (int)(at % p.hidden);
  const int* slots = p.slots + (int64_t)row * p.top;
  f32x4_t sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int j0 = 0; j0 <= p.top; j0 += ADD_AT_ONCE) {
    f32x4_t part[ADD_AT_ONCE][2];
    bool have[ADD_AT_ONCE];
#pragma unroll
    for (int u = 0; u < ADD_AT_ONCE; ++u) {
      const int j = j0 + u;
      const int64_t slot = j < p.top ? slots[j] : (j == p.top && p.shared ? p.rows * (int64_t)p.top + row : -1);
      have[u] = slot >= 0;
      const float* from = parts + (have[u] ? slot : 0) * p.hidden + column;      // (some part, and not added)
      part[u][0] = *reinterpret_cast<const f32x4_t*>(from);
      part[u][1] = *reinterpret_cast<const f32x4_t*>(from + 4);
    }
#pragma unroll
    for (int u = 0; u < ADD_AT_ONCE; ++u)
      if (have[u]) sum[0] += part[u][0], sum[1] += part[u][1];
  }
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x4_t*>(y + at) = sum[0];
    *reinterpret_cast<f32x4_t*>(y + at + 4) = sum[1];
  } else {
    uint4 o;
    T* oe = reinterpret_cast<T*>(&o);
#pragma unroll
    for (int v = 0; v < 8; ++v) oe[v] = Elem<T>::store(sum[v / 4][v % 4]);
    *reinterpret_cast<uint4*>(y + at) = o;
  }
}

// The lists of a step, on a stream.
static inline void make_lists(const MoeRows& p, hipStream_t s) {
  moe_lists_kernel<<<p.experts + (p.rows + LIST_THREADS - 1) / LIST_THREADS, LIST_THREADS, 0, s>>>(p);
}
template <typename T>
static inline void add_parts(const MoeRows& p, const float* parts, T* y, hipStream_t s) {
  moe_add_parts_kernel<T><<<(unsigned)(((int64_t)p.rows * p.hidden + 2047) / 2048), 256, 0, s>>>(parts, y, p);
}
}  // namespace moe_lists
