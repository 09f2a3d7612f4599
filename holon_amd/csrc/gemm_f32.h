// What the 32-bit path's products are made of (gemm_f32.hip, moe_f32.hip): the order of their sums, and a block's 64 x 64 results.
#pragma once
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace f32_sums {
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

// The products of groups of k `first` .. `last` of NT rows of w and MT rows of x, the lane's own of each tile, added to acc in order;
// DEPTH groups of a wave are asked for at a time.
template <int MT, int NT, int DEPTH, bool VEC>
__device__ __forceinline__ void share_sums(f32x4_t (&acc)[MT][NT], const float* const (&wr)[NT], const float* const (&xr)[MT], int first,
                                           int last) {
  const int g = threadIdx.x % WAVE / 16;
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
}

// The same sums for half a tile, eight rows of w (`wr`: row lane % 8 of them): a load takes two groups of each, lanes 8 .. 15 of a row
// of lanes the second one, which then changes places with the first. Of the tile's columns the first eight are results.
template <int DEPTH, bool VEC>
__device__ __forceinline__ void half_sums(f32x4_t& acc, const float* wr, const float* xr, int first, int last) {
  const int g = threadIdx.x % WAVE / 16, second = threadIdx.x % 16 / 8;
  for (int k0 = first; k0 < last; k0 += 2 * DEPTH * GROUP) {
    f32x4_t a[DEPTH], b[DEPTH][2];
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      const int k = k0 + 2 * s * GROUP + 4 * g;
      a[s] = load4<VEC>(wr, k + GROUP * second, last);
      b[s][0] = load4<VEC>(xr, k, last);
      b[s][1] = load4<VEC>(xr, k + GROUP, last);
    }
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i], b[s][0][i], acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int other = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, (float)a[s][i]), 0x128, 0xf, 0xf, true);      // (8 lanes on)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, other), b[s][1][i], acc, 0, 0, 0);
      }
    }
  }
}

// More rows: bound by the matrix cores. A block owns 32 MT x 32 NT results; four waves (16 MT x 16 NT each) walk a run of K whose rows of x
// and w they stage in LDS, CHUNK of k at a time, into one of two buffers while the other is multiplied; pieces of 16 bytes lie at
// place p ^ (row % 8) of their row. SIDE 4: sixteen waves, the four quarters of K side by side: what fills the chip where an output of
// some hundred rows has few tiles, four waves a SIMD covering each other's barriers. SIDE 1: four waves, the quarters one after the
// other: several blocks share a unit, so that one's first loads and its stores lie under the others' products; that is the better
// one where there are tiles for it, the more the shorter K. Either ends at K (what lies behind it would add zeros).
// Whole chunks of K go from memory straight into LDS: no register holds them on their way, which leaves room for five blocks of 64 x 64 a
// unit instead of four, no instruction writes LDS, and a chunk has one barrier. Against the form that passes registers, us, weights from memory:
// 825 x 16384 x 2048 550 -> 493 (360 at the rate of a large product; in a model's trace 553 -> 526 to 562, for a reason not found), 825 x 2048 x 8192
// 304 -> 279, 2048 x 2048 x 2048 164 -> 152, 2048 x 9248 x 256 115 -> 102. What is left there is mostly the last round of blocks; 128 x 64 a
// block (three blocks a unit) takes 6 to 17 % longer, and an XCD a run of columns of its own gained nothing that a model shows.
// Every thread of the block comes here. `xr`, `wr`: the rows of either operand that the thread stages, row tid / 8 of 32 and those 32
// further on (tid: the thread within its quarter). emit(sums, row, column): four results of a row, once each, behind the block's last
// barrier over the stage.
enum How { BY_VALUE, BY_FOUR, DIRECT };                    // what a thread reads at a time; DIRECT: K is a multiple of CHUNK too
template <int SIDE, int MT, int NT>
using Stage = float[SIDE][2][32 * (MT + NT) * CHUNK];      // quarter, buffer; rows of x, then rows of w
template <int SIDE, int MT, int NT, How HOW, typename Emit>
__device__ __forceinline__ void tile_sums(Stage<SIDE, MT, NT>& stage, const float* const (&xr)[MT], const float* const (&wr)[NT], int K,
                                          Emit emit) {
  const int quarter = SIDE > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / 256) : 0, tid = threadIdx.x % 256;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int g = lane / 16, c = lane % 16;
  const int share = share_length(K), first = quarter * 4 * share, per_share = share / CHUNK;
  const int chunks = (min(K, (SIDE > 1 ? 4 : 16) * share) + CHUNK - 1) / CHUNK;      // (of the block: the first quarter's)
  // what this thread stages: piece tid % 8 of its rows
  const int r0 = tid / 8, p0 = tid % 8;
  const auto row_of = [&](int i) { return i < MT ? xr[i < MT ? i : 0] : wr[i < MT ? 0 : i - MT]; };
  f32x4_t held[MT + NT];
  auto fetch = [&](int chunk) {
    const int k = first + chunk * CHUNK + 4 * p0;
#pragma unroll
    for (int i = 0; i < MT + NT; ++i) held[i] = load4<HOW == BY_FOUR>(row_of(i), k, K);
  };
  auto keep = [&](int buf) {
#pragma unroll
    for (int i = 0; i < MT + NT; ++i)
      *reinterpret_cast<f32x4_t*>(&stage[quarter][buf][(r0 + 32 * i) * CHUNK + 4 * (p0 ^ (r0 % 8))]) = held[i];
  };
  // DIRECT: a wave's 64 lanes land in eight rows of LDS, one behind the other, so a lane asks for the piece that belongs where it lands.
  const float* from[MT + NT];
#pragma unroll
  for (int i = 0; i < MT + NT; ++i) from[i] = row_of(i) + first + 4 * (p0 ^ (r0 % 8));
  const uint32_t place = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&stage[quarter][0][wave * 8 * CHUNK];
  auto copy = [&](int chunk) {                             // (chunks in order: each moves the lane's addresses on)
    if (first + chunk * CHUNK >= K) return;                // (behind the end of K nothing is read; the same in the whole quarter)
#pragma unroll
    for (int i = 0; i < MT + NT; ++i) {
      load_to_lds16_from(from[i], place + ((chunk & 1) * (MT + NT) + i) * 32 * CHUNK * sizeof(float));
      from[i] += CHUNK;
    }
  };
  // where this lane reads: row 16 MT (half) + 16 t + c, pieces g and 4 + g
  const int xrow = wave / 2 * 16 * MT + c, wrow = 32 * MT + wave % 2 * 16 * NT + c;
  const int at[2] = {4 * (g ^ (c % 8)), 4 * ((4 + g) ^ (c % 8))};
  // the sums of a share, of a quarter's shares so far (SIDE 1), and of all that is behind them
  f32x4_t acc[MT][NT], part[SIDE > 1 ? 1 : MT][NT], total[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[t][u] = total[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int left = per_share, shares = 0;
  const auto end_share = [&]() {
    const bool begins = SIDE > 1 ? shares == 0 : shares % 4 == 0, ends = shares % 4 == 3, first_quarter = shares < 4;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u) {
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
  const auto multiply = [&](int ch) {
    if (SIDE > 1 && first + ch * CHUNK >= K) return;
    const float* rows = stage[quarter][ch & 1];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f32x4_t b[MT], a[NT];
#pragma unroll
      for (int t = 0; t < MT; ++t) b[t] = *reinterpret_cast<const f32x4_t*>(&rows[(xrow + 16 * t) * CHUNK + at[s]]);
#pragma unroll
      for (int u = 0; u < NT; ++u) a[u] = *reinterpret_cast<const f32x4_t*>(&rows[(wrow + 16 * u) * CHUNK + at[s]]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int u = 0; u < NT; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[t][i], acc[t][u], 0, 0, 0);
    }
    if (--left == 0) end_share();
  };
  if constexpr (HOW == DIRECT) {
    copy(0);
    for (int ch = 0; ch < chunks; ++ch) {
      wait_loads_but<0>();                                // (this wave's part of the chunk is there)
      lds_barrier();                                      // all of it is, and the other buffer has been read
      if (ch + 1 < chunks) copy(ch + 1);
      multiply(ch);
    }
    lds_barrier();
  } else {
    fetch(0);
    keep(0);
    if (chunks > 1) fetch(1);
    lds_barrier();
    for (int ch = 0; ch < chunks; ++ch) {
      if (ch + 1 < chunks) keep((ch + 1) & 1);            // (read last in front of the barrier behind us)
      if (ch + 2 < chunks) fetch(ch + 2);
      multiply(ch);
      lds_barrier();                                      // (what was fetched stays under way)
    }
  }
  if (left < per_share) end_share();                      // (K ends inside a share)
  if constexpr (SIDE > 1) {
    static_assert(MT == 2 && NT == 2, "a tile a wave");
    // the quarters' sums through LDS: tile (4 t' + u') of the block's 16, one a wave
    f32x4_t(*sums)[16][WAVE] = reinterpret_cast<f32x4_t(*)[16][WAVE]>(&stage[0][0][0]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) sums[quarter][(wave / 2 * 2 + t) * 4 + wave % 2 * 2 + u][lane] = total[t][u];
    __syncthreads();
    const int tile = quarter * 4 + wave;
    f32x4_t sum = sums[0][tile][lane];
#pragma unroll
    for (int q = 1; q < QUARTERS; ++q) sum += sums[q][tile][lane];
    emit(sum, tile / 4 * 16 + c, tile % 4 * 16 + 4 * g);
  } else {
    const bool pending = shares % 4 != 0, only = shares < 4;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const f32x4_t sum = pending ? (only ? part[t][u] : total[t][u] + part[t][u]) : total[t][u];
        emit(sum, (wave / 2 * MT + t) * 16 + c, (wave % 2 * NT + u) * 16 + 4 * g);
      }
  }
}
}  // namespace f32_sums
