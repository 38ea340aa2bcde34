// gcmf_block.hpp -- wave and block helpers shared by the HIP translation
// units: scans over a wave and a block, the ranks of a few thousand keys, and
// the stores of a read-back's values into the mapped staging buffer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gcmf {

template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = __lane_id();
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    T u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// Block-wide exclusive scan of one value per thread; returns the block total.
template <typename T>
__device__ __forceinline__ T block_excl_scan(T v, T *lds_waves, T &total) {
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
  T inc = wave_incl_scan(v);
  if (lane == 63) lds_waves[wave] = inc;
  __syncthreads();
  T wbase = 0, tot = 0;
  const int nw = blockDim.x >> 6;
  for (int w = 0; w < nw; w++) {
    T s = lds_waves[w];
    if (w < wave) wbase += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return wbase + inc - v;
}

// value j of a read-back (the last one the look-back error word)
__device__ __forceinline__ void put_slots(long long *slots, const long long *v, int n,
                                          const long long *lbErr) {
  if (!slots) return;
  for (int j = 0; j < n; j++) slots[j] = v[j];
  slots[n] = lbErr ? *lbErr : 0;
}

// The place of each of n <= kRankSort keys (keyAt(j)) in their stable order, by
// counting the keys before it: a block takes
// kRankKeys keys and compares them with all n, which it holds in LDS: four
// lanes per key, each with two keys of a 16-byte read, the reads shared out
// over the waves.  The n^2 compares are so spread over the chip; the radix
// passes of one block that did this before are a chain of about 5 us each.
// 4000 keys of 54 bits on one MI355X: 35 us in passes, 6 this way (15
// with the keys read through scalar loads, 29 with lanes read out one by one,
// a block per 64 keys).  Returns key blockIdx.x * kRankKeys + threadIdx.x's
// place in the first kRankKeys threads.
constexpr int kRankSort = 8192;
constexpr int kRankThreads = 1024;
constexpr int kRankKeys = 16;

struct RankLds {
  ulonglong2 keys[kRankSort / 2];
  int cnt[kRankThreads / 64][kRankKeys];
};

template <typename F>
__device__ __forceinline__ int rank_among(int n, RankLds &l, F keyAt) {
  constexpr int W = kRankThreads / 64;
  const int lane = __lane_id(), w = threadIdx.x >> 6;
  const int T = (n + 7) / 8;  // groups of eight keys, one read of a wave each
  uint64_t *k = (uint64_t *)l.keys;
  for (int j = threadIdx.x; j < 8 * T; j += kRankThreads)
    k[j] = j < n ? keyAt(j) : ~0ULL;  // past the end: after every key
  __syncthreads();
  const int i0 = (int)blockIdx.x * kRankKeys, i = i0 + (lane & (kRankKeys - 1));
  const uint64_t ki = i < n ? k[i] : 0;
  const ulonglong2 *mine = l.keys + (lane >> 4);
  const int own0 = i0 / 8, own1 = min(own0 + kRankKeys / 8, T);
  int c = 0, t = w;
#pragma unroll 4
  for (; t < own0; t += W) {  // an equal key before it counts
    const ulonglong2 q = mine[4 * t];
    c += (q.x <= ki) + (q.y <= ki);
  }
  for (; t < own1; t += W) {
    const ulonglong2 q = mine[4 * t];
    const int j = 8 * t + 2 * (lane >> 4);
    c += (q.x < ki || (q.x == ki && j < i)) + (q.y < ki || (q.y == ki && j + 1 < i));
  }
#pragma unroll 4
  for (; t < T; t += W) {
    const ulonglong2 q = mine[4 * t];
    c += (q.x < ki) + (q.y < ki);
  }
  c += __shfl_xor(c, 16, 64);
  c += __shfl_xor(c, 32, 64);
  if (lane < kRankKeys) l.cnt[w][lane] = c;
  __syncthreads();
  int s = 0;
  if (threadIdx.x < kRankKeys)
    for (int x = 0; x < W; x++) s += l.cnt[x][threadIdx.x];
  return s;
}

}  // namespace gcmf
