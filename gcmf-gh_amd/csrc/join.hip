// join.hip -- the GCMF filter-and-refine spatial join on gfx950.
//
// Stages (reference semantics in brackets):
//   1. MBR filter as sort-and-sweep [Join.h:5-153, GPU_MBR.h:339-539]: the
//      2(B+O) x-endpoint keys (mod 1e16, the reference sorts 16 decimal
//      digits) are radix sorted with the endpoint index as a stable
//      tie-break; each polygon then scans the contiguous rank range between
//      its own two endpoints in a structure-of-arrays record stream
//      (endpoint id, partner y-interval), one wave64 per polygon, ballots
//      for counting and ordered output.
//   2. CMBR + PiP candidate flags [Join.h:397-432, GPU_Join.h:461-508],
//   3. PiP "within" refine, crossing parity from ballot popcounts
//      [Join.h:437-467, GPU_Join.h:839-943],
//   4. CMF edge filter, ordered edge lists from ballot ranks
//      [Join.h:157-287, GPU_Join.h:511-735],
//   5. Segment-intersection refine with a uniform early exit
//      [Join.h:356-393, GPU_Join.h:326-456]: two fused passes over the
//      candidates, one group of 8, 16 or 64 lanes each; as kernels of their
//      own for the entry points that run one stage.
#include <algorithm>
#include <vector>

#include "gcmf_block.hpp"
#include "gcmf_device.hpp"
#include "gcmf_internal.hpp"
#include "gcmf_join.hpp"

namespace gcmf {

constexpr uint64_t kKeyMod = 10000000000000000ULL;  // 16 decimal digits

// ------------------------------------------------------------ stage 1 ----
// mm: x key min, x key max, y key min, y key max (over both corners), when
// the vertex counts are given their sum, and the height class of the y strips
constexpr int kMmVals = 6;
constexpr unsigned kEndpointBlocks = 1024;
constexpr int kStripSample = 1024;

struct MinMax {
  uint64_t v[5];
};
__device__ __forceinline__ MinMax mm_none() { return MinMax{{~0ULL, 0, ~0ULL, 0, 0}}; }
__device__ __forceinline__ void mm_merge(MinMax &a, const MinMax &b) {
  a.v[0] = min(a.v[0], b.v[0]);
  a.v[1] = max(a.v[1], b.v[1]);
  a.v[2] = min(a.v[2], b.v[2]);
  a.v[3] = max(a.v[3], b.v[3]);
  a.v[4] += b.v[4];
}
// of the whole block, in thread 0 (lds: one per wave)
__device__ __forceinline__ void mm_block(MinMax &a, MinMax *lds) {
  for (int off = 32; off > 0; off >>= 1) {
    MinMax o;
#pragma unroll
    for (int j = 0; j < 5; j++) o.v[j] = __shfl_xor(a.v[j], off, 64);
    mm_merge(a, o);
  }
  if (__lane_id() == 0) lds[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) mm_merge(a, lds[w]);
}

// Keys, ids and y values of every endpoint; each block's minima and maxima
// go to part (bound by that reduction when it was five atomics per block on
// one cache line: 66 us for 550 000 polygons on one MI355X, against 8 us of
// loads and stores; 13 us this way).
__global__ void __launch_bounds__(256)
    k_endpoints(long B, long O, const uint64_t *bMBR, const uint64_t *oMBR, const int *bVNum,
                const int *oVNum, uint64_t *keys, int *idx, uint64_t *Y, MinMax *part) {
  __shared__ MinMax lds[4];
  MinMax a = mm_none();
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < B + O;
       e += (long)gridDim.x * blockDim.x) {
    const uint64_t *m = e < B ? bMBR + 4 * e : oMBR + 4 * (e - B);
    const uint64_t x1 = m[0] % kKeyMod, x2 = m[2] % kKeyMod, y1 = m[1], y2 = m[3];
    keys[2 * e] = x1;
    keys[2 * e + 1] = x2;
    idx[2 * e] = (int)(2 * e);
    idx[2 * e + 1] = (int)(2 * e + 1);
    Y[2 * e] = y1;
    Y[2 * e + 1] = y2;
    mm_merge(a, MinMax{{min(x1, x2), max(x1, x2), min(y1, y2), max(y1, y2),
                        bVNum ? (uint64_t)(e < B ? bVNum[e] : oVNum[e - B]) : 0}});
  }
  mm_block(a, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = a;
}

// The blocks' minima and maxima combined, and the class of the median MBR
// height of ns sampled polygons (j N / ns, j < ns): the power of two at or
// above twice a height.  The class never decreases with the height, so the
// median's class is the classes' median, found from their histogram.  One
// block of kStripSample threads; the values also go to slots.
__global__ void __launch_bounds__(kStripSample)
    k_minmax_final(const MinMax *part, int nPart, long N, const uint64_t *Y, int ns,
                   long long *mm, long long *slots, const long long *lbErr) {
  __shared__ MinMax lds[kStripSample / 64];
  __shared__ int hist[66];
  if (threadIdx.x < 66) hist[threadIdx.x] = 0;
  __syncthreads();
  const int j = threadIdx.x;
  if (j < ns) {
    const long e = (long)((long long)j * N / ns);
    const uint64_t a = Y[2 * e], b = Y[2 * e + 1], h = a > b ? a - b : b - a;
    atomicAdd(&hist[h == 0 ? 0 : h == 1 ? 1 : 65 - __clzll(h - 1)], 1);
  }
  MinMax a = mm_none();
  for (int i = j; i < nPart; i += kStripSample) mm_merge(a, part[i]);
  mm_block(a, lds);
  __syncthreads();
  if (threadIdx.x != 0) return;
  int cls = 0;
  for (int c = hist[0]; cls < 65 && c <= ns / 2; c += hist[cls]) cls++;
  long long v[kMmVals];
  for (int k = 0; k < 5; k++) v[k] = (long long)a.v[k];
  v[5] = cls;
  for (int k = 0; k < kMmVals; k++) mm[k] = v[k];
  put_slots(slots, v, kMmVals, lbErr);
}

__global__ void k_sub_key(uint64_t *keys, long n, const long long *mn) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) keys[i] -= (uint64_t)*mn;
}

// The sorted endpoint stream: endpoint ids and, for left endpoints (the only
// ones a polygon takes as a candidate), the polygon's y interval; as arrays
// for the sweep, whose lanes read consecutive ranks, or as one record a rank
// for the strips, whose lanes read ranks far apart.
struct SweepRec {
  int id;
  uint64_t y1, y2;
};
struct SweepRecs {
  int *id = nullptr;
  uint64_t *ylo = nullptr, *yhi = nullptr;
  SweepRec *aos = nullptr;
};

struct Strips {
  uint64_t y0;
  int shift, S;
};
__device__ __forceinline__ int strip_of(const Strips &g, uint64_t y) {
  const uint64_t s = (y - g.y0) >> g.shift;
  return s >= (uint64_t)g.S ? g.S - 1 : (int)s;
}

// rank[perm[i]] = i and the stream's record at rank i; with strips also
// cnt[i], the number of strips the record is listed in
__global__ void __launch_bounds__(256)
    k_sweep_prep(const int *perm, long n, const uint64_t *Y, int *rank, SweepRecs r, Strips g,
                 int *cnt) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int e = perm[i];
  rank[e] = (int)i;
  const bool left = !(e & 1);
  const uint64_t a = left ? Y[e] : 0, b = left ? Y[e + 1] : 0;
  if (r.aos) {
    r.aos[i] = SweepRec{e, a, b};
    cnt[i] = left ? strip_of(g, a < b ? b : a) - strip_of(g, a < b ? a : b) + 1 : 0;
    return;
  }
  r.id[i] = e;
  if (left) {
    r.ylo[i] = a;
    r.yhi[i] = b;
  }
}

// The order of at most kRankSort endpoints: their places among all keys, and
// with them the ranks and records, in one launch and without the read-back
// of the keys' range that the radix passes need.  Every block makes all keys
// itself (a few per thread).
__global__ void __launch_bounds__(kRankThreads)
    k_order_few(int B, int O, const uint64_t *bMBR, const uint64_t *oMBR, uint64_t *Y, int *perm,
                int *rank, SweepRecs rec) {
  __shared__ RankLds lds;
  const int n = 2 * (B + O);
  auto mbr_of = [&](int e) { return e < B ? bMBR + 4L * e : oMBR + 4L * (e - B); };
  const int i = rank_among(n, lds, [&](int j) { return mbr_of(j >> 1)[2 * (j & 1)] % kKeyMod; });
  const int e = (int)blockIdx.x * kRankKeys + (int)threadIdx.x;
  if (threadIdx.x >= kRankKeys || e >= n) return;
  const uint64_t *m = mbr_of(e >> 1);
  perm[i] = e;
  rank[e] = i;
  rec.id[i] = e;
  Y[e] = m[2 * (e & 1) + 1];
  if (e & 1) return;
  rec.ylo[i] = m[1];
  rec.yhi[i] = m[3];
}

// One wave walks polygon e's rank range: the number of candidates, or with
// WRITE the candidates to pairs[pos..] (those below cap).  Bound by the loop's
// own steps on long ranges, most of which hold no candidate: 10 polygons under
// 30 000 take 410 us a pass, 527 with a place worked out for every step.
template <bool AOS, bool WRITE>
__device__ __forceinline__ int sweep_polygon(long e, long B, const int *rank, const SweepRecs &r,
                                             const uint64_t *Y, long long pos, int *pairs,
                                             long long cap) {
  const int lane = __lane_id();
  const int lo = rank[2 * e], hi = rank[2 * e + 1];
  const uint64_t ey1 = Y[2 * e], ey2 = Y[2 * e + 1];
  const bool overlay = e >= B;
  const int lim = (int)(2 * B);
  int cnt = 0;
  for (int i0 = lo + 1; i0 < hi; i0 += 64) {
    int i = i0 + lane;
    bool ok = false;
    int m = 0;
    if (i < hi) {
      m = AOS ? r.aos[i].id : r.id[i];
      bool other = overlay ? (m < lim) : (m >= lim);
      ok = other && !(m & 1) && !(ey1 > (AOS ? r.aos[i].y2 : r.yhi[i])) &&
           !((AOS ? r.aos[i].y1 : r.ylo[i]) > ey2);
    }
    const unsigned long long msk = __ballot(ok);
    if (msk == 0) continue;
    if (WRITE) {
      const long long p = pos + __popcll(msk & ((1ULL << lane) - 1ULL));
      if (ok && p < cap) {
        pairs[2 * p] = overlay ? m / 2 : (int)e;
        pairs[2 * p + 1] = overlay ? (int)(e - B) : m / 2 - (int)B;
      }
      pos += __popcll(msk);
    } else {
      cnt += __popcll(msk);
    }
  }
  return cnt;
}

// one wave per polygon: the counts, or with WRITE the pairs (none when there
// are more than cap in all)
template <bool WRITE>
__global__ void __launch_bounds__(256)
    k_sweep(long B, long O, const int *rank, SweepRecs r, const uint64_t *Y, int *counts,
            const long long *offs, int *pairs, long long cap) {
  const long e = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= B + O || (WRITE && offs[B + O] > cap)) return;
  const int cnt = sweep_polygon<false, WRITE>(e, B, rank, r, Y, WRITE ? offs[e] : 0, pairs, cap);
  if (!WRITE && __lane_id() == 0) counts[e] = cnt;
}

// the same over the *nList polygons of list, on a fixed grid (an empty list
// costs one launch and no read-back of its length)
constexpr unsigned kHeavyBlocks = 512;
template <bool WRITE>
__global__ void __launch_bounds__(256)
    k_sweep_heavy(long B, const int *rank, SweepRecs r, const uint64_t *Y, int *counts,
                  const long long *offs, int *pairs, long long cap, const int *list,
                  const int *nList) {
  const int n = *nList;
  for (int w = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6); w < n; w += (int)gridDim.x * 4) {
    const long e = list[w];
    const int cnt =
        sweep_polygon<true, WRITE>(e, B, rank, r, Y, WRITE ? offs[e] : 0, pairs, cap);
    if (!WRITE && __lane_id() == 0) counts[e] = cnt;
  }
}

// sum of v over a block of 256 threads
__device__ __forceinline__ long long block_sum256(long long v, long long *lds) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if (__lane_id() == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  return lds[0] + lds[1] + lds[2] + lds[3];
}

// The write pass of a small call: each block sums the counts before its four
// polygons itself, in place of a scan launch (at most kFewPolys counts, from
// L2); the last block stores their total in *total.
__global__ void __launch_bounds__(256)
    k_sweep_write_few(long B, long O, const int *rank, SweepRecs r, const uint64_t *Y,
                      const int *counts, int *pairs, long long cap, long long *total) {
  __shared__ long long lds[4];
  const int e0 = (int)blockIdx.x * 4, N = (int)(B + O);
  long long s = 0;
  for (int i = threadIdx.x; i < e0; i += 256) s += counts[i];
  s = block_sum256(s, lds);
  if (threadIdx.x == 0 && e0 + 4 >= N) {
    long long t = s;
    for (int i = e0; i < N; i++) t += counts[i];
    *total = t;
  }
  const int e = e0 + (int)(threadIdx.x >> 6);
  if (e >= N || s >= cap) return;
  for (int i = e0; i < e; i++) s += counts[i];
  sweep_polygon<false, true>(e, B, rank, r, Y, s, pairs, cap);
}

// ------------------------------------------------ stage 1, y strips ----
// The sweep above walks a polygon's whole rank range, so its work grows with
// the sum of the ranges (about N^1.5 for N evenly spread polygons), not with
// the candidates.  For layers of Tuning::stripMin polygons or more the y
// range of the MBR keys is cut into S strips of height 2^shift (the power of
// two at or above twice the median MBR height of 1024 sampled polygons), and
// every left-endpoint record is listed, per layer and in rank order, in each
// strip its y interval touches.  A polygon then visits, in each strip its
// own y interval touches, the other layer's records whose rank lies
// strictly between its endpoints' ranks (a binary search for the first,
// then a walk), applies the sweep's y test, and takes a record only in the
// strip of the larger of the two intervals' lower ends, where both
// intervals are listed, so each candidate is found once.  A polygon's
// candidates are merged over its strips in rank order, the sweep's order.
// Polygons touching more than kStripSpan strips, or with more than
// kStripScan records to visit, are counted and written by the sweep itself
// (one wave each), so the candidate list is the sweep's, entry for entry.
constexpr int kStripSpan = 4;
constexpr int kStripScan = 256;
constexpr long kStripMax = 1L << 22;

// (layer * S + strip, rank) for every listing, in rank order; layer 1 is
// the overlay (endpoint ids from 2B)
__global__ void k_strip_rec_emit(long n, long B, const SweepRec *rec, Strips g,
                                 const long long *off, uint64_t *keys, int *vals) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const SweepRec x = rec[i];
  if (x.id & 1) return;
  const int s0 = strip_of(g, x.y1 < x.y2 ? x.y1 : x.y2),
            s1 = strip_of(g, x.y1 < x.y2 ? x.y2 : x.y1);
  const uint64_t side = x.id < 2 * B ? 0 : 1;
  long long o = off[i];
  for (int s = s0; s <= s1; s++, o++) {
    keys[o] = side * (uint64_t)g.S + (uint64_t)s;
    vals[o] = (int)i;
  }
}

// sOff[k] = the first listing of key k in the sorted keys, k <= 2S (each
// entry written once: the keys in (key[i - 1], key[i]] start at i); also
// clears the length of the list of polygons left to the sweep
__global__ void k_strip_bounds(long R, const uint64_t *skeys, long nk, long long *sOff,
                               int *heavy) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) heavy[0] = 0;
  if (i > R) return;
  const long cur = i < R ? (long)skeys[i] : nk;
  const long prev = i > 0 ? (long)skeys[i - 1] : -1;
  for (long k = prev + 1; k <= cur; k++) sOff[k] = i;
}

// first index of [l, r) whose rank is above v
__device__ __forceinline__ long first_above(const int *a, long l, long r, int v) {
  while (l < r) {
    const long m = (l + r) >> 1;
    if (a[m] > v) r = m;
    else l = m + 1;
  }
  return l;
}

// One polygon's strip ranges: returns false when the sweep takes it (more
// than kStripSpan strips or kStripScan records).
struct StripQuery {
  int sa, ns;
  long p0[kStripSpan], p1[kStripSpan];
};
__device__ __forceinline__ bool strip_query(const Strips &g, const long long *sOff,
                                            const int *list, int side, int lo, int hi,
                                            uint64_t ya, uint64_t yb, StripQuery &q) {
  q.sa = strip_of(g, ya);
  q.ns = strip_of(g, yb) - q.sa + 1;
  if (q.ns > kStripSpan) return false;
  long left = kStripScan;
#pragma unroll
  for (int t = 0; t < kStripSpan; t++) {
    q.p0[t] = q.p1[t] = 0;
    if (t < q.ns) {
      const long k = (long)side * g.S + q.sa + t;
      const long l = sOff[k], r = sOff[k + 1];
      long p = first_above(list, l, r, lo);
      q.p0[t] = p;
      while (p < r && list[p] < hi) {
        if (left-- == 0) return false;
        p++;
      }
      q.p1[t] = p;
    }
  }
  return true;
}

// the sweep's y test and the strip that owns the pair
__device__ __forceinline__ bool strip_hit(const Strips &g, int s, uint64_t ey1, uint64_t ey2,
                                          uint64_t ya, uint64_t ry1, uint64_t ry2) {
  if (ey1 > ry2 || ry1 > ey2) return false;
  const uint64_t rlo = ry1 < ry2 ? ry1 : ry2;
  return strip_of(g, ya > rlo ? ya : rlo) == s;
}

// Count (pairs == nullptr) or write.  The count pass runs one thread per
// listing (R of them, skeys / list): a polygon is taken at the listing of
// its own record in the first strip it touches, so every polygon once, in
// (layer, strip, rank) order -- neighbouring threads then search the same
// strip's list near each other.  It keeps the first kStripInline
// candidates' endpoint ids in inl (rank order), so the write pass (one
// thread per polygon) copies them and searches again only for polygons with
// more; a polygon the sweep takes is marked inl[e, 0] = -1 and appended to
// heavy (heavy[0] counts them, the list follows).
constexpr int kStripInline = 8;
__global__ void __launch_bounds__(256)
    k_strip_query(long B, long O, Strips g, const long long *sOff, const int *list,
                  const uint64_t *skeys, long R, const int *rank, const SweepRec *qrec,
                  const uint64_t *Y, int *counts, const long long *offs, int *pairs,
                  int *heavy, int *inl) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long e = t;
  int lo, hi;
  uint64_t ey1, ey2;
  if (pairs) {
    if (e >= B + O) return;
    lo = rank[2 * e];
    hi = rank[2 * e + 1];
    ey1 = Y[2 * e];
    ey2 = Y[2 * e + 1];
  } else {
    if (t >= R) return;
    lo = list[t];
    const SweepRec me = qrec[lo];
    e = me.id / 2;
    ey1 = me.y1;
    ey2 = me.y2;
    const long key = (long)skeys[t];
    if ((key >= g.S ? key - g.S : key) != strip_of(g, ey1 < ey2 ? ey1 : ey2)) return;
    hi = rank[me.id + 1];
  }
  const bool overlay = e >= B;
  int *mine = inl + (long long)kStripInline * e;
  long long pos = 0;
  int cnt = 0;
  if (pairs) {
    cnt = counts[e];
    if (cnt == 0 || mine[0] < 0) return;
    pos = offs[e];
    if (cnt <= kStripInline) {
      for (int j = 0; j < cnt; j++) {
        const int m = mine[j];
        pairs[2 * (pos + j)] = overlay ? m / 2 : (int)e;
        pairs[2 * (pos + j) + 1] = overlay ? (int)(e - B) : m / 2 - (int)B;
      }
      return;
    }
  }
  const uint64_t ya = ey1 < ey2 ? ey1 : ey2, yb = ey1 < ey2 ? ey2 : ey1;
  StripQuery q;
  if (!strip_query(g, sOff, list, overlay ? 0 : 1, lo, hi, ya, yb, q)) {
    counts[e] = 0;
    mine[0] = -1;
    heavy[1 + atomicAdd(heavy, 1)] = (int)e;
    return;
  }
  // merge the strips' lists by rank
  cnt = 0;
  for (;;) {
    int best = -1, br = 0x7fffffff;
#pragma unroll
    for (int u = 0; u < kStripSpan; u++)
      if (q.p0[u] < q.p1[u]) {
        const int r = list[q.p0[u]];
        if (r < br) {
          br = r;
          best = u;
        }
      }
    if (best < 0) break;
#pragma unroll
    for (int u = 0; u < kStripSpan; u++)
      if (u == best) q.p0[u]++;
    const SweepRec x = qrec[br];
    if (!strip_hit(g, q.sa + best, ey1, ey2, ya, x.y1, x.y2)) continue;
    const int m = x.id;
    if (pairs) {
      pairs[2 * pos] = overlay ? m / 2 : (int)e;
      pairs[2 * pos + 1] = overlay ? (int)(e - B) : m / 2 - (int)B;
      pos++;
    } else {
      if (cnt < kStripInline) mine[cnt] = m;
      cnt++;
    }
  }
  if (!pairs) counts[e] = cnt;
}

// The order of the endpoints and the stream of records (mbr_order).
constexpr long kFewPolys = kRankSort / 2;
struct MbrOrder {
  long B = 0, O = 0;
  bool few = false;     // made by k_order_few
  bool strips = false;  // y strips: records as SweepRec, with their listings
  double avg = -1.0;    // mean vertex count per polygon (-1: unknown)
  int *perm = nullptr, *rank = nullptr;
  uint64_t *Y = nullptr;
  SweepRecs rec;
  Strips g{0, 0, 1};
  int *cnt = nullptr;  // listings per rank
};

static void mbr_order(Context &c, long B, long O, const uint64_t *bMBR, const uint64_t *oMBR,
                      const int *bVNum, const int *oVNum, MbrOrder &m) {
  const long N = B + O, n = 2 * N;
  m.B = B;
  m.O = O;
  m.strips = N >= c.tune.stripMin;
  m.few = N <= kFewPolys && !m.strips;
  m.Y = (uint64_t *)c.ws.get("mbr_Y", 8 * (size_t)n);
  m.perm = (int *)c.ws.get("mbr_perm", 4 * (size_t)n);
  m.rank = (int *)c.ws.get("mbr_rank", 4 * (size_t)n);
  if (m.strips) {
    m.rec.aos = (SweepRec *)c.ws.get("mbr_recs", sizeof(SweepRec) * (size_t)n);
    m.cnt = (int *)c.ws.get("strip_cnt", 4 * (size_t)n);
  } else {
    m.rec.id = (int *)c.ws.get("mbr_rec_id", 4 * (size_t)n);
    m.rec.ylo = (uint64_t *)c.ws.get("mbr_rec_ylo", 8 * (size_t)n);
    m.rec.yhi = (uint64_t *)c.ws.get("mbr_rec_yhi", 8 * (size_t)n);
  }
  if (m.few) {
    LaunchTimer t(c, "mbr_endpoints");
    hipLaunchKernelGGL(k_order_few, dim3(grid_for(n, kRankKeys)), dim3(kRankThreads), 0, c.stream,
                       (int)B, (int)O, bMBR, oMBR, m.Y, m.perm, m.rank, m.rec);
    HIP_CHECK(hipGetLastError());
    return;
  }
  uint64_t *keys = (uint64_t *)c.ws.get("mbr_keys", 8 * (size_t)n);
  int *idx = (int *)c.ws.get("mbr_idx", 4 * (size_t)n);
  uint64_t *skeys = (uint64_t *)c.ws.get("mbr_skeys", 8 * (size_t)n);
  MinMax *part = (MinMax *)c.ws.get("mbr_minmax_part", sizeof(MinMax) * kEndpointBlocks);
  long long *mm = (long long *)c.ws.get("mbr_minmax", 8 * kMmVals);
  const unsigned eb = std::min(grid_for(N, 256), kEndpointBlocks);
  const bool verts = bVNum && oVNum;
  {
    LaunchTimer t(c, "mbr_endpoints");
    hipLaunchKernelGGL(k_endpoints, dim3(eb), dim3(256), 0, c.stream, B, O, bMBR, oMBR,
                       verts ? bVNum : nullptr, oVNum, keys, idx, m.Y, part);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_minmax_final, dim3(1), dim3(kStripSample), 0, c.stream,
                       (const MinMax *)part, (int)eb, N, (const uint64_t *)m.Y,
                       (int)std::min<long>(kStripSample, N), mm, slots_begin(c),
                       (const long long *)c.lb_err);
    HIP_CHECK(hipGetLastError());
  }
  long long h[kHostSlots];
  slots_end(c, {mm, mm + 1, mm + 2, mm + 3, mm + 4, mm + 5}, h);
  m.avg = verts ? (double)h[4] / (double)N : -1.0;
  const uint64_t range = (uint64_t)h[1] - (uint64_t)h[0];
  int bits = 0;
  while (bits < 64 && (range >> bits) != 0) bits++;
  hipLaunchKernelGGL(k_sub_key, dim3(grid_for(n, 256)), dim3(256), 0, c.stream, keys, n,
                     (const long long *)mm);
  HIP_CHECK(hipGetLastError());
  radix_sort_u64(c, keys, idx, skeys, m.perm, n, bits);
  if (m.strips) {
    // at most kStripMax strips
    const uint64_t yr = (uint64_t)h[3] - (uint64_t)h[2];
    int shift = std::min((int)h[5], 63);
    while (shift < 63 && (yr >> shift) + 1 > (uint64_t)kStripMax) shift++;
    m.g = Strips{(uint64_t)h[2], shift, (int)((yr >> shift) + 1)};
  }
  LaunchTimer t(c, "mbr_sweep_prep");
  hipLaunchKernelGGL(k_sweep_prep, dim3(grid_for(n, 256)), dim3(256), 0, c.stream,
                     (const int *)m.perm, n, (const uint64_t *)m.Y, m.rank, m.rec, m.g, m.cnt);
  HIP_CHECK(hipGetLastError());
}

// The strip form of the sweep: fills counts[N] and offs[N + 1] and returns
// the candidate count, with the pairs written to *pairs_out; returns -1
// (nothing written) when the records would be listed more than four times
// each on average, where the polygons are swept instead.
static long strip_sweep(Context &c, const MbrOrder &m, int *counts, long long *offs,
                        int **pairs_out) {
  const long B = m.B, O = m.O, N = B + O, n = 2 * N;
  const Strips g = m.g;
  int *heavy = (int *)c.ws.get("strip_heavy", 4 * (size_t)(N + 1));
  const int *hlist = heavy + 1;
  // listings, in rank order, then stably sorted by (layer, strip)
  long long *off = (long long *)c.ws.get("strip_off", 8 * (size_t)(n + 1));
  scan_i32_to_i64(c, m.cnt, off, n);
  const long R = (long)read_scalar(c, off + n);
  if (R > 4 * N) return -1;
  const long nk = 2L * g.S;
  const size_t R1 = (size_t)std::max(R, 1L);
  uint64_t *keys = (uint64_t *)c.ws.get("strip_keys", 8 * R1);
  int *vals = (int *)c.ws.get("strip_vals", 4 * R1);
  uint64_t *skeys = (uint64_t *)c.ws.get("strip_skeys", 8 * R1);
  int *list = (int *)c.ws.get("strip_list", 4 * R1);
  long long *sOff = (long long *)c.ws.get("strip_soff", 8 * (size_t)(nk + 1));
  {
    LaunchTimer t(c, "mbr_strip_build");
    hipLaunchKernelGGL(k_strip_rec_emit, dim3(grid_for(n, 256)), dim3(256), 0, c.stream, n, B,
                       (const SweepRec *)m.rec.aos, g, (const long long *)off, keys, vals);
    HIP_CHECK(hipGetLastError());
  }
  int kbits = 0;
  while (kbits < 64 && ((uint64_t)(nk - 1) >> kbits) != 0) kbits++;
  radix_sort_u64(c, keys, vals, skeys, list, R, kbits);
  {
    LaunchTimer t(c, "mbr_strip_build");
    hipLaunchKernelGGL(k_strip_bounds, dim3(grid_for(R + 1, 256)), dim3(256), 0, c.stream, R,
                       (const uint64_t *)skeys, nk, sOff, heavy);
    HIP_CHECK(hipGetLastError());
  }
  // counts; the polygons the strips leave to the sweep
  int *inl = (int *)c.ws.get("strip_inline", 4 * (size_t)kStripInline * (size_t)N);
  {
    LaunchTimer t(c, "mbr_strip_count");
    hipLaunchKernelGGL(k_strip_query, dim3(grid_for(R, 256)), dim3(256), 0, c.stream, B, O, g,
                       (const long long *)sOff, (const int *)list, (const uint64_t *)skeys, R,
                       (const int *)m.rank, (const SweepRec *)m.rec.aos, (const uint64_t *)m.Y,
                       counts, (const long long *)nullptr, (int *)nullptr, heavy, inl);
    HIP_CHECK(hipGetLastError());
  }
  {
    LaunchTimer t(c, "mbr_sweep_count");
    hipLaunchKernelGGL(k_sweep_heavy<false>, dim3(kHeavyBlocks), dim3(256), 0, c.stream, B,
                       (const int *)m.rank, m.rec, (const uint64_t *)m.Y, counts,
                       (const long long *)nullptr, (int *)nullptr, 0LL, hlist,
                       (const int *)heavy);
    HIP_CHECK(hipGetLastError());
  }
  scan_i32_to_i64(c, counts, offs, N);
  const long K = (long)read_scalar(c, offs + N);
  int *pairs = (int *)c.ws.get("mbr_pairs", 8 * (size_t)(K > 0 ? K : 1));
  if (K > 0) {
    {
      LaunchTimer t(c, "mbr_strip_write");
      hipLaunchKernelGGL(k_strip_query, dim3(grid_for(N, 256)), dim3(256), 0, c.stream, B, O, g,
                         (const long long *)sOff, (const int *)list, (const uint64_t *)skeys, R,
                         (const int *)m.rank, (const SweepRec *)m.rec.aos,
                         (const uint64_t *)m.Y, counts, (const long long *)offs, pairs, heavy,
                         inl);
      HIP_CHECK(hipGetLastError());
    }
    LaunchTimer t(c, "mbr_sweep_write");
    hipLaunchKernelGGL(k_sweep_heavy<true>, dim3(kHeavyBlocks), dim3(256), 0, c.stream, B,
                       (const int *)m.rank, m.rec, (const uint64_t *)m.Y, counts,
                       (const long long *)offs, pairs, (long long)K, hlist,
                       (const int *)heavy);
    HIP_CHECK(hipGetLastError());
  }
  *pairs_out = pairs;
  return K;
}

// The pairs of the counted candidates (fold: from the counts alone), into
// places for K of them.
static void mbr_write(Context &c, const MbrOrder &m, long K, bool fold, int *counts,
                      long long *offs, int **pairs_out) {
  const long B = m.B, O = m.O, N = B + O;
  int *pairs = (int *)c.ws.get("mbr_pairs", 8 * (size_t)(K > 0 ? K : 1));
  *pairs_out = pairs;
  if (K <= 0) return;
  LaunchTimer t(c, "mbr_sweep_write");
  if (fold)
    hipLaunchKernelGGL(k_sweep_write_few, dim3(grid_for(N, 4)), dim3(256), 0, c.stream, B, O,
                       (const int *)m.rank, m.rec, (const uint64_t *)m.Y, (const int *)counts,
                       pairs, (long long)K, offs + N);
  else
    hipLaunchKernelGGL(k_sweep<true>, dim3(grid_for(N, 4)), dim3(256), 0, c.stream, B, O,
                       (const int *)m.rank, m.rec, (const uint64_t *)m.Y, counts,
                       (const long long *)offs, pairs, (long long)K);
  HIP_CHECK(hipGetLastError());
}

// Counts per polygon, their offsets, and the candidate pairs.  With cap <= 0
// the count is read back and the pairs are sized to it; with cap > 0 they are
// given cap places without a read-back and the count stays at *kDev, which
// the caller compares with cap when it reads it.
static long mbr_candidates(Context &c, MbrOrder &m, long cap, int *counts, long long *offs,
                           int **pairs_out, const long long **kDev) {
  const long B = m.B, O = m.O, N = B + O;
  if (m.strips) {
    const long K = strip_sweep(c, m, counts, offs, pairs_out);
    if (K >= 0) return K;
    // records as arrays for the sweep of every polygon
    const long n = 2 * N;
    m.strips = false;
    m.rec.aos = nullptr;
    m.rec.id = (int *)c.ws.get("mbr_rec_id", 4 * (size_t)n);
    m.rec.ylo = (uint64_t *)c.ws.get("mbr_rec_ylo", 8 * (size_t)n);
    m.rec.yhi = (uint64_t *)c.ws.get("mbr_rec_yhi", 8 * (size_t)n);
    LaunchTimer t(c, "mbr_sweep_prep");
    hipLaunchKernelGGL(k_sweep_prep, dim3(grid_for(n, 256)), dim3(256), 0, c.stream,
                       (const int *)m.perm, n, (const uint64_t *)m.Y, m.rank, m.rec, m.g,
                       (int *)nullptr);
    HIP_CHECK(hipGetLastError());
  }
  {
    LaunchTimer t(c, "mbr_sweep_count");
    hipLaunchKernelGGL(k_sweep<false>, dim3(grid_for(N, 4)), dim3(256), 0, c.stream, B, O,
                       (const int *)m.rank, m.rec, (const uint64_t *)m.Y, counts,
                       (const long long *)nullptr, (int *)nullptr, 0LL);
    HIP_CHECK(hipGetLastError());
  }
  const bool fold = m.few && cap > 0;
  long K = cap;
  if (!fold) scan_i32_to_i64(c, counts, offs, N);
  if (cap <= 0) K = (long)read_scalar(c, offs + N);
  if (kDev) *kDev = offs + N;
  mbr_write(c, m, K, fold, counts, offs, pairs_out);
  return K;
}

long mbr_filter(Context &c, long B, long O, const uint64_t *bMBR, const uint64_t *oMBR,
                int **counts_out, int **pairs_out) {
  const long N = B + O;
  if (N <= 0) return 0;
  MbrOrder m;
  mbr_order(c, B, O, bMBR, oMBR, nullptr, nullptr, m);
  *counts_out = (int *)c.ws.get("mbr_counts", 4 * (size_t)N);
  long long *offs = (long long *)c.ws.get("mbr_offs", 8 * (size_t)(N + 1));
  return mbr_candidates(c, m, 0, *counts_out, offs, pairs_out, nullptr);
}

// -------------------------------------------------------- stages 2 to 5 ----
__device__ __forceinline__ void cmbr_of(const double *bm, const double *om, double *box,
                                        int &type) {
  const double x1 = bm[0], x2 = bm[2], y1 = bm[1], y2 = bm[3];
  const double a1 = om[0], a2 = om[2], b1 = om[1], b2 = om[3];
  box[0] = a1 > x1 ? a1 : x1;
  box[1] = b1 > y1 ? b1 : y1;
  box[2] = a2 < x2 ? a2 : x2;
  box[3] = b2 < y2 ? b2 : y2;
  type = x1 == box[0] && x2 == box[2] && y1 == box[1] && y2 == box[3]   ? 1
         : a1 == box[0] && a2 == box[2] && b1 == box[1] && b2 == box[3] ? 2
                                                                        : 0;
}

__global__ void k_get_cmbr(long K, const int *pairs, const double *bMBR2, const double *oMBR2,
                           double *cmbr, int *pipFlag, signed char *pipType, int *joinFlag) {
  long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= K) return;
  double box[4];
  int t;
  cmbr_of(bMBR2 + 4L * pairs[2 * k], oMBR2 + 4L * pairs[2 * k + 1], box, t);
  for (int j = 0; j < 4; j++) cmbr[4 * k + j] = box[j];
  joinFlag[k] = 1;
  pipFlag[k] = t != 0;
  pipType[k] = (signed char)t;
}

// Groups of G lanes (8, 16 or 64, a wave's aligned parts) take one candidate
// each; their ballots are masked to the group, so groups of one wave may be
// at different loop counts.
template <int G>
__device__ __forceinline__ unsigned long long group_ballot(bool v) {
  const unsigned long long m = __ballot(v);
  if (G == 64) return m;
  return m & (((1ULL << (G & 63)) - 1ULL) << ((int)__lane_id() & ~(G - 1)));
}

// crossing parity of the point over the ring, one edge per lane
template <int G>
__device__ __forceinline__ int pip_parity(double pX, double pY, const double *poly, long vNum) {
  const int g = (int)__lane_id() & (G - 1);
  int parity = 0;
  for (long i0 = 0; i0 < vNum; i0 += G) {
    long i = i0 + g;
    bool tog = false;
    if (i < vNum) {
      long j = i == 0 ? vNum - 1 : i - 1;
      double X1 = poly[2 * i], Y1 = poly[2 * i + 1], X2 = poly[2 * j], Y2 = poly[2 * j + 1];
      if ((Y1 > pY) != (Y2 > pY)) tog = pX < (X2 - X1) * (pY - Y1) / (Y2 - Y1) + X1;
    }
    parity ^= __popcll(group_ballot<G>(tog)) & 1;
  }
  return parity;
}

struct PolyRefs {
  const double *bCoords, *oCoords;
  const int *bVNum, *oVNum;
  const long *bVPSNum, *oVPSNum;
};
static PolyRefs poly_refs(const JoinInputs &in) {
  return PolyRefs{in.bCoords, in.oCoords, in.bVNum, in.oVNum, in.bVPSNum, in.oVPSNum};
}

// the PiP test of a candidate of type 1 (base in overlay) or 2
template <int G>
__device__ __forceinline__ int pip_within(const PolyRefs &p, int b, int o, int type) {
  const long bS = b > 0 ? p.bVPSNum[b - 1] : 0, oS = o > 0 ? p.oVPSNum[o - 1] : 0;
  const double *pt = type == 1 ? p.bCoords + 2 * bS : p.oCoords + 2 * oS;
  return type == 1 ? pip_parity<G>(pt[0], pt[1], p.oCoords + 2 * oS, p.oVPSNum[o] - oS)
                   : pip_parity<G>(pt[0], pt[1], p.bCoords + 2 * bS, p.bVPSNum[b] - bS);
}

__global__ void __launch_bounds__(256)
    k_pip(long nCand, const int *cand, const int *pairs, const signed char *pipType, PolyRefs p,
          int *pipFlag, int *joinFlag) {
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nCand) return;
  const int k = cand[w];
  const int parity = pip_within<64>(p, pairs[2 * k], pairs[2 * k + 1], pipType[k]);
  if (__lane_id() == 0) {
    pipFlag[k] = parity;
    if (parity == 1) joinFlag[k] = 0;
  }
}

// ------------------------------------------------------------ stage 4 ----
// A vertex in one load: as two numbers, the compiler puts the second behind
// the test of the first, one more wait a step (the count of 486 000 pairs of
// rings of 100 to 300 vertices: 674 us so, 440 in one load).
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ d2 ld2(const double *c, int i) { return *(const d2 *)(c + 2L * i); }

__device__ __forceinline__ bool cmf_edge(const double *c, int vNum, int i, double cX1, double cY1,
                                         double cX2, double cY2) {
  const d2 v = ld2(c, i), w = ld2(c, i < vNum - 1 ? i + 1 : 0);
  if ((cX1 > v.x && cX1 > w.x) || (cX2 < v.x && cX2 < w.x)) return false;
  if ((cY1 > v.y && cY1 > w.y) || (cY2 < v.y && cY2 < w.y)) return false;
  return true;
}

// The edges of one ring that the box keeps, counted and, when asked for,
// listed in ring order: out[0..] in global memory and the first kSegList of
// them in lds.
constexpr int kSegList = 64;
template <typename EdgeT, int G>
__device__ __forceinline__ int cmf_ring(const double *c, int vNum, const double *box, EdgeT *out,
                                        int *lds) {
  const int lane = __lane_id(), g = lane & (G - 1);
  int n = 0;
  for (int i0 = 0; i0 < vNum; i0 += G) {
    const int i = i0 + g;
    const bool ok = i < vNum && cmf_edge(c, vNum, i, box[0], box[1], box[2], box[3]);
    const unsigned long long m = group_ballot<G>(ok);
    if (out && ok) {
      const int p = n + __popcll(m & ((1ULL << lane) - 1ULL));
      out[p] = (EdgeT)i;
      if (lds && p < kSegList) lds[p] = i;
    }
    n += __popcll(m);
  }
  return n;
}

__device__ __forceinline__ const double *ring_of(const double *c, const long *vps, int k) {
  return c + 2 * (k > 0 ? vps[k - 1] : 0);
}

// the reference's two passes, one wave per listed pair: counts (and clears
// joinFlag when a side has no edge) ...
__global__ void __launch_bounds__(256)
    k_cmf_count(long nList, const int *list, const int *pairs, const double *cmbr, PolyRefs p,
                int *joinFlag, int *bCount, int *oCount) {
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nList) return;
  const int k = list[w], b = pairs[2 * k], o = pairs[2 * k + 1];
  const int nb = cmf_ring<int, 64>(ring_of(p.bCoords, p.bVPSNum, b), p.bVNum[b], cmbr + 4L * k,
                                   nullptr, nullptr);
  const int no = cmf_ring<int, 64>(ring_of(p.oCoords, p.oVPSNum, o), p.oVNum[o], cmbr + 4L * k,
                                   nullptr, nullptr);
  if (__lane_id() != 0) return;
  const bool keep = nb && no;
  if (!keep) joinFlag[k] = 0;
  bCount[k] = keep ? nb : 0;
  oCount[k] = keep ? no : 0;
}

// ... and writes the 16-bit edge lists at its inclusive prefix
__device__ __forceinline__ long long incl_base(const long long *off, int k) {
  return k > 0 ? off[k - 1] : 0;
}
__global__ void __launch_bounds__(256)
    k_cmf_apply(long nList, const int *list, const int *pairs, const double *cmbr, PolyRefs p,
                const long long *bIncl, const long long *oIncl, short *bEdge, short *oEdge) {
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nList) return;
  const int k = list[w], b = pairs[2 * k], o = pairs[2 * k + 1];
  cmf_ring<short, 64>(ring_of(p.bCoords, p.bVPSNum, b), p.bVNum[b], cmbr + 4L * k,
                      bEdge + incl_base(bIncl, k), nullptr);
  cmf_ring<short, 64>(ring_of(p.oCoords, p.oVPSNum, o), p.oVNum[o], cmbr + 4L * k,
                      oEdge + incl_base(oIncl, k), nullptr);
}

// ------------------------------------------------------------ stage 5 ----
__device__ __forceinline__ bool seg_hit(double bX1, double bY1, double bX2, double bY2,
                                        double oX1, double oY1, double oX2, double oY2) {
  if (((bX2 < oX1) && (bX2 < oX2)) && ((bX1 < oX1) && (bX1 < oX2))) return false;
  if (((bX2 > oX1) && (bX2 > oX2)) && ((bX1 > oX1) && (bX1 > oX2))) return false;
  if (((bY2 < oY1) && (bY2 < oY2)) && ((bY1 < oY1) && (bY1 < oY2))) return false;
  if (((bY2 > oY1) && (bY2 > oY2)) && ((bY1 > oY1) && (bY1 > oY2))) return false;
  double denom = ((bX1 - bX2) * (oY1 - oY2)) - ((bY1 - bY2) * (oX1 - oX2));
  if (denom == 0) {
    if ((oX1 == oX2 && oX1 == bX1) || (bX1 == bX2 && bX1 == oX1)) return true;
    double oM = (oY2 - oY1) / (oX2 - oX1);
    double bM = (bY2 - bY1) / (bX2 - bX1);
    double oB = oY1 - oM * oX1;
    double bB = bY1 - bM * bX1;
    return oB == bB;
  }
  double nomX = (((bX1 * bY2) - (bY1 * bX2)) * (oX1 - oX2)) -
                ((bX1 - bX2) * ((oX1 * oY2) - (oY1 * oX2)));
  double nomY = ((((bX1 * bY2) - (bY1 * bX2)) * (oY1 - oY2)) -
                 (((bY1 - bY2) * ((oX1 * oY2) - (oY1 * oX2)))));
  double x0 = nomX / denom, y0 = nomY / denom;
  if ((x0 > bX1 && x0 > bX2) || (x0 < bX1 && x0 < bX2)) return false;
  if ((x0 > oX1 && x0 > oX2) || (x0 < oX1 && x0 < oX2)) return false;
  if ((y0 > bY1 && y0 > bY2) || (y0 < bY1 && y0 < bY2)) return false;
  if ((y0 > oY1 && y0 > oY2) || (y0 < oY1 && y0 < oY2)) return false;
  return true;
}

constexpr int kSegStage = 4;

__device__ __forceinline__ int gcd_int(int a, int b) {
  while (b) {
    const int t = a % b;
    a = b;
    b = t;
  }
  return a;
}

// The order in which a pair's base edges are taken: i -> (i * S) mod bE,
// S coprime to bE and near 0.618 bE, a permutation that spreads successive
// rounds over the whole base list.  The flag is "some edge pair hits", so
// the order changes only how soon a pair that hits stops: its hits cluster
// where the rings cross, which index order reaches after half the list on
// average and this order after about bE / (number of base edges with hits).
__device__ __forceinline__ int seg_stride(int bE) {
  if (bE <= 2) return 1;
  int S = (int)(0.6180339887498949 * bE);
  if (S < 1) S = 1;
  while (gcd_int(S, bE) != 1) S++;
  return S;
}

// Whether some pair of the two edge lists (bAt(i), oAt(j): ring positions)
// hits, over a group of G lanes.
template <int G, typename FB, typename FO>
__device__ __forceinline__ int seg_any(const double *bc, int bV, const double *oc, int oV, int bE,
                                       int oE, FB bAt, FO oAt) {
  const int lane = (int)__lane_id() & (G - 1);
  // pairs per lane a round: a small group's few pairs fill one
  constexpr int U = G == 64 ? kSegStage : 1;
  const long long total = (long long)bE * oE;
  int flag = 0;
  if (total >= 0x7fffffffLL) {
    // lists of 2^31 pairs or more (rings of tens of thousands of listed
    // edges): one pair per lane a round, 64-bit indices
    for (long long t0 = 0; t0 < total && !flag; t0 += G) {
      const long long t = t0 + lane;
      bool hit = false;
      if (t < total) {
        const int bi = bAt((int)(t / oE)), oi = oAt((int)(t % oE));
        const int b2 = bi < bV - 1 ? bi + 1 : 0, o2 = oi < oV - 1 ? oi + 1 : 0;
        const double v0 = bc[2 * bi], v1 = bc[2 * bi + 1], v2 = bc[2 * b2], v3 = bc[2 * b2 + 1];
        hit = !(v0 == v2 && v1 == v3) && seg_hit(v0, v1, v2, v3, oc[2 * oi], oc[2 * oi + 1],
                                                 oc[2 * o2], oc[2 * o2 + 1]);
      }
      flag = group_ballot<G>(hit) != 0ULL;
    }
    return flag;
  }
  // U edge pairs per lane a round, all their loads issued before
  // the tests; the flag is "some pair hits", which testing pairs past the
  // first hit cannot change
  const unsigned tot = (unsigned)total, uoE = (unsigned)(oE > 0 ? oE : 1);
  const unsigned long long S = (unsigned long long)(tot > G * U ? seg_stride(bE) : 1);
  for (unsigned t0 = 0; t0 < tot && !flag; t0 += G * U) {
    int bi[U], oi[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned t = t0 + G * u + lane;
      bi[u] = oi[u] = -1;
      if (t >= tot) continue;
      const unsigned q = t / uoE;
      bi[u] = bAt(S == 1 ? (int)q : (int)(q * S % (unsigned long long)bE));
      oi[u] = oAt((int)(t - q * uoE));
    }
    d2 s[U][4];
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (bi[u] < 0) continue;
      const int b2 = bi[u] < bV - 1 ? bi[u] + 1 : 0, o2 = oi[u] < oV - 1 ? oi[u] + 1 : 0;
      s[u][0] = ld2(bc, bi[u]);
      s[u][1] = ld2(bc, b2);
      s[u][2] = ld2(oc, oi[u]);
      s[u][3] = ld2(oc, o2);
    }
    bool hit = false;
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (bi[u] < 0) continue;
      if (!(s[u][0].x == s[u][1].x && s[u][0].y == s[u][1].y))
        hit |= seg_hit(s[u][0].x, s[u][0].y, s[u][1].x, s[u][1].y, s[u][2].x, s[u][2].y,
                       s[u][3].x, s[u][3].y);
    }
    flag = group_ballot<G>(hit) != 0ULL;
  }
  return flag;
}

// the reference's refine: one wave per listed pair over 16-bit lists at the
// inclusive prefixes, the flag by list position
__global__ void __launch_bounds__(256)
    k_segjoin(long nList, const int *list, const int *pairs, PolyRefs p, const long long *bIncl,
              const long long *oIncl, const short *bEdge, const short *oEdge, int *flagByList) {
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nList) return;
  const int k = list[w], b = pairs[2 * k], o = pairs[2 * k + 1];
  const long bS = b > 0 ? p.bVPSNum[b - 1] : 0, oS = o > 0 ? p.oVPSNum[o - 1] : 0;
  const long long b0 = incl_base(bIncl, k), o0 = incl_base(oIncl, k);
  const short *be = bEdge + b0, *oe = oEdge + o0;
  const int flag = seg_any<64>(
      p.bCoords + 2 * bS, (int)(p.bVPSNum[b] - bS), p.oCoords + 2 * oS, (int)(p.oVPSNum[o] - oS),
      (int)(bIncl[k] - b0), (int)(oIncl[k] - o0), [&](int i) { return (int)be[i]; },
      [&](int i) { return (int)oe[i]; });
  if (__lane_id() == 0) flagByList[w] = flag;
}

// ------------------------------------------------- stages 2 to 5, fused ----
// A candidate goes through CMBR, PiP and the CMF count in one pass by one
// group of lanes (k_refine_count) and, once the edge lists have their places,
// through the CMF lists and the segment test in a second one
// (k_refine_apply), its short edge lists in LDS between the two.  For 550 000
// polygons of 8 vertices on one MI355X the stages as passes of their own over
// compacted lists, one wave per pair in the segment test, took 600 us of
// kernel time in 13 launches: that test alone 331 us with 64 lanes on about
// nine edge pairs.  The two passes take 53 and 87 us (88 and 131 with a vertex
// loaded as two numbers; then 110 and 170 with 16 lanes per candidate instead
// of 8).  What bounds both now is the chain of
// dependent loads (pair, ring bounds, vertices); groups of 8 lanes keep eight
// chains per wave in flight.
//
// n is the length of the per-candidate arrays; the candidates are *kDev of
// them (all n without it); when *kDev exceeds n, every count is 0 and nothing
// else is touched.
struct RefineOut {
  double *cmbr;
  int *pipFlag, *joinFlag, *bCount, *oCount, *segFlag, *joined;
  signed char *pipType;
};

template <int G>
__global__ void __launch_bounds__(256)
    k_refine_count(long n, const long long *kDev, const int *pairs, PolyRefs p,
                   const double *bMBR2, const double *oMBR2, RefineOut r) {
  long K = kDev ? (long)*kDev : n;
  if (K > n) K = 0;
  const int g = (int)__lane_id() & (G - 1);
  const long step = (long)gridDim.x * (256 / G);
  for (long k = (long)blockIdx.x * (256 / G) + threadIdx.x / G; k < n; k += step) {
    if (k >= K) {  // past the candidates: the scans' inputs
      if (g == 0) r.bCount[k] = r.oCount[k] = r.joined[k] = 0;
      continue;
    }
    const int b = pairs[2 * k], o = pairs[2 * k + 1];
    const double *bc = ring_of(p.bCoords, p.bVPSNum, b), *oc = ring_of(p.oCoords, p.oVPSNum, o);
    const int bn = p.bVNum[b], on = p.oVNum[o];
    double box[4];
    int type;
    cmbr_of(bMBR2 + 4L * b, oMBR2 + 4L * o, box, type);
    const int within = type ? pip_within<G>(p, b, o, type) : 0;
    int nb = 0, no = 0;
    if (!within) {
      nb = cmf_ring<int, G>(bc, bn, box, nullptr, nullptr);
      if (nb) no = cmf_ring<int, G>(oc, on, box, nullptr, nullptr);
    }
    const bool keep = nb && no;
    if (g < 4) r.cmbr[4 * k + g] = g == 0 ? box[0] : g == 1 ? box[1] : g == 2 ? box[2] : box[3];
    if (g == 0) {
      r.pipFlag[k] = within;
      r.pipType[k] = (signed char)type;
      r.joinFlag[k] = keep;
      r.bCount[k] = keep ? nb : 0;
      r.oCount[k] = keep ? no : 0;
      r.segFlag[k] = 0;
      r.joined[k] = within;
    }
  }
}

// FOLD (small calls): each block takes a run of candidates and sums the
// counts before it itself, in place of a scan launch, and writes the offsets.
// A list that would end beyond capB or capO is not written: the totals tell.
template <int G, bool FOLD>
__global__ void __launch_bounds__(256)
    k_refine_apply(long n, const long long *kDev, const int *pairs, PolyRefs p, RefineOut r,
                   long long *bOff, long long *oOff, int *bEdge, int *oEdge, long long capB,
                   long long capO) {
  constexpr int per = 256 / G;
  __shared__ int lists[per][2][kSegList];
  __shared__ long long lds[4];
  const long K = kDev ? (long)*kDev : n;
  if (K > n) return;
  const int g = (int)__lane_id() & (G - 1), grp = threadIdx.x / G;
  int *lb = lists[grp][0], *lo = lists[grp][1];
  long k0 = (long)blockIdx.x * per, k1 = K, step = (long)gridDim.x * per, run = 0;
  long long sb = 0, so = 0;
  if (FOLD) {
    run = (K + (long)gridDim.x * per - 1) / ((long)gridDim.x * per) * per;
    k0 = (long)blockIdx.x * run;
    k1 = k0 + run < K ? k0 + run : K;
    step = per;
    if (k0 >= K && !(blockIdx.x == 0 && K == 0)) return;
    for (long j = threadIdx.x; j < k0; j += 256) {
      sb += r.bCount[j];
      so += r.oCount[j];
    }
    sb = block_sum256(sb, lds);
    so = block_sum256(so, lds);
    if (threadIdx.x == 0 && k1 == K) {
      long long tb = sb, to = so;
      for (long j = k0; j < K; j++) {
        tb += r.bCount[j];
        to += r.oCount[j];
      }
      bOff[K] = tb;
      oOff[K] = to;
    }
  }
  for (long k = k0 + grp, prev = k0; k < k1; k += step) {
    long long pb, po;
    if (FOLD) {
      for (; prev < k; prev++) {
        sb += r.bCount[prev];
        so += r.oCount[prev];
      }
      pb = sb;
      po = so;
      if (g == 0) {
        bOff[k] = pb;
        oOff[k] = po;
      }
    } else {
      pb = bOff[k];
      po = oOff[k];
    }
    // (no branch before the ring loops, so that every load of a step of the
    // chain is in flight at once; a list without places is left empty)
    const int b = pairs[2 * k], o = pairs[2 * k + 1];
    int bE = r.bCount[k], oE = r.oCount[k];
    if (pb + bE > capB || po + oE > capO) bE = oE = 0;
    const double *bc = ring_of(p.bCoords, p.bVPSNum, b), *oc = ring_of(p.oCoords, p.oVPSNum, o);
    int *be = bEdge + pb, *oe = oEdge + po;
    const int bn = bE ? p.bVNum[b] : 0, on = oE ? p.oVNum[o] : 0;
    double box[4];
    for (int j = 0; j < 4; j++) box[j] = r.cmbr[4 * k + j];
    __threadfence_block();  // the last candidate's list reads, before the writes
    cmf_ring<int, G>(bc, bn, box, be, lb);
    cmf_ring<int, G>(oc, on, box, oe, lo);
    __threadfence_block();  // the lists, before other lanes read them
    const int bV = (int)(p.bVPSNum[b] - (b > 0 ? p.bVPSNum[b - 1] : 0)),
              oV = (int)(p.oVPSNum[o] - (o > 0 ? p.oVPSNum[o - 1] : 0));
    const int flag =
        bE <= kSegList && oE <= kSegList
            ? seg_any<G>(bc, bV, oc, oV, bE, oE, [&](int i) { return lb[i]; },
                         [&](int i) { return lo[i]; })
            : seg_any<G>(bc, bV, oc, oV, bE, oE, [&](int i) { return be[i]; },
                         [&](int i) { return oe[i]; });
    if (g == 0 && flag) {
      r.segFlag[k] = 1;
      r.joined[k] = 1;
    }
  }
}

// What a join reads back: candidates, edges listed on either side, PiP
// candidates, within, CMF survivors and intersecting pairs; of a small call
// also the layers' vertices, which it has not summed before.
constexpr int kJoinStats = 7;

// The end of a small call in one block: the joined pairs in order and the
// read-back values.  Rounds of four candidates per thread.
__global__ void __launch_bounds__(1024)
    k_refine_out_few(long n, const long long *kDev, const int *pairs, PolyRefs p, long B, long O,
                     RefineOut r, const long long *bOff, const long long *oOff, long long capB,
                     long long capO, int *jidx, int *jpairs, long long *st, long long *slots,
                     const long long *lbErr) {
  __shared__ int lds[16];
  __shared__ long long lds64[16];
  const long K = (long)*kDev;
  long long acc = 0;  // PiP candidates, within, survivors, hits: 16 bits each (n <= 2^15)
  const bool fits = K <= n && bOff[K] <= capB && oOff[K] <= capO;
  int base = 0;
  for (long k0 = 0; fits && k0 < K; k0 += 4096) {
    int f[4], c = 0;
    for (int u = 0; u < 4; u++) {
      const long k = k0 + 4 * threadIdx.x + u;
      f[u] = k < K ? r.joined[k] : 0;
      c += f[u];
      if (k < K)
        acc += (r.pipType[k] != 0) + ((long long)(r.pipFlag[k] == 1) << 16) +
               ((long long)(r.joinFlag[k] != 0) << 32) + ((long long)(r.segFlag[k] != 0) << 48);
    }
    int tot;
    int at = base + block_excl_scan<int>(c, lds, tot);
    for (int u = 0; u < 4; u++) {
      if (!f[u]) continue;
      const long k = k0 + 4 * threadIdx.x + u;
      jidx[at] = (int)k;
      jpairs[2 * at] = pairs[2 * k];
      jpairs[2 * at + 1] = pairs[2 * k + 1];
      at++;
    }
    base += tot;
  }
  long long all;
  block_excl_scan<long long>(acc, lds64, all);
  if (threadIdx.x != 0) return;
  long long v[kJoinStats + 1] = {K, K <= n ? bOff[K] : 0, K <= n ? oOff[K] : 0};
  for (int i = 0; i < 4; i++) v[3 + i] = (all >> (16 * i)) & 0xffff;
  v[kJoinStats] = (B ? p.bVPSNum[B - 1] : 0) + (O ? p.oVPSNum[O - 1] : 0);
  for (int i = 0; i <= kJoinStats; i++) st[i] = v[i];
  put_slots(slots, v, kJoinStats + 1, lbErr);
}

// The same end in two launches: the pairs of the compacted list and each
// block's counts, then their sums.
constexpr unsigned kOutBlocks = 512;
__global__ void __launch_bounds__(256)
    k_refine_out(long n, const long long *kDev, const int *pairs, RefineOut r, const int *jidx,
                 const long long *nJoined, int *jpairs, long long *part) {
  __shared__ long long lds[4];
  const long K = kDev ? (long)*kDev : n;
  long long c[4] = {0, 0, 0, 0};
  if (K <= n) {
    const long nj = (long)*nJoined, step = (long)gridDim.x * 256;
    for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < K; k += step) {
      if (k < nj) {
        const int j = jidx[k];
        jpairs[2 * k] = pairs[2 * j];
        jpairs[2 * k + 1] = pairs[2 * j + 1];
      }
      c[0] += r.pipType[k] != 0;
      c[1] += r.pipFlag[k] == 1;
      c[2] += r.joinFlag[k] != 0;
      c[3] += r.segFlag[k] != 0;
    }
  }
  for (int i = 0; i < 4; i++) {
    const long long s = block_sum256(c[i], lds);
    if (threadIdx.x == 0) part[4 * blockIdx.x + i] = s;
  }
}
__global__ void __launch_bounds__(256)
    k_refine_stats(long n, const long long *kDev, const long long *bOff, const long long *oOff,
                   const long long *part, int nPart, long long *st, long long *slots,
                   const long long *lbErr) {
  __shared__ long long lds[4];
  long long v[kJoinStats];
  for (int i = 0; i < 4; i++) {
    long long s = 0;
    for (int j = threadIdx.x; j < nPart; j += 256) s += part[4 * j + i];
    v[3 + i] = block_sum256(s, lds);
  }
  if (threadIdx.x != 0) return;
  v[0] = kDev ? *kDev : n;
  v[1] = bOff[n];
  v[2] = oOff[n];
  for (int i = 0; i < kJoinStats; i++) st[i] = v[i];
  put_slots(slots, v, kJoinStats, lbErr);
}

// polygons of at most this many vertices on average take groups of 16 lanes
// (one group per candidate, eight per wave, of at most kCmfTiny)
constexpr double kCmfSmall = 32.0, kCmfTiny = 12.0;
constexpr long long kEdgeGuess = 1LL << 22;

// Stages 2 to 5 over n candidate places, *kDev of them candidates (null: all
// n); avg, the mean vertex count per polygon, is set by a small call.  Returns
// false when there are more than n candidates: r.K is their number and nothing
// else of r is valid.
static bool refine(Context &c, const JoinInputs &in, long n, const long long *kDev, bool few,
                   double &avg, const int *pairs, JoinRefine &r) {
  const size_t n1 = (size_t)std::max(n, 1L);
  r.cmbr = (double *)c.ws.get("jr_cmbr", 32 * n1);
  r.pipFlag = (int *)c.ws.get("jr_pipFlag", 4 * n1);
  r.pipType = (signed char *)c.ws.get("jr_pipType", n1);
  r.joinFlag = (int *)c.ws.get("jr_joinFlag", 4 * n1);
  r.bCount = (int *)c.ws.get("jr_bCount", 4 * n1);
  r.oCount = (int *)c.ws.get("jr_oCount", 4 * n1);
  long long *bOff = (long long *)c.ws.get("jr_bOff", 8 * (n1 + 1));
  long long *oOff = (long long *)c.ws.get("jr_oOff", 8 * (n1 + 1));
  r.segFlag = (int *)c.ws.get("jr_segFlag", 4 * n1);
  int *joined = (int *)c.ws.get("jr_joined", 4 * n1);
  int *jidx = (int *)c.ws.get("jr_joined_idx", 4 * n1);
  r.joinedPairs = (int *)c.ws.get("jr_joinedPairs", 8 * n1);
  r.K = r.pipNum = r.within = r.cmfCand = r.E = r.hits = r.nJoined = 0;
  r.nbEdges = r.noEdges = 0;
  if (n <= 0) return true;
  const PolyRefs p = poly_refs(in);
  const RefineOut o{r.cmbr,   r.pipFlag, r.joinFlag, r.bCount,
                    r.oCount, r.segFlag, joined,     r.pipType};
  long long *st = (long long *)c.ws.get("jr_stats", 8 * (kJoinStats + 1));
  // Edge lists are given a place before their lengths are known: the polygons'
  // mean vertex count per candidate, within 8 to 32.  Totals beyond that (or
  // beyond what an earlier call left) cost the second pass again.  Above
  // kEdgeGuess places that would cost more than the 12 us of a read-back, and
  // memory; under capture a read-back costs nothing on replay: there the
  // totals are read first, and the lists get what they need.
  const long long est = n * (avg < 0 ? 32 : (long long)std::min(std::max(avg, 8.0), 32.0));
  auto cap_of = [&](const char *name) {
    const long long have = c.replay ? 0 : (long long)(c.ws.slots[name].bytes / 4);
    return std::max(est, have);
  };
  long long capB = cap_of("jr_bEdge"), capO = cap_of("jr_oEdge");
  // four candidates per wave where the layers' polygons are small on average;
  // a small call has waves to spare
  const int G = c.tune.cmfGroup         ? c.tune.cmfGroup
                : few || avg < 0        ? 64
                : avg <= kCmfTiny       ? 8
                : avg <= kCmfSmall      ? 16
                                        : 64;
  const int per = 256 / G;
  // known counts: a group per candidate; else at most four times the waves
  // that the GPU holds, as most places are empty
  const unsigned full = 32u * (unsigned)c.cu_count;
  const unsigned grid = kDev ? std::min(grid_for(n, per), full) : grid_for(n, per);
  {
    LaunchTimer t(c, "refine_count");
    auto kern = G == 8 ? k_refine_count<8> : G == 16 ? k_refine_count<16> : k_refine_count<64>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, c.stream, n, kDev, pairs, p, in.bMBR2,
                       in.oMBR2, o);
    HIP_CHECK(hipGetLastError());
  }
  if (!few) scan_i32_to_i64_multi(c, {{r.bCount, bOff, n}, {r.oCount, oOff, n}});
  if (!few && (c.replay || (!kDev && est > kEdgeGuess))) {
    long long tot[kHostSlots];
    read_scalars(c, {bOff + n, oOff + n}, tot);
    capB = std::max(tot[0], 1LL);
    capO = std::max(tot[1], 1LL);
  }
  for (;;) {
    r.bEdge = (int *)c.ws.get("jr_bEdge", 4 * (size_t)capB);
    r.oEdge = (int *)c.ws.get("jr_oEdge", 4 * (size_t)capO);
    {
      LaunchTimer t(c, "refine_apply");
      auto kern = few       ? (G == 16 ? k_refine_apply<16, true> : k_refine_apply<64, true>)
                  : G == 8  ? k_refine_apply<8, false>
                  : G == 16 ? k_refine_apply<16, false>
                            : k_refine_apply<64, false>;
      hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, c.stream, n, kDev, pairs, p, o, bOff,
                         oOff, r.bEdge, r.oEdge, capB, capO);
      HIP_CHECK(hipGetLastError());
    }
    if (few) {
      hipLaunchKernelGGL(k_refine_out_few, dim3(1), dim3(1024), 0, c.stream, n, kDev, pairs, p,
                         in.B, in.O, o, (const long long *)bOff, (const long long *)oOff, capB,
                         capO, jidx, r.joinedPairs, st, slots_begin(c),
                         (const long long *)c.lb_err);
      HIP_CHECK(hipGetLastError());
    } else {
      const long long *nj = compact_flags_dev(c, joined, n, jidx, "joined");
      long long *part = (long long *)c.ws.get("jr_stats_part", 32 * (size_t)kOutBlocks);
      const unsigned ob = std::min(grid_for(n, 256), kOutBlocks);
      hipLaunchKernelGGL(k_refine_out, dim3(ob), dim3(256), 0, c.stream, n, kDev, pairs, o,
                         (const int *)jidx, nj, r.joinedPairs, part);
      HIP_CHECK(hipGetLastError());
      hipLaunchKernelGGL(k_refine_stats, dim3(1), dim3(256), 0, c.stream, n, kDev,
                         (const long long *)bOff, (const long long *)oOff,
                         (const long long *)part, (int)ob, st, slots_begin(c),
                         (const long long *)c.lb_err);
      HIP_CHECK(hipGetLastError());
    }
    long long v[kHostSlots];
    if (few) {
      slots_end(c, {st, st + 1, st + 2, st + 3, st + 4, st + 5, st + 6, st + 7}, v);
      avg = (double)v[kJoinStats] / (double)(in.B + in.O);
    } else {
      slots_end(c, {st, st + 1, st + 2, st + 3, st + 4, st + 5, st + 6}, v);
    }
    r.K = (long)v[0];
    if (v[0] > n) return false;
    if (v[1] <= capB && v[2] <= capO) {
      r.nbEdges = (long)v[1];
      r.noEdges = (long)v[2];
      r.pipNum = (long)v[3];
      r.within = (long)v[4];
      r.E = (long)v[5];
      r.hits = (long)v[6];
      break;
    }
    capB = std::max(capB, v[1]);
    capO = std::max(capO, v[2]);
  }
  // a candidate within the other polygon goes no further, so the CMF takes
  // the rest and the joined pairs are the within and the intersecting ones
  r.cmfCand = r.K - r.within;
  r.nJoined = r.within + r.hits;
  return true;
}

// Layers of at most this many polygons are joined without reading the
// candidate count back in between: the candidates get kOptFew (when the order
// takes one block) or kOptMid places per polygon.  More candidates than that
// cost the attempt's nearly empty launches; the polygons of larger layers,
// whose idle places would cost more than the 12 us of a read-back, are counted
// first.
constexpr long kOptPolys = 1L << 16;
constexpr long kOptFew = 8, kOptMid = 4;
static_assert(kOptFew * kFewPolys <= 1L << 15, "16-bit sums of k_refine_out_few");

long join_run(Context &c, const JoinInputs &in, int **counts_out, int **pairs_out,
              MbrSortView *sv, JoinRefine &r) {
  const long N = in.B + in.O;
  MbrOrder m;
  if (N <= 0) {
    refine(c, in, 0, nullptr, false, m.avg, nullptr, r);
    return 0;
  }
  mbr_order(c, in.B, in.O, in.bMBR, in.oMBR, in.bVNum, in.oVNum, m);
  int *counts = (int *)c.ws.get("mbr_counts", 4 * (size_t)N);
  long long *offs = (long long *)c.ws.get("mbr_offs", 8 * (size_t)(N + 1));
  if (!m.strips && N <= kOptPolys) {
    const long cap = (m.few ? kOptFew : kOptMid) * N;
    const long long *kDev = nullptr;
    mbr_candidates(c, m, cap, counts, offs, pairs_out, &kDev);
    if (!refine(c, in, cap, kDev, m.few, m.avg, *pairs_out, r)) {
      // counted by now: places for all, and the pairs once more
      const long K = r.K;
      if (m.few) scan_i32_to_i64(c, counts, offs, N);
      mbr_write(c, m, K, false, counts, offs, pairs_out);
      refine(c, in, K, nullptr, false, m.avg, *pairs_out, r);
    }
  } else {
    const long K = mbr_candidates(c, m, 0, counts, offs, pairs_out, nullptr);
    refine(c, in, K, nullptr, false, m.avg, *pairs_out, r);
  }
  *counts_out = counts;
  sv->perm = m.perm;
  sv->rank = m.rank;
  sv->n = 2 * N;
  return r.K;
}

// ------------------------------------------- single-stage launchers ----
void launch_get_cmbr(Context &c, long K, const int *pairs, const double *bMBR2,
                     const double *oMBR2, double *cmbr, int *pipFlag, signed char *pipType,
                     int *joinFlag) {
  if (K <= 0) return;
  LaunchTimer t(c, "get_cmbr");
  hipLaunchKernelGGL(k_get_cmbr, dim3(grid_for(K, 256)), dim3(256), 0, c.stream, K, pairs, bMBR2,
                     oMBR2, cmbr, pipFlag, pipType, joinFlag);
  HIP_CHECK(hipGetLastError());
}

void launch_pip(Context &c, long nCand, const int *cand, const int *pairs,
                const signed char *pipType, const double *bCoords, const long *bVPSNum,
                const double *oCoords, const long *oVPSNum, int *pipFlag, int *joinFlag) {
  if (nCand <= 0) return;
  LaunchTimer t(c, "pip");
  hipLaunchKernelGGL(k_pip, dim3(grid_for(nCand, 4)), dim3(256), 0, c.stream, nCand, cand, pairs,
                     pipType, (PolyRefs{bCoords, oCoords, nullptr, nullptr, bVPSNum, oVPSNum}),
                     pipFlag, joinFlag);
  HIP_CHECK(hipGetLastError());
}

void launch_cmf_count(Context &c, long nList, const int *list, const int *pairs,
                      const double *cmbr, const JoinInputs &in, int *joinFlag, int *bCount,
                      int *oCount) {
  if (nList <= 0) return;
  LaunchTimer t(c, "cmf_count");
  hipLaunchKernelGGL(k_cmf_count, dim3(grid_for(nList, 4)), dim3(256), 0, c.stream, nList, list,
                     pairs, cmbr, poly_refs(in), joinFlag, bCount, oCount);
  HIP_CHECK(hipGetLastError());
}

void launch_cmf_apply_short(Context &c, long nList, const int *list, const int *pairs,
                            const double *cmbr, const JoinInputs &in, const long long *bIncl,
                            const long long *oIncl, short *bEdge, short *oEdge) {
  if (nList <= 0) return;
  LaunchTimer t(c, "cmf_apply");
  hipLaunchKernelGGL(k_cmf_apply, dim3(grid_for(nList, 4)), dim3(256), 0, c.stream, nList, list,
                     pairs, cmbr, poly_refs(in), bIncl, oIncl, bEdge, oEdge);
  HIP_CHECK(hipGetLastError());
}

void launch_segjoin_short(Context &c, long nList, const int *list, const int *pairs,
                          const JoinInputs &in, const long long *bIncl, const long long *oIncl,
                          const short *bEdge, const short *oEdge, int *flagByList) {
  if (nList <= 0) return;
  LaunchTimer t(c, "segment_join");
  hipLaunchKernelGGL(k_segjoin, dim3(grid_for(nList, 4)), dim3(256), 0, c.stream, nList, list,
                     pairs, poly_refs(in), bIncl, oIncl, bEdge, oEdge, flagByList);
  HIP_CHECK(hipGetLastError());
}

}  // namespace gcmf
