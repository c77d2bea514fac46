// Ordered triangle counting on gfx950.
//
// Reference: OrderedCount (src/tc.cc:52-71).  Each triangle u > v > w is
// counted once, at its largest vertex u: for every neighbour v < u of u,
// the neighbours w of u below v that are also neighbours of v.  The graph
// must be undirected with sorted, duplicate-free lists (the builder
// guarantees it, tc.cc:31-35).  Whether to relabel by degree first (Hybrid /
// WorthRelabelling, tc.cc:75-100) is the caller's choice; the relabelled
// graph is counted the same way.
//
// Writing N+(x) for x's neighbours below x (a prefix of its sorted list) and
// d+(x) = |N+(x)|, the reference's count is the sum over the pairs
// (u, v in N+(u)) of |N+(u) & N+(v)| (every w of N+(v) is below v, so the
// reference's "w <= v" bound is implied).  Each pair's intersection is
// found by probing the shorter list into a set made of the longer: vertex x
// stages N+(x) once for its lower neighbours v with d+(v) <= d+(x) and its
// higher neighbours u with d+(u) < d+(x), so every pair is counted at
// exactly one of its ends.
//   * TcForward: d+(x) by binary search, and the work items per vertex span;
//   * TcItemScan / TcItemFill: (vertex, partner range) items in vertex order
//     (block prefix sums; no atomics), long lists and short lists apart;
//   * TcNarrow: the ids of N+(x) below 2^16 as 16-bit values, packed;
//   * TcCountLong: a block per item, d+(x) >= kLongList, the set in LDS bits;
//     where most ids are above 2^16, TcCountHash instead, the set in LDS hash
//     tables (and no TcNarrow);
//   * TcCountShort: a wavefront per item, the set a sorted LDS array.
// Counts are summed per block and added to 64 striped counters.
#include "gg_common.h"

namespace gg {
namespace {

constexpr int kBS = 256;
constexpr int kStripes = 64;
// Lists of this many entries or more are staged by a block as LDS bits; the
// rest (two thirds of the vertices but 0.1% of the probes on a degree-ordered
// Kronecker 21 graph) by a wavefront, without block barriers.
constexpr int kLongList = 32;
constexpr int kLongPartners = kBS;     // partners per long item, one per thread
constexpr int kShortPartners = kWave;  // partners per short item, one per lane
// The LDS set: ids below kExact have a bit of their own; larger ids share
// kFilter bits (id mod kFilter) and a hit there is checked against the list.
// kExact is where 16-bit ids end: on a degree-ordered graph nearly every
// probed id is a hub's (Kronecker 21: 98.6% below 2^16), so the probe streams
// are 2 B per entry.  12 KB of bits and 4 KB of partner lists leave eight
// 256-thread blocks, every wavefront slot, per CU.
constexpr int kExact = 1 << 16;
constexpr int kFilter = 1 << 15;
constexpr int kSetWords = (kExact + kFilter) / 32;
constexpr uint32_t kNoBit = kExact + kFilter;  // a bit that is never set
static_assert(kExact % kFilter == 0, "SetBit ORs the shared bit's index into kExact");
constexpr int kUnroll = 3;        // loads of a probe list in flight per lane,
constexpr int kLists = 4;         // for this many lists
constexpr int kCountBlocksPerCu = 64;
// TcCountHash: entries of N+(x) staged at a time, table slots (load factor
// <= 1/2) and list entries in flight per thread.
constexpr int kSetSlice = 2048;
constexpr int kTable = 2 * kSetSlice;
constexpr int kHashUnroll = 4;
constexpr unsigned kSliceWays = 4;  // blocks per item where a list can have several slices
// Share of the forward entries below kExact from which TcCountLong counts the
// long lists.  The whole call in ms, with it / with TcCountHash, by the share
// of entries at kExact or above: Kronecker 17, degree 64 (25%) 4.4 / 6.3, and
// degree 32 1.09 / 1.05; uniform 2^17, degree 256 (25%) 2.7 / 4.4; Kronecker
// 18 (55%) 3.6 / 2.1; uniform 2^18, degree 256 (56%) 9.0 / 8.5; Kronecker 19
// (77%) 11.9 / 5.0.
constexpr double kBitsShare = 0.5;

// d+(x), and how many of the entries are below kExact.
struct alignas(8) TcDegrees {
  int32_t d, low;
};

struct alignas(8) TcItem {
  int32_t x;   // the vertex whose lower neighbours are staged
  int32_t pb;  // first partner (index into x's list)
};

// Index of the first entry of the sorted range [b, e) that is >= x.
__device__ __forceinline__ int64_t LowerBound(const int32_t* dst, int64_t b, int64_t e, int32_t x) {
  while (b < e) {
    const int64_t m = b + ((e - b) >> 1);
    if (dst[m] < x)
      b = m + 1;
    else
      e = m;
  }
  return b;
}

// Items of a vertex of degree deg: its partners are its whole list.  A pair
// needs two entries in the staged list to hold a triangle.
__device__ __forceinline__ bool IsLong(int32_t dplus) { return dplus >= kLongList; }
__device__ __forceinline__ int64_t ItemsOf(int32_t dplus, int64_t deg) {
  if (dplus < 2) return 0;
  const int per = IsLong(dplus) ? kLongPartners : kShortPartners;
  return (deg + per - 1) / per;
}

// Vertices are split into gridDim.x contiguous spans; block b handles span b.
__device__ __forceinline__ void Span(int64_t n, int64_t& lo, int64_t& hi) {
  const int64_t per = (n + gridDim.x - 1) / gridDim.x;
  lo = per * blockIdx.x;
  hi = lo + per < n ? lo + per : n;
  if (lo > n) lo = n;
}

// What a span holds, for the prefix sums: long items, short items, 16-bit ids.
constexpr int kSpanKinds = 3;

// d+ of every vertex, and each span's totals (span_items[kSpanKinds * span]).
__global__ __launch_bounds__(kBS) void TcForward(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                 int64_t n, TcDegrees* __restrict__ fdeg,
                                                 unsigned long long* __restrict__ span_items) {
  __shared__ unsigned long long s_red[kBS / kWave];
  int64_t lo, hi;
  Span(n, lo, hi);
  unsigned long long nlong = 0, nshort = 0, nlow = 0;
  for (int64_t x = lo + threadIdx.x; x < hi; x += kBS) {
    const int64_t b = off[x], e = off[x + 1];
    const int64_t f = LowerBound(dst, b, e, static_cast<int32_t>(x));
    const int32_t d = static_cast<int32_t>(f - b);
    const int32_t low = x <= kExact ? d : static_cast<int32_t>(LowerBound(dst, b, f, kExact) - b);
    fdeg[x] = TcDegrees{d, low};
    (IsLong(d) ? nlong : nshort) += static_cast<unsigned long long>(ItemsOf(d, e - b));
    nlow += static_cast<unsigned long long>(low);
  }
  nlong = BlockSum<kBS>(nlong, s_red);
  nshort = BlockSum<kBS>(nshort, s_red);
  nlow = BlockSum<kBS>(nlow, s_red);
  if (threadIdx.x == 0) {
    span_items[kSpanKinds * blockIdx.x] = nlong;
    span_items[kSpanKinds * blockIdx.x + 1] = nshort;
    span_items[kSpanKinds * blockIdx.x + 2] = nlow;
  }
}

// Inclusive scan of one 64-bit value per thread of the block, and the total.
__device__ __forceinline__ unsigned long long BlockScan64(unsigned long long v, unsigned long long* total,
                                                          unsigned long long* sh) {
  const int lane = LaneId(), wid = threadIdx.x / kWave;
  for (int o = 1; o < kWave; o <<= 1) {
    const unsigned long long t = __shfl_up(v, o);
    if (lane >= o) v += t;
  }
  if (lane == kWave - 1) sh[wid] = v;
  __syncthreads();
  unsigned long long base = 0, tot = 0;
  for (int w = 0; w < kBS / kWave; w++) {
    if (w < wid) base += sh[w];
    tot += sh[w];
  }
  __syncthreads();
  *total = tot;
  return base + v;
}

// Exclusive prefixes of the span totals; the grand totals.  One block.
__global__ __launch_bounds__(kBS) void TcItemScan(unsigned long long* span_items, int spans,
                                                  unsigned long long* totals) {
  __shared__ unsigned long long s_scan[kBS / kWave];
  for (int kind = 0; kind < kSpanKinds; kind++) {
    unsigned long long base = 0;
    for (int t = 0; t < spans; t += kBS) {
      const int i = t + threadIdx.x;
      const unsigned long long c = i < spans ? span_items[kSpanKinds * i + kind] : 0;
      unsigned long long total;
      const unsigned long long inc = BlockScan64(c, &total, s_scan);
      if (i < spans) span_items[kSpanKinds * i + kind] = base + inc - c;
      base += total;
    }
    if (threadIdx.x == 0) totals[kind] = base;
  }
}

// The items, and (low_off non-null) every vertex's first 16-bit id.
__global__ __launch_bounds__(kBS) void TcItemFill(const int64_t* __restrict__ off,
                                                  const TcDegrees* __restrict__ fdeg, int64_t n,
                                                  const unsigned long long* __restrict__ span_base,
                                                  TcItem* __restrict__ longs, TcItem* __restrict__ shorts,
                                                  int64_t* __restrict__ low_off) {
  __shared__ unsigned long long s_scan[kBS / kWave];
  int64_t lo, hi;
  Span(n, lo, hi);
  const unsigned long long* at = span_base + kSpanKinds * blockIdx.x;
  unsigned long long base[kSpanKinds] = {at[0], at[1], at[2]};
  for (int64_t t = lo; t < hi; t += kBS) {
    const int64_t x = t + threadIdx.x;
    const TcDegrees f = x < hi ? fdeg[x] : TcDegrees{0, 0};
    const int64_t deg = x < hi ? off[x + 1] - off[x] : 0;
    unsigned long long total;
    for (int kind = 0; kind < 2; kind++) {
      const unsigned long long ni =
          IsLong(f.d) == (kind == 0) ? static_cast<unsigned long long>(ItemsOf(f.d, deg)) : 0;
      const unsigned long long pos = base[kind] + BlockScan64(ni, &total, s_scan) - ni;
      const int per = kind == 0 ? kLongPartners : kShortPartners;
      TcItem* items = kind == 0 ? longs : shorts;
      for (unsigned long long i = 0; i < ni; i++)
        items[pos + i] = TcItem{static_cast<int32_t>(x), static_cast<int32_t>(i) * per};
      base[kind] += total;
    }
    const unsigned long long nlow = static_cast<unsigned long long>(f.low);
    const unsigned long long pos = base[2] + BlockScan64(nlow, &total, s_scan) - nlow;
    if (low_off && x < hi) low_off[x] = static_cast<int64_t>(pos);
    base[2] += total;
  }
}

// The 16-bit ids: kNarrowLanes lanes per vertex.
constexpr int kNarrowLanes = 16;
__global__ __launch_bounds__(kBS) void TcNarrow(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                const TcDegrees* __restrict__ fdeg,
                                                const int64_t* __restrict__ low_off, int64_t n,
                                                uint16_t* __restrict__ low) {
  constexpr int kRows = kBS / kNarrowLanes;
  const int lane = threadIdx.x % kNarrowLanes;
  for (int64_t x = int64_t(blockIdx.x) * kRows + threadIdx.x / kNarrowLanes; x < n; x += int64_t(gridDim.x) * kRows) {
    const int32_t c = fdeg[x].low;
    if (c == 0) continue;
    const int64_t from = off[x], to = low_off[x];
    for (int32_t i = lane; i < c; i += kNarrowLanes) low[to + i] = static_cast<uint16_t>(dst[from + i]);
  }
}

// Partner j of x (x's list starts at xb, d = d+(x)): its degrees, zero when
// the pair is counted at the partner's end.
__device__ __forceinline__ TcDegrees Partner(const int32_t* dst, const TcDegrees* fdeg, int64_t xb, int64_t deg,
                                             int32_t d, int64_t j, int32_t& p) {
  p = 0;
  if (j >= deg) return TcDegrees{0, 0};
  p = dst[xb + j];
  const TcDegrees f = fdeg[p];
  return (j < d ? f.d <= d : f.d < d) ? f : TcDegrees{0, 0};
}

__device__ __forceinline__ void FlushCounts(unsigned long long count, unsigned long long probes,
                                            unsigned long long* counts, unsigned long long* s_red) {
  count = BlockSum<kBS>(count, s_red);
  probes = BlockSum<kBS>(probes, s_red);
  if (threadIdx.x == 0) {
    const int slot = 2 * (blockIdx.x & (kStripes - 1));
    if (count) atomicAdd(&counts[slot], count);
    if (probes) atomicAdd(&counts[slot + 1], probes);
  }
}

// The bit of id w: w itself below kExact, else its shared bit (which is never
// above w).
__device__ __forceinline__ uint32_t SetBit(uint32_t w) {
  const uint32_t shared = kExact | (w & (kFilter - 1));
  return w < shared ? w : shared;
}

// A 64-bit value that every lane of the wavefront holds, in scalar registers.
__device__ __forceinline__ int64_t Scalar(int64_t v) {
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// How many of a load's two ids (pair j of a list of n halves, the first
// `skip` of them before the list) are in the set.
__device__ __forceinline__ uint32_t PairHits(const uint32_t* set, uint32_t w, int j, int skip, int n) {
  uint32_t a = w & 0xFFFF, b = w >> 16;
  if (skip) a = j == 0 ? kNoBit : a;
  if (2 * (j | (kWave - 1)) + 2 > n) {  // uniform: the wavefront's last pair reaches past the list
    a = 2 * j < n ? a : kNoBit;
    b = 2 * j + 1 < n ? b : kNoBit;
  }
  return __builtin_amdgcn_ubfe(set[a >> 5], a, 1) + __builtin_amdgcn_ubfe(set[b >> 5], b, 1);
}

// Long lists.  The block sets N+(x)'s bits, lists the partners to probe, and
// each wavefront streams whole probe lists; afterwards only the words that
// were set are cleared.  A probe list's ids below kExact come packed, two per
// 4-byte load from an even position (the halves before and after the list
// look at kNoBit); its larger ids, read from dst, matter only when N+(x) has
// one too.  Bound by the probe streams, two thirds of whose lines miss L2
// (4.7 TB/s of misses).  Measured on a degree-ordered Kronecker 21 graph
// (4.84 G probes): 3.4 ms, 1.4 T probes/s.  Slices of 2048 entries in an LDS
// hash table, with a binary search for each probe's list, took 15.1 ms; these
// bits with 32-bit probe lists 5.1 ms; one 16-bit list at a time 4.4 ms.
__global__ __launch_bounds__(kBS) void TcCountLong(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                   const TcDegrees* __restrict__ fdeg,
                                                   const int64_t* __restrict__ low_off,
                                                   const uint16_t* __restrict__ low,
                                                   const TcItem* __restrict__ items, int64_t nitems,
                                                   unsigned long long* counts) {
  __shared__ uint32_t s_set[kSetWords + 1];
  __shared__ int64_t s_beg[kLongPartners];  // first packed id
  __shared__ int32_t s_low[kLongPartners];  // packed ids
  __shared__ int32_t s_p[kLongPartners];    // the partner
  __shared__ int s_scan[kBS / kWave];
  __shared__ unsigned long long s_red[kBS / kWave];
  const int tid = threadIdx.x, lane = LaneId(), wid = tid / kWave;
  unsigned long long total = 0, probes = 0;
  for (int i = tid; i <= kSetWords; i += kBS) s_set[i] = 0;
  __syncthreads();
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const TcItem item = items[it];
    const int64_t xb = off[item.x], deg = off[item.x + 1] - xb;
    const TcDegrees fx = fdeg[item.x];
    for (int32_t i = tid; i < fx.d; i += kBS) {
      const uint32_t b = SetBit(static_cast<uint32_t>(dst[xb + i]));
      atomicOr(&s_set[b >> 5], 1u << (b & 31));
    }
    int32_t p;
    const TcDegrees f = Partner(dst, fdeg, xb, deg, fx.d, int64_t(item.pb) + tid, p);
    int nlists = 0;
    const int at = BlockExclusiveScan<kBS>(f.d > 0, &nlists, s_scan);
    if (f.d > 0) {
      s_beg[at] = low_off[p];
      s_low[at] = f.low;
      s_p[at] = p;
      probes += static_cast<unsigned long long>(f.d);
    }
    __syncthreads();
    uint32_t count = 0;  // this lane's of one item
    for (int l0 = wid * kLists; l0 < nlists; l0 += kLists * (kBS / kWave)) {
      // kLists lists at a time, their first kUnroll loads each in flight together.
      const uint32_t* pairs[kLists];
      int skip[kLists], n[kLists];
      uint32_t w[kLists][kUnroll];
#pragma unroll
      for (int q = 0; q < kLists; q++) {
        const int l = l0 + q < nlists ? l0 + q : l0;
        // The list is the wavefront's: its place and length in scalar registers.
        const int64_t beg = Scalar(s_beg[l]);
        skip[q] = static_cast<int>(beg & 1);  // halves before the list
        n[q] = l0 + q < nlists ? __builtin_amdgcn_readfirstlane(s_low[l]) + skip[q] : 0;
        pairs[q] = reinterpret_cast<const uint32_t*>(low + (beg - skip[q]));
        // Pairs past the list read its last one, so that no load waits for a branch.
        const int last = n[q] > 0 ? (n[q] - 1) >> 1 : 0;
#pragma unroll
        for (int k = 0; k < kUnroll; k++) {
          const int j = k * kWave + lane;
          w[q][k] = pairs[q][static_cast<uint32_t>(j < last ? j : last)];
        }
      }
#pragma unroll
      for (int q = 0; q < kLists; q++) {
#pragma unroll
        for (int k = 0; k < kUnroll; k++)
          if (2 * k * kWave < n[q]) count += PairHits(s_set, w[q][k], k * kWave + lane, k == 0 ? skip[q] : 0, n[q]);
        for (int j0 = kUnroll * kWave; 2 * j0 < n[q]; j0 += kWave) {
          const int j = j0 + lane;
          const uint32_t v = 2 * j < n[q] ? pairs[q][static_cast<uint32_t>(j)] : 0;
          count += PairHits(s_set, v, j, 0, n[q]);
        }
      }
    }
    if (fx.low < fx.d) {
      for (int l = wid; l < nlists; l += kBS / kWave) {
        const int32_t pl = s_p[l];
        const int64_t pb = off[pl];
        const int32_t n = fdeg[pl].d;
        for (int32_t i = s_low[l] + lane; i < n; i += kWave) {
          const int32_t w = dst[pb + i];
          const uint32_t b = SetBit(static_cast<uint32_t>(w));
          if (!((s_set[b >> 5] >> (b & 31)) & 1)) continue;
          const int64_t q = LowerBound(dst, xb + fx.low, xb + fx.d, w);
          count += q < xb + fx.d && dst[q] == w;
        }
      }
    }
    total += count;
    __syncthreads();
    for (int32_t i = tid; i < fx.d; i += kBS) s_set[SetBit(static_cast<uint32_t>(dst[xb + i])) >> 5] = 0;
    __syncthreads();
  }
  FlushCounts(total, probes, counts, s_red);
}

// Long lists where most ids have no bit of their own.  The block stages N+(x)
// kSetSlice entries at a time in an LDS hash table and probes it with all of
// the item's lists, laid out as one flat range (block prefix sum, owner by
// binary search).  The slices of a list are shared out among gridDim.y blocks,
// or the largest hubs outlast the launch (Kronecker 18, the whole call: 3.1 ms
// with one block, 2.05 with four, 1.95 with eight).  A slice holds the sorted
// values [lo_w, hi_w]; probes outside skip the table.  In TcCountLong such ids
// share kFilter bits, one wavefront walks a list of them at a time, and where
// N+(x) fills the shared bits every probe is a binary search in memory:
// Kronecker 21 as uploaded (94% of the entries at 2^16 or above) 90.3 ms, 37.2
// here; uniform 2^22, degree 64 (97%) 36.4 and 14.5.
__device__ __forceinline__ uint32_t Hash(int32_t w, uint32_t mask) {
  return (static_cast<uint32_t>(w) * 2654435761u >> 7) & mask;
}

__global__ __launch_bounds__(kBS) void TcCountHash(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                   const TcDegrees* __restrict__ fdeg,
                                                   const TcItem* __restrict__ items, int64_t nitems,
                                                   unsigned long long* counts) {
  __shared__ int32_t table[kTable];
  __shared__ int64_t s_beg[kLongPartners];
  __shared__ int s_pre[kLongPartners];
  __shared__ int s_scan[kBS / kWave];
  __shared__ unsigned long long s_red[kBS / kWave];
  static_assert(kLongPartners == kBS, "a partner per thread");
  const int tid = threadIdx.x;
  unsigned long long count = 0, probes = 0;
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const TcItem item = items[it];
    const int64_t xb = off[item.x], deg = off[item.x + 1] - xb;
    const int32_t d = fdeg[item.x].d, sb0 = blockIdx.y * kSetSlice;
    if (sb0 >= d) continue;  // uniform: another block's
    int32_t p;
    const int len = Partner(dst, fdeg, xb, deg, d, int64_t(item.pb) + tid, p).d;
    s_beg[tid] = off[p];
    if (sb0 == 0) probes += static_cast<unsigned long long>(len);
    int total = 0;
    s_pre[tid] = BlockExclusiveScan<kBS>(len, &total, s_scan);
    for (int32_t sb = sb0; sb < d && total > 0; sb += gridDim.y * kSetSlice) {
      const int32_t slice = sb + kSetSlice < d ? kSetSlice : d - sb;
      uint32_t size = 64;
      while (size < 2u * static_cast<uint32_t>(slice)) size <<= 1;
      const uint32_t mask = size - 1;
      for (uint32_t i = tid; i < size; i += kBS) table[i] = -1;
      __syncthreads();
      for (int32_t i = tid; i < slice; i += kBS) {
        const int32_t w = dst[xb + sb + i];
        uint32_t h = Hash(w, mask);
        while (atomicCAS(&table[h], -1, w) != -1) h = (h + 1) & mask;
      }
      const int32_t lo_w = dst[xb + sb], hi_w = dst[xb + sb + slice - 1];
      __syncthreads();
      for (int j0 = 0; j0 < total; j0 += kBS * kHashUnroll) {
        int32_t w[kHashUnroll];
#pragma unroll
        for (int k = 0; k < kHashUnroll; k++) {
          const int j = j0 + k * kBS + tid;
          int at = 0;  // the last list starting at or before j: the one that owns it
#pragma unroll
          for (int step = kLongPartners / 2; step > 0; step >>= 1)
            if (s_pre[at + step] <= j) at += step;
          w[k] = j < total ? dst[s_beg[at] + (j - s_pre[at])] : -1;
        }
#pragma unroll
        for (int k = 0; k < kHashUnroll; k++) {
          if (w[k] < lo_w || w[k] > hi_w) continue;
          uint32_t h = Hash(w[k], mask);
          while (true) {
            const int32_t t = table[h];
            if (t == w[k]) {
              count++;
              break;
            }
            if (t < 0) break;
            h = (h + 1) & mask;
          }
        }
      }
      __syncthreads();
    }
    __syncthreads();  // (also where no list is probed: the next item rewrites s_pre)
  }
  FlushCounts(count, probes, counts, s_red);
}

// Short lists: the wavefront keeps N+(x) sorted in LDS; each lane walks one
// partner's list (shorter than kLongList) and binary-searches it there.
__global__ __launch_bounds__(kBS) void TcCountShort(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                    const TcDegrees* __restrict__ fdeg,
                                                    const TcItem* __restrict__ items, int64_t nitems,
                                                    unsigned long long* counts) {
  __shared__ int32_t s_list[kBS / kWave][kLongList];
  __shared__ unsigned long long s_red[kBS / kWave];
  const int lane = LaneId(), wid = threadIdx.x / kWave;
  int32_t* mine = s_list[wid];
  unsigned long long count = 0, probes = 0;
  const int64_t wave = int64_t(blockIdx.x) * (kBS / kWave) + wid;
  const int64_t nwaves = int64_t(gridDim.x) * (kBS / kWave);
  for (int64_t it = wave; it < nitems; it += nwaves) {
    const TcItem item = items[it];
    const int64_t xb = off[item.x], deg = off[item.x + 1] - xb;
    const int32_t d = fdeg[item.x].d;
    // Past the end: larger than any id, so the search below needs no bound.
    if (lane < kLongList) mine[lane] = lane < d ? dst[xb + lane] : INT32_MAX;
    int32_t p;
    const int len = Partner(dst, fdeg, xb, deg, d, int64_t(item.pb) + lane, p).d;
    const int64_t lbeg = off[p];
    WaveSync();
    for (int i = 0; i < len; i++) {
      const int32_t w = dst[lbeg + i];
      int at = 0;
#pragma unroll
      for (int step = kLongList / 2; step > 0; step >>= 1)
        if (mine[at + step - 1] < w) at += step;
      count += mine[at] == w;
    }
    probes += static_cast<unsigned long long>(len);
    WaveSync();
  }
  FlushCounts(count, probes, counts, s_red);
}

__global__ void TcClear(unsigned long long* counts) {
  for (int i = threadIdx.x; i < 2 * kStripes; i += blockDim.x) counts[i] = 0;
}

}  // namespace
}  // namespace gg

using namespace gg;

extern "C" int gg_tc(gg_graph* g, uint64_t* count, gg_stats* stats) {
  return Guard([&] {
    WallTimer wt;
    StatsReset(stats);
    GG_REQUIRE(g != nullptr, GG_EINVAL, "null graph");
    GG_REQUIRE(!g->weighted, GG_ENOTSUP, "TC needs an unweighted graph upload");
    GG_REQUIRE(!g->directed, GG_ENOTSUP, "TC needs an undirected graph");
    GG_REQUIRE(count != nullptr, GG_EINVAL, "null count output");
    GG_HIP(hipSetDevice(g->device));
    const int64_t n = g->n;
    hipStream_t st = g->stream;
    const int spans = static_cast<int>(GridFor(n, kBS * 2, g->cu_count * 8));
    // One buffer per phase: a fresh handle pays for every allocation (a
    // relabelled graph is counted once).  8-byte arrays first.
    TcDegrees* fdeg = g->Scratch<TcDegrees>("tc.work", n + 1 + 2 * kStripes + kSpanKinds * (1 + int64_t(spans)));
    unsigned long long* counts = reinterpret_cast<unsigned long long*>(fdeg + n + 1);
    unsigned long long* span_items = counts + 2 * kStripes + kSpanKinds;
    const dim3 blk(kBS);
    const double N = static_cast<double>(n);
    int64_t launches = 0;
    BeginTiming(g);
    Run(g, "tc_clear", 0, TcClear, dim3(1), blk, counts);
    Run(g, "tc_forward", 16.0 * N + 4.0 * N, TcForward, dim3(spans), blk, static_cast<const int64_t*>(g->out_off),
        static_cast<const int32_t*>(g->out_dst), n, fdeg, span_items);
    Run(g, "tc_items", 0, TcItemScan, dim3(1), blk, span_items, spans, counts + 2 * kStripes);
    launches += 3;
    unsigned long long* h = g->Pinned<unsigned long long>(2 * kStripes + kSpanKinds);
    GG_HIP(hipMemcpyAsync(h, counts + 2 * kStripes, kSpanKinds * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
    GG_HIP(hipStreamSynchronize(st));
    const int64_t nlong = static_cast<int64_t>(h[0]), nshort = static_cast<int64_t>(h[1]), nlow = static_cast<int64_t>(h[2]);
    // Entries are counted once per edge in the lists N+: half of all.
    // Items; then, for TcCountLong, the first 16-bit id of every vertex and the
    // ids, readable to the end of the pair after the last one.  Where these do
    // not fit beside the graph, TcCountHash does without.
    const int64_t nitems = nlong + nshort + 1, nids = n + 1 + (nlow + 3) / 4;
    TcItem* items = nullptr;
    if (nlow >= static_cast<int64_t>(kBitsShare * 0.5 * static_cast<double>(g->out_entries)))
      items = g->TryScratch<TcItem>("tc.items", nitems + nids);
    const bool bits = items != nullptr;
    if (!bits) items = g->Scratch<TcItem>("tc.items", nitems);
    TcItem* shorts = items + nlong;
    int64_t* low_off = bits ? reinterpret_cast<int64_t*>(shorts + nshort) : nullptr;
    uint16_t* low = bits ? reinterpret_cast<uint16_t*>(low_off + n + 1) : nullptr;
    Run(g, "tc_items", 24.0 * N + 8.0 * (nlong + nshort), TcItemFill, dim3(spans), blk,
        static_cast<const int64_t*>(g->out_off), static_cast<const TcDegrees*>(fdeg), n,
        static_cast<const unsigned long long*>(span_items), items, shorts, low_off);
    launches++;
    // Compulsory bytes: one pass over the CSR, 8 (n + 1) + 4 m.  The merge
    // work (probes, stats->edges_examined) is reported apart: its re-reads
    // of lists and LDS probes are not compulsory traffic.
    const double csr = 8.0 * (N + 1) + 4.0 * static_cast<double>(g->out_entries);
    const dim3 grid_long(GridFor(nlong, 1, g->cu_count * kCountBlocksPerCu));
    if (nlong > 0 && bits) {
      Run(g, "tc_narrow", 16.0 * N + 6.0 * nlow, TcNarrow, dim3(GridFor(n, kBS / kNarrowLanes, g->cu_count * 32)), blk,
          static_cast<const int64_t*>(g->out_off), static_cast<const int32_t*>(g->out_dst),
          static_cast<const TcDegrees*>(fdeg), static_cast<const int64_t*>(low_off), n, low);
      Run(g, "tc_count", csr, TcCountLong, grid_long, blk, static_cast<const int64_t*>(g->out_off),
          static_cast<const int32_t*>(g->out_dst), static_cast<const TcDegrees*>(fdeg),
          static_cast<const int64_t*>(low_off), static_cast<const uint16_t*>(low),
          static_cast<const TcItem*>(items), nlong, counts);
      launches += 2;
    } else if (nlong > 0) {
      const unsigned ways = g->max_degree > kSetSlice ? kSliceWays : 1;
      Run(g, "tc_count", csr, TcCountHash, dim3(grid_long.x, ways), blk, static_cast<const int64_t*>(g->out_off),
          static_cast<const int32_t*>(g->out_dst), static_cast<const TcDegrees*>(fdeg),
          static_cast<const TcItem*>(items), nlong, counts);
      launches++;
    }
    if (nshort > 0) {
      Run(g, "tc_count_short", 0, TcCountShort, dim3(GridFor(nshort, kBS / kWave, g->cu_count * kCountBlocksPerCu)),
          blk, static_cast<const int64_t*>(g->out_off), static_cast<const int32_t*>(g->out_dst),
          static_cast<const TcDegrees*>(fdeg), static_cast<const TcItem*>(shorts), nshort, counts);
      launches++;
    }
    GG_HIP(hipGetLastError());
    GG_HIP(hipMemcpyAsync(h, counts, sizeof(unsigned long long) * 2 * kStripes, hipMemcpyDeviceToHost, st));
    GG_HIP(hipStreamSynchronize(st));
    unsigned long long total = 0, probes = 0;
    for (int i = 0; i < kStripes; i++) {
      total += h[2 * i];
      probes += h[2 * i + 1];
    }
    FinishTiming(g, stats, wt);
    g->ws.Spare("tc.items");
    *count = total;
    if (stats) {
      stats->total_ms = wt.ms();
      stats->iterations = 1;
      stats->edges_examined = static_cast<int64_t>(probes);
      stats->launches = launches;
    }
  });
}
