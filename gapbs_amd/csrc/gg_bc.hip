// Brandes betweenness centrality on gfx950.
//
// Reference: Brandes / PBFS (src/bc.cc:51-150).  Kept, per root:
//   * a level-synchronous top-down BFS claiming depths with a compare-and-
//     swap (bc.cc:65-77); the reached vertices in BFS order with per-level
//     boundaries (the reference's queue and depth_index, bc.cc:56-87);
//   * shortest-path counts sigma in double (bc.cc:47, 78-80);
//   * successors of u are the out-neighbours one level deeper -- the
//     reference records them in an edge bitmap during the BFS (bc.cc:76),
//     here they are re-derived from depths, as its verifier does
//     (bc.cc:207);
//   * for depths from the deepest down to 0 (the root included, whose own
//     dependency is added to its score): delta_u = sum over successors v of
//     (sigma_u / sigma_v) * (1 + delta_v), the double term added into a
//     float delta_u (bc.cc:123-136), then score_u += delta_u;
//   * after all roots, every score divided by the largest (bc.cc:141-148).
// GPU design:
//   * discovery expands the level with gg_expand.h and appends the next
//     level to the same queue through an LDS-staged queue;
//   * sigma is pulled: each newly discovered vertex sums sigma over its
//     in-neighbours at the previous level (no floating-point atomics; the
//     sums are exact integers below 2^53, so the order does not matter);
//   * the sigma pull runs one thread per vertex below 64 in-edges; longer
//     lists are cut into chunks of 1024, a wavefront each, whose sums are
//     combined with one double atomic per chunk;
//   * whether a neighbour lies on the next (or previous) level is one bit of
//     that level's bitmap, which stays in L2, rather than its depth; a
//     vertex's path count and dependency share a 16-byte record, one
//     transaction per successor;
//   * delta runs one thread per vertex below 64 edges and one wavefront or
//     block per vertex above: 64 successor terms are computed at a time and
//     folded into the accumulator as if in successor order (FoldTerms), so
//     every vertex's delta is rounded exactly as the reference rounds it;
//   * GG_BC_FP32: the reference's float arithmetic throughout (its verifier
//     allows only FLT_EPSILON); GG_BC_FP32_KAHAN: float dependencies and
//     scores, each per-vertex dependency sum and each score sum over roots
//     carrying a float compensation term; GG_BC_FP64: double dependencies
//     and scores.
#include <algorithm>
#include <type_traits>

#include "gg_common.h"
#include "gg_expand.h"

namespace gg {
namespace {

constexpr int kBS = 256;
constexpr int kQueueCap = 2048;
constexpr int kStripes = 64;
constexpr int64_t kWaveEdges = 64;   // vertices with this many edges use a wavefront ...
constexpr int kSigmaChunkLog2 = 10;    // ... per this many, as a power of two (sigma pull)
// The same two where levels are discovered one by one, or where the longer
// chunk list does not fit.
constexpr int64_t kFewWaveEdges = 256;
constexpr int kFewChunkLog2 = 12;
constexpr int64_t kKindsVertices = int64_t(1) << 20;  // up to this many BcLevelKinds looks at every search
constexpr int kThreadUnroll = 4;     // edges in flight per thread below that
constexpr int kBcWaveUnroll = 4;     // 64-edge runs per wavefront step
constexpr int32_t kSideLevel = 65536;  // vertices of a level from which BcDeltaWave takes a stream too
constexpr int64_t kBcHubEdges = 4096;  // ... and with this many, a block (BcDeltaHub)
constexpr int kBcHubProducers = 15;
constexpr int kBcHubUnroll = 4;  // 64-edge runs per producer wavefront and round
constexpr int kBcHubGrid = 2;    // BcDeltaHub blocks per CU
constexpr int kBcHubBS = (kBcHubProducers + 1) * kWave;

// A vertex's path count and dependency, read together by its predecessors.
template <class T>
struct alignas(16) BcNode {
  double sigma;
  T delta;
};
static_assert(sizeof(BcNode<float>) == sizeof(BcNode<double>), "one buffer serves both precisions");

// Tells whether a vertex lies on one level: its bit in the level's bitmap,
// or, without bitmaps (deep traversals), its depth.
struct OnLevel {
  const uint32_t* bits;
  const int32_t* depth;
  int32_t level;
  __device__ __forceinline__ bool operator()(int32_t v) const {
    return bits ? (bits[v >> 5] >> (v & 31)) & 1 : depth[v] == level;
  }
};

struct BcCounters {
  int32_t tail;     // queue length (all levels so far)
  int32_t nchunks;  // discovery chunks
  int32_t nred;     // sigma reduction chunks
  int32_t nwave;    // delta: vertices handed to the wavefront kernel
  int32_t nhub;     // delta: vertices handed to the hub kernel
  int32_t hub_next; // BcDeltaHub: next hub list entry to take
  unsigned long long examined[kStripes];
};

__device__ __forceinline__ int32_t Load(const int32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class T>
__global__ __launch_bounds__(kBS) void BcResetSource(int32_t* __restrict__ depth, int64_t n, int32_t src,
                                                     BcNode<T>* __restrict__ node, int32_t* __restrict__ queue,
                                                     BcCounters* c) {
  for (int64_t i = blockIdx.x * int64_t(kBS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBS)
    depth[i] = i == src ? 0 : -1;
  if (blockIdx.x == 0) {
    if (threadIdx.x < kStripes) c->examined[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
      node[src].sigma = 1.0;
      queue[0] = src;
      c->tail = 1;
      c->nchunks = 0;
      c->nred = 0;
      c->nwave = 0;
      c->nhub = 0;
      c->hub_next = 0;
    }
  }
}

struct DiscoverVisit {
  const int32_t* dst;
  int32_t* depth;
  int32_t next_depth;
  LdsQueue<kQueueCap>* lq;
  int32_t* queue;
  int32_t* tail;
  int most = 0;  // queue entries at most
  __device__ __forceinline__ void Visit(const int32_t (&)[kExpandEdges], const int32_t (&)[kExpandEdges],
                                        const int64_t (&e)[kExpandEdges], const bool (&valid)[kExpandEdges]) {
    int32_t v[kExpandEdges];
    bool won[kExpandEdges];
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++) v[k] = dst[e[k]];
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++) won[k] = Load(&depth[v[k]]) == -1;
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++)
      won[k] = valid[k] && won[k] && atomicCAS(&depth[v[k]], -1, next_depth) == -1;
    LdsQueuePushMany(*lq, won, v, queue, tail);
  }
  __device__ __forceinline__ void StepEnd(int edges) { LdsQueueMakeRoom(*lq, queue, tail, most, edges); }
};

// Claims the next level's vertices and appends them to the queue.
__global__ __launch_bounds__(kBS) void BcDiscover(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                  int32_t* depth, int32_t* queue, int32_t qb, int32_t qn,
                                                  int32_t next_depth, BcCounters* c, EdgeChunk* chunks) {
  __shared__ ExpandShared sh;
  __shared__ LdsQueue<kQueueCap> lq;
  __shared__ unsigned long long s_red[kBS / kWave];
  LdsQueueInit(lq);
  DiscoverVisit visit{dst, depth, next_depth, &lq, queue, &c->tail};
  unsigned long long ex = 0;
  for (int64_t tile = int64_t(blockIdx.x) * kBS; tile < qn; tile += int64_t(gridDim.x) * kBS) {
    const int64_t i = tile + threadIdx.x;
    int64_t beg = 0, end = 0;
    if (i < qn) {
      const int32_t u = queue[qb + i];
      beg = off[u];
      end = off[u + 1];
      ex += static_cast<unsigned long long>(end - beg);
    }
    ExpandTile<FrontierCut>(sh, 0, 0, beg, end, visit, chunks, &c->nchunks, FrontierCut::MinFor(qn));
  }
  LdsQueueFlush(lq, queue, &c->tail);
  ex = BlockSum<kBS>(ex, s_red);
  if (threadIdx.x == 0 && ex) atomicAdd(&c->examined[blockIdx.x & (kStripes - 1)], ex);
}

__global__ __launch_bounds__(kBS) void BcDiscoverChunks(const int32_t* __restrict__ dst, int32_t* depth,
                                                        int32_t* queue, int32_t next_depth, BcCounters* c,
                                                        const EdgeChunk* chunks) {
  __shared__ LdsQueue<kQueueCap> lq;
  LdsQueueInit(lq);
  DiscoverVisit visit{dst, depth, next_depth, &lq, queue, &c->tail};
  ExpandChunks<FrontierCut>(chunks, c->nchunks, visit);
  LdsQueueFlush(lq, queue, &c->tail);
}

// sigma[v] for the new level: sum of sigma over in-neighbours one level up.
// Vertices with wave_min in-edges or more are listed in chunks of 2^chunk_log2
// edges (one reservation per wavefront) and summed by BcSigmaChunks; those of
// several chunks start from sigma = 0 here.
template <class T>
__global__ __launch_bounds__(kBS) void BcSigma(const int64_t* __restrict__ in_off, const int32_t* __restrict__ in_dst,
                                               OnLevel prev, BcNode<T>* node, const int32_t* __restrict__ queue,
                                               int32_t qb, int32_t qn, EdgeChunk* __restrict__ chunks, int64_t wave_min,
                                               int chunk_log2, BcCounters* c, unsigned long long* work) {
  __shared__ unsigned long long s_red[kBS / kWave];
  const int64_t chunk = int64_t(1) << chunk_log2;
  unsigned long long ent = 0, mat = 0;
  for (int64_t base = int64_t(blockIdx.x) * kBS; base < qn; base += int64_t(gridDim.x) * kBS) {
    const int64_t i = base + threadIdx.x;
    int32_t v = 0;
    int64_t b = 0, e = 0;
    if (i < qn) {
      v = queue[qb + i];
      b = in_off[v];
      e = in_off[v + 1];
    }
    const int nc = e - b >= wave_min ? static_cast<int>((e - b + chunk - 1) >> chunk_log2) : 0;
    const int upto = WaveInclusiveScan(nc);
    const int total = __builtin_amdgcn_readlane(upto, kWave - 1);
    if (total) {
      int at = 0;
      if (LaneId() == 0) at = atomicAdd(&c->nred, total);
      at = __builtin_amdgcn_readfirstlane(at) + upto - nc;
      for (int k = 0; k < nc; k++) {
        const int64_t cb = b + k * chunk;
        // payload: whether the chunk is the whole list (its sum is stored)
        chunks[at + k] = EdgeChunk{cb, cb + chunk < e ? cb + chunk : e, v, nc == 1};
      }
      if (nc > 1) node[v].sigma = 0.0;
    }
    if (nc || i >= qn) continue;
    double s = 0.0;
    for (int64_t k = b; k < e; k += kThreadUnroll) {
      int32_t u[kThreadUnroll];
      bool has[kThreadUnroll];
      double x[kThreadUnroll];
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) u[j] = in_dst[k + j < e ? k + j : k];
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) has[j] = prev(u[j]) && k + j < e;
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) x[j] = has[j] ? node[u[j]].sigma : 0.0;
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) {
        s += x[j];
        mat += has[j];
      }
    }
    ent += static_cast<unsigned long long>(e - b);
    node[v].sigma = s;
  }
  WorkAdd(work, BlockSum<kBS>(ent, s_red), BlockSum<kBS>(mat, s_red));
}

// One wavefront per chunk.
template <class T>
__global__ __launch_bounds__(kBS) void BcSigmaChunks(const int32_t* __restrict__ in_dst, OnLevel prev,
                                                     BcNode<T>* node, const EdgeChunk* __restrict__ chunks,
                                                     const BcCounters* c, unsigned long long* work) {
  __shared__ unsigned long long s_cnt[kBS / kWave];
  const int lane = LaneId();
  const int32_t nc = c->nred;
  const int32_t wave = blockIdx.x * (kBS / kWave) + threadIdx.x / kWave;
  const int32_t nwaves = gridDim.x * (kBS / kWave);
  unsigned long long ent = 0, mat = 0;
  for (int32_t ci = wave; ci < nc; ci += nwaves) {
    const EdgeChunk ch = chunks[ci];
    double s = 0.0;
    for (int64_t k = ch.beg + lane; k - lane < ch.end; k += kWave * kThreadUnroll) {
      int32_t u[kThreadUnroll];
      bool has[kThreadUnroll];
      double x[kThreadUnroll];
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) u[j] = in_dst[k + j * kWave < ch.end ? k + j * kWave : ch.beg];
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) has[j] = prev(u[j]) && k + j * kWave < ch.end;
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) x[j] = has[j] ? node[u[j]].sigma : 0.0;
#pragma unroll
      for (int j = 0; j < kThreadUnroll; j++) {
        s += x[j];
        mat += has[j];
      }
    }
    s = WaveSum(s);
    if (lane == 0) {
      ent += static_cast<unsigned long long>(ch.end - ch.beg);
      if (ch.payload)
        node[ch.u].sigma = s;
      else if (s != 0.0)
        atomicAdd(&node[ch.u].sigma, s);
    }
  }
  WorkAdd(work, BlockSum<kBS>(ent, s_cnt), BlockSum<kBS>(mat, s_cnt));
}

// delta for one level, the reference's way: a double term added into a
// float (or double) accumulator, in successor order.
__device__ __forceinline__ double DeltaTerm(double sig_u, double sig_v, float delta_v) {
  return __dmul_rn(__ddiv_rn(sig_u, sig_v), static_cast<double>(__fadd_rn(1.0f, delta_v)));
}
__device__ __forceinline__ double DeltaTerm(double sig_u, double sig_v, double delta_v) {
  return __dmul_rn(__ddiv_rn(sig_u, sig_v), __dadd_rn(1.0, delta_v));
}
// Per-vertex dependency accumulators.  RefAcc rounds like the reference (a
// double term added into a float, or double, total); KahanAcc keeps a float
// sum plus a float compensation, fed with each double term split into a
// float head and a float tail.
template <class T>
struct RefAcc {
  T v;
  __device__ __forceinline__ static RefAcc Zero() { return RefAcc{T(0)}; }
  __device__ __forceinline__ void Add(double t) { v = static_cast<T>(__dadd_rn(static_cast<double>(v), t)); }
  __device__ __forceinline__ T Value() const { return v; }
};

struct KahanAcc {
  float s, c;
  __device__ __forceinline__ static KahanAcc Zero() { return KahanAcc{0.0f, 0.0f}; }
  __device__ __forceinline__ void AddF(float x) {  // Neumaier
    const float t = __fadd_rn(s, x);
    const float e = fabsf(s) >= fabsf(x) ? __fadd_rn(__fsub_rn(s, t), x) : __fadd_rn(__fsub_rn(x, t), s);
    c = __fadd_rn(c, e);
    s = t;
  }
  __device__ __forceinline__ void Add(double t) {
    const float hi = static_cast<float>(t);
    const float lo = static_cast<float>(__dsub_rn(t, static_cast<double>(hi)));
    AddF(hi);
    c = __fadd_rn(c, lo);
  }
  __device__ __forceinline__ float Value() const { return __fadd_rn(s, c); }
};

template <class T, bool kKahan>
struct AccFor {
  using Type = RefAcc<T>;
};
template <>
struct AccFor<float, true> {
  using Type = KahanAcc;
};

// Inclusive scan within the wavefront by data-parallel moves (no LDS).
__device__ __forceinline__ int WaveScanDpp(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31
  return v;
}

__device__ __forceinline__ double ReadLane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Adds the terms of the lanes in m (wave-uniform) to acc (wave-uniform) in
// lane order, one after another.
template <class Acc>
__device__ __forceinline__ void FoldTerms(Acc& acc, double term, uint64_t m) {
  while (m) {
    const int j = __builtin_ctzll(m);
    acc.Add(ReadLane(term, j));
    m &= m - 1;
  }
}

// The same sum, bit for bit, without the chain of widen / add / round per
// term.  While the total stays in one binade [2^E, 2^(E+1)) every rounding
// is to the same grid g = 2^(E-23), on which the total already lies, so
// adding t moves it by t rounded to the grid, whatever the total: the terms
// become whole numbers of grid steps and add up in any order.  That fails
// only for a term within 2^-30 g of a grid midpoint (there the rounding to
// double before the one to float, or the tie rule, decides) or once the
// binade is left, so a lane takes part when its term is at least 2^-28 g
// from a midpoint and every lane before it (inclusive scan) stays below
// 2^24 steps; the first lane that does not is added the reference's way and
// the rest tried again with the new binade.  Terms are not negative; NaN and
// infinities compare false and go the reference's way.  A hub's total
// crosses a binade only as often as it doubles.  Measured on Kronecker 22,
// 4 roots: the wavefront kernel 8.7 to 3.9 ms,
// the hub kernel 10.5 to 6.5 ms with hubs from 4096 instead of 16384
// successors.
template <>
__device__ __forceinline__ void FoldTerms(RefAcc<float>& acc, double term, uint64_t m) {
  const int lane = LaneId();
  constexpr int kSteps = 1 << 24;
  while (m) {
    const uint32_t bits = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(__float_as_int(acc.v)));
    const uint32_t e = bits >> 23;  // the sign is 0
    if (e != 0 && e < 255) {
      const double x = term * __hiloint2double(static_cast<int>(1023 + 150 - e) << 20, 0);  // exact: / g
      const double r = rint(x);
      const bool whole = fabs(x - r) < 0.5 - 0x1p-28 && r < 0x1p24;
      const bool in = (m >> lane) & 1;
      const int sum = WaveScanDpp(in ? (whole ? static_cast<int>(r) : kSteps) : 0);
      const int start = static_cast<int>((bits & 0x7FFFFF) | 0x800000);
      const uint64_t past = __ballot(in && start + sum >= kSteps);
      const uint64_t take = past ? m & ((past & -past) - 1) : m;
      if (take) {
        const int last = 63 - __builtin_clzll(take);
        const uint32_t steps = static_cast<uint32_t>(start + __builtin_amdgcn_readlane(sum, last));
        acc.v = __uint_as_float((e << 23) | (steps & 0x7FFFFF));
        m &= ~take;
      }
      if (!m) break;
    }
    acc.Add(ReadLane(term, __builtin_ctzll(m)));
    m &= m - 1;
  }
}

// K runs of up to 64 terms, run by run.
template <int K, class Acc>
__device__ __forceinline__ void FoldRuns(Acc& acc, const double (&term)[K], const uint64_t (&m)[K]) {
#pragma unroll
  for (int k = 0; k < K; k++) FoldTerms(acc, term[k], m[k]);
}

// The same: all K runs in one sum when none of their terms is near a midpoint
// and the binade holds them all, else run by run.  A row's fold is a chain of
// wavefront scans, which bounds the hub kernel; one scan per K runs with K = 4
// (the hub kernel before: two runs a round) took Brandes from four roots of a
// Kronecker 22 graph from 12.7 to 11.0 ms.
template <int K>
__device__ __forceinline__ void FoldRuns(RefAcc<float>& acc, const double (&term)[K], const uint64_t (&m)[K]) {
  const int lane = LaneId();
  constexpr int kSteps = 1 << 24;
  uint64_t any = 0;
#pragma unroll
  for (int k = 0; k < K; k++) any |= m[k];
  if (!any) return;
  const uint32_t bits = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(__float_as_int(acc.v)));
  const uint32_t e = bits >> 23;
  if (e != 0 && e < 255) {
    const double scale = __hiloint2double(static_cast<int>(1023 + 150 - e) << 20, 0);
    int mine = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const double x = term[k] * scale, r = rint(x);
      const bool whole = fabs(x - r) < 0.5 - 0x1p-28 && r < 0x1p24;
      if ((m[k] >> lane) & 1) mine += whole ? static_cast<int>(r) : kSteps;
    }
    // (a lane's sum is cut at kSteps, so that 64 of them fit an int)
    const int sum = WaveScanDpp(mine < kSteps ? mine : kSteps);
    const int steps = static_cast<int>((bits & 0x7FFFFF) | 0x800000) + __builtin_amdgcn_readlane(sum, kWave - 1);
    if (steps < kSteps) {
      acc.v = __uint_as_float((e << 23) | (static_cast<uint32_t>(steps) & 0x7FFFFF));
      return;
    }
  }
#pragma unroll
  for (int k = 0; k < K; k++) FoldTerms(acc, term[k], m[k]);
}

// score += delta: plain, or with a Kahan compensation term (float only).
template <bool kKahan>
__device__ __forceinline__ void AddScore(float* score, float* comp, int32_t u, float d) {
  if (kKahan) {
    const float y = __fsub_rn(d, comp[u]);
    const float s = score[u];
    const float t = __fadd_rn(s, y);
    comp[u] = __fsub_rn(__fsub_rn(t, s), y);
    score[u] = t;
  } else {
    score[u] = __fadd_rn(score[u], d);
  }
}
template <bool kKahan>
__device__ __forceinline__ void AddScore(double* score, double*, int32_t u, double d) {
  score[u] = __dadd_rn(score[u], d);
}

// The level's vertices of kWaveEdges or more edges, listed for BcDeltaWave, and
// those of kBcHubEdges or more for BcDeltaHub, each in the queue's order within
// a block's tile.  Listed ahead of the level's work, not in BcDelta, so that the
// three dependency kernels run side by side (Kronecker 22, 4 roots: 11.0 ms
// with the lists made by BcDelta, 10.1 so); one reservation per tile, because
// additions to a list's one counter follow each other at 12 ns.
constexpr int kListRows = 8;
constexpr int kListTile = kBS * kListRows;
__global__ __launch_bounds__(kBS) void BcDeltaLists(const int64_t* __restrict__ off, const int32_t* __restrict__ queue,
                                                    int32_t qb, int32_t qn, int32_t* __restrict__ wave_list,
                                                    int32_t* __restrict__ hub_list, BcCounters* c) {
  constexpr int kWaves = kBS / kWave;
  __shared__ int32_t s_at[2][kWaves];  // a wavefront's entries in each list, then their place
  const int lane = LaneId(), wid = threadIdx.x / kWave;
  for (int64_t base = int64_t(blockIdx.x) * kListTile; base < qn; base += int64_t(gridDim.x) * kListTile) {
    const int64_t first = base + wid * (kListRows * kWave) + lane;
    int32_t u[kListRows];
    int64_t d[kListRows];
#pragma unroll
    for (int j = 0; j < kListRows; j++) u[j] = queue[qb + (first + j * kWave < qn ? first + j * kWave : qn - 1)];
#pragma unroll
    for (int j = 0; j < kListRows; j++) d[j] = off[u[j] + 1] - off[u[j]];
    int nw = 0, nh = 0;
#pragma unroll
    for (int j = 0; j < kListRows; j++) {
      if (first + j * kWave >= qn) d[j] = 0;
      nw += __popcll(__ballot(d[j] >= kWaveEdges && d[j] < kBcHubEdges));
      nh += __popcll(__ballot(d[j] >= kBcHubEdges));
    }
    if (lane == 0) {
      s_at[0][wid] = nw;
      s_at[1][wid] = nh;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      int32_t sum = 0;
      for (int w = 0; w < kWaves; w++) sum += s_at[threadIdx.x][w];
      int32_t at = sum ? atomicAdd(threadIdx.x ? &c->nhub : &c->nwave, sum) : 0;
      for (int w = 0; w < kWaves; w++) {
        const int32_t mine = s_at[threadIdx.x][w];
        s_at[threadIdx.x][w] = at;
        at += mine;
      }
    }
    __syncthreads();
    int32_t aw = s_at[0][wid], ah = s_at[1][wid];
#pragma unroll
    for (int j = 0; j < kListRows; j++) {
      const bool wave = d[j] >= kWaveEdges && d[j] < kBcHubEdges, hub = d[j] >= kBcHubEdges;
      const uint64_t mw = __ballot(wave), mh = __ballot(hub);
      if (wave) wave_list[aw + __popcll(LanesBelow(mw))] = u[j];
      if (hub) hub_list[ah + __popcll(LanesBelow(mh))] = u[j];
      aw += __popcll(mw);
      ah += __popcll(mh);
    }
    __syncthreads();  // read by all before the next tile's counts
  }
}

// Thread per vertex below kWaveEdges edges (the others: BcDeltaLists).
template <class T, bool kKahan>
__global__ __launch_bounds__(kBS) void BcDelta(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                               OnLevel next, BcNode<T>* node, T* __restrict__ score,
                                               T* __restrict__ comp, const int32_t* __restrict__ queue, int32_t qb,
                                               int32_t qn, unsigned long long* work) {
  __shared__ unsigned long long s_red[kBS / kWave];
  unsigned long long ent = 0, mat = 0;
  for (int64_t base = int64_t(blockIdx.x) * kBS; base < qn; base += int64_t(gridDim.x) * kBS) {
    const int64_t i = base + threadIdx.x;
    if (i < qn) {
      const int32_t u = queue[qb + i];
      const int64_t b = off[u], e = off[u + 1];
      if (e - b < kWaveEdges) {
        const double su = node[u].sigma;
        typename AccFor<T, kKahan>::Type acc = AccFor<T, kKahan>::Type::Zero();
        for (int64_t k = b; k < e; k += kThreadUnroll) {
          int32_t v[kThreadUnroll];
          bool has[kThreadUnroll];
          BcNode<T> x[kThreadUnroll];
#pragma unroll
          for (int j = 0; j < kThreadUnroll; j++) v[j] = dst[k + j < e ? k + j : k];
#pragma unroll
          for (int j = 0; j < kThreadUnroll; j++) has[j] = next(v[j]) && k + j < e;
#pragma unroll
          for (int j = 0; j < kThreadUnroll; j++) x[j] = node[has[j] ? v[j] : u];
#pragma unroll
          for (int j = 0; j < kThreadUnroll; j++) {
            if (!has[j]) continue;
            acc.Add(DeltaTerm(su, x[j].sigma, x[j].delta));
            mat++;
          }
        }
        ent += static_cast<unsigned long long>(e - b);
        const T d = acc.Value();
        node[u].delta = d;
        AddScore<kKahan>(score, comp, u, d);
      }
    }
  }
  WorkAdd(work, BlockSum<kBS>(ent, s_red), BlockSum<kBS>(mat, s_red));
}

// One wavefront per listed vertex: 64 successor terms computed at once,
// folded into the accumulator in edge order.
template <class T, bool kKahan>
__global__ __launch_bounds__(kBS) void BcDeltaWave(const int64_t* __restrict__ off, const int32_t* __restrict__ dst,
                                                   OnLevel next, BcNode<T>* node, T* __restrict__ score,
                                                   T* __restrict__ comp, const int32_t* __restrict__ wave_list,
                                                   const BcCounters* c, unsigned long long* work) {
  __shared__ unsigned long long s_red[kBS / kWave];
  const int lane = LaneId();
  unsigned long long ent = 0, mat = 0;  // lane 0's
  const int32_t nw = c->nwave;
  const int64_t wave = (int64_t(blockIdx.x) * kBS + threadIdx.x) / kWave;
  const int64_t nwaves = int64_t(gridDim.x) * (kBS / kWave);
  for (int64_t i = wave; i < nw; i += nwaves) {
    const int32_t u = wave_list[i];
    const int64_t b = off[u], e = off[u + 1];
    const double su = node[u].sigma;
    typename AccFor<T, kKahan>::Type acc = AccFor<T, kKahan>::Type::Zero();
    for (int64_t base = b; base < e; base += kWave * kBcWaveUnroll) {
      // kBcWaveUnroll runs of 64 edges, their loads issued together.
      int32_t v[kBcWaveUnroll];
      bool has[kBcWaveUnroll];
      BcNode<T> x[kBcWaveUnroll];
      double term[kBcWaveUnroll];
      const int64_t k = base + lane;
#pragma unroll
      for (int r = 0; r < kBcWaveUnroll; r++) v[r] = dst[k + r * kWave < e ? k + r * kWave : b];
#pragma unroll
      for (int r = 0; r < kBcWaveUnroll; r++) has[r] = next(v[r]) && k + r * kWave < e;
      // (a lane without a successor reads the vertex's own record)
#pragma unroll
      for (int r = 0; r < kBcWaveUnroll; r++) x[r] = node[has[r] ? v[r] : u];
#pragma unroll
      for (int r = 0; r < kBcWaveUnroll; r++) term[r] = DeltaTerm(su, x[r].sigma, x[r].delta);
      uint64_t m[kBcWaveUnroll];
#pragma unroll
      for (int r = 0; r < kBcWaveUnroll; r++) {
        m[r] = __ballot(has[r]);
        if (lane == 0) mat += static_cast<unsigned long long>(__popcll(m[r]));
      }
      FoldRuns(acc, term, m);
    }
    if (lane == 0) {
      ent += static_cast<unsigned long long>(e - b);
      const T d = acc.Value();
      node[u].delta = d;
      AddScore<kKahan>(score, comp, u, d);
    }
  }
  WorkAdd(work, BlockSum<kBS>(ent, s_red), BlockSum<kBS>(mat, s_red));
}

// The hub list's vertices (at least kBcHubEdges successors), one block each:
// per round, producer wavefront p computes the terms of 64 kBcHubUnroll
// consecutive edges (from b + 64 kBcHubUnroll (round kBcHubProducers + p))
// and packs the matched ones, in edge order, into one half of an LDS double
// buffer; the last wavefront folds the previous round's terms in edge
// order (FoldTerms).  Same terms, same order, same arithmetic as
// BcDeltaWave.  Two blocks fit a CU, of the compensated variant one (68
// registers; held to 64 it took the same time: Kronecker 22, 4 roots, 22.1 and
// 22.3 ms).  Blocks take hubs from a counter, so a block held by a large hub
// takes no others meanwhile (the list follows the level's queue, which on a
// degree-ordered layout runs roughly from the largest hub down).
template <class T, bool kKahan>
__global__ __launch_bounds__(kBcHubBS) void BcDeltaHub(const int64_t* __restrict__ off,
                                                       const int32_t* __restrict__ dst,
                                                       OnLevel next, BcNode<T>* node, T* __restrict__ score,
                                                       T* __restrict__ comp, const int32_t* __restrict__ hub_list,
                                                       BcCounters* c, unsigned long long* work) {
  __shared__ double terms[2][kBcHubProducers][kWave * kBcHubUnroll];
  __shared__ int counts[2][kBcHubProducers];
  __shared__ int32_t s_take;
  __shared__ unsigned long long s_red[kBcHubBS / kWave];
  const int lane = LaneId(), wid = threadIdx.x / kWave;
  unsigned long long ent = 0, mat = 0;  // lane 0 of each producer's
  const int32_t nh = c->nhub;
  constexpr int64_t kRound = int64_t(kBcHubProducers) * kWave * kBcHubUnroll;
  for (;;) {
    if (threadIdx.x == 0) s_take = atomicAdd(&c->hub_next, 1);
    __syncthreads();
    const int32_t i = s_take;
    __syncthreads();  // read by all before the next take overwrites it
    if (i >= nh) break;
    const int32_t u = hub_list[i];
    const int64_t b = off[u], e = off[u + 1];
    const double su = node[u].sigma;
    typename AccFor<T, kKahan>::Type acc = AccFor<T, kKahan>::Type::Zero();
    const int64_t rounds = (e - b + kRound - 1) / kRound;
    // kBcHubUnroll consecutive runs of 64 edges per producer and round; the
    // successor ids of the next round are loaded while this one's records
    // are on their way.
    const int64_t mine = b + int64_t(wid) * (kWave * kBcHubUnroll) + lane;
    auto id_at = [&](int64_t round, int r) {
      const int64_t at = mine + round * kRound + r * kWave;
      return dst[at < e ? at : b];
    };
    int32_t v[kBcHubUnroll];
    if (wid < kBcHubProducers) {
#pragma unroll
      for (int r = 0; r < kBcHubUnroll; r++) v[r] = id_at(0, r);
    }
    for (int64_t k = 0; k <= rounds; k++) {
      if (wid < kBcHubProducers) {
        if (k < rounds) {
          const int64_t k0 = mine + k * kRound;
          bool has[kBcHubUnroll];
          BcNode<T> x[kBcHubUnroll];
#pragma unroll
          for (int r = 0; r < kBcHubUnroll; r++) has[r] = next(v[r]) && k0 + r * kWave < e;
          // (a lane without a successor reads the hub's own record)
#pragma unroll
          for (int r = 0; r < kBcHubUnroll; r++) x[r] = node[has[r] ? v[r] : u];
#pragma unroll
          for (int r = 0; r < kBcHubUnroll; r++) v[r] = id_at(k + 1, r);
          double term[kBcHubUnroll];
#pragma unroll
          for (int r = 0; r < kBcHubUnroll; r++) term[r] = DeltaTerm(su, x[r].sigma, x[r].delta);
          int pos = 0;
#pragma unroll
          for (int r = 0; r < kBcHubUnroll; r++) {
            const uint64_t m = __ballot(has[r]);
            if (has[r]) terms[k & 1][wid][pos + __popcll(LanesBelow(m))] = term[r];
            pos += __popcll(m);
            const uint64_t in = __ballot(k0 + r * kWave < e);
            if (lane == 0) ent += static_cast<unsigned long long>(__popcll(in));
          }
          if (lane == 0) {
            counts[k & 1][wid] = pos;
            mat += static_cast<unsigned long long>(pos);
          }
        }
      } else if (k >= 1) {
        const int h = (k - 1) & 1;
        for (int p = 0; p < kBcHubProducers; p++) {
          const int cnt = counts[h][p];
          if constexpr (std::is_same_v<decltype(acc), RefAcc<float>>) {
            double t[kBcHubUnroll];
            uint64_t m[kBcHubUnroll];
#pragma unroll
            for (int r = 0; r < kBcHubUnroll; r++) {
              const int left = cnt - r * kWave;  // of this run
              t[r] = lane < left ? terms[h][p][r * kWave + lane] : 0.0;
              m[r] = left >= kWave ? ~uint64_t(0) : left > 0 ? (uint64_t(1) << left) - 1 : 0;
            }
            FoldRuns(acc, t, m);
          } else {
            // One after another: every lane reads the same term, eight ahead
            // of the ordered fold (taking them lane by lane from a register
            // costs several times an addition each).
            int j = 0;
            for (; j + 8 <= cnt; j += 8) {
              double t[8];
#pragma unroll
              for (int q = 0; q < 8; q++) t[q] = terms[h][p][j + q];
#pragma unroll
              for (int q = 0; q < 8; q++) acc.Add(t[q]);
            }
            for (; j < cnt; j++) acc.Add(terms[h][p][j]);
          }
        }
      }
      __syncthreads();
    }
    if (wid == kBcHubProducers && lane == 0) {
      const T d = acc.Value();
      node[u].delta = d;
      AddScore<kKahan>(score, comp, u, d);
    }
  }
  WorkAdd(work, BlockSum<kBcHubBS>(ent, s_red), BlockSum<kBcHubBS>(mat, s_red));
}


// ---- discovery by DOBFS ------------------------------------------------------
//
// Depths are unique, so the direction-optimizing BFS (RunDobfs) gives the
// levels of the reference's top-down PBFS at a fraction of the edges.  The
// vertices are then bucketed by depth into the queue layout the sigma and
// dependency passes read (level d at queue[bounds[d], bounds[d + 1]); the
// order inside a level does not affect any result).
constexpr int kBucketLevels = 4096;  // deeper traversals use the top-down discovery
constexpr int kBitLevels = 32;       // up to this many levels also get bitmaps (n / 8 bytes each)
// Vertices per block of the bucketing: enough blocks to fill the chip, few
// enough that their reservations on a level's one cursor stay cheap.
inline int64_t BucketChunk(int64_t n) { return std::max<int64_t>(4096, ((n >> 11) + 255) / 256 * 256); }

// For each level d present among the wavefront's 64 depths: op(d, its lanes).
template <class Op>
__device__ __forceinline__ void ForLevels(int32_t d, int nlev, Op op) {
  uint64_t left = __ballot(d >= 0 && d < nlev);
  while (left) {
    const int32_t ld = __builtin_amdgcn_readlane(d, __builtin_ctzll(left));
    const uint64_t m = __ballot(d == ld);
    op(ld, m);
    left &= ~m;
  }
}

// Vertices per level, and (bits non-null, zeroed before) each level's bitmap
// of nwords words.  A wavefront takes 64 consecutive vertices and counts a
// level's by ballot: an LDS atomic per vertex put most of a wavefront on one
// address (76 us on Kronecker 22 against 30 us, with the bitmaps).
__global__ __launch_bounds__(kBS) void BcLevelCount(const int32_t* __restrict__ depth, int64_t n, int nlev,
                                                    int32_t* counts, uint64_t* __restrict__ bits) {
  __shared__ int32_t h[kBucketLevels];
  for (int i = threadIdx.x; i < nlev; i += kBS) h[i] = 0;
  __syncthreads();
  const int lane = LaneId();
  const int64_t nwords = (n + 63) >> 6;
  for (int64_t w = (int64_t(blockIdx.x) * kBS + threadIdx.x) / kWave; w < nwords;
       w += int64_t(gridDim.x) * (kBS / kWave)) {
    const int64_t v = w * 64 + lane;
    ForLevels(v < n ? depth[v] : -1, nlev, [&](int32_t d, uint64_t m) {
      if (lane != 0) return;
      atomicAdd(&h[d], __popcll(m));
      if (bits) bits[d * nwords + w] = m;
    });
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nlev; i += kBS)
    if (h[i]) atomicAdd(&counts[i], h[i]);
}

// cursor[d] starts at bounds[d]; each block (`chunk` vertices) reserves its
// ranges with one atomic per level it holds.  Kronecker 22: 113 us with 64
// blocks of 65536 vertices, 28 us with 2048.
__global__ __launch_bounds__(kBS) void BcLevelScatter(const int32_t* __restrict__ depth, int64_t n, int64_t chunk,
                                                      int nlev, int32_t* cursor, int32_t* __restrict__ queue) {
  __shared__ int32_t h[kBucketLevels];
  for (int i = threadIdx.x; i < nlev; i += kBS) h[i] = 0;
  __syncthreads();
  const int lane = LaneId();
  const int64_t lo = int64_t(blockIdx.x) * chunk;
  const int64_t hi = lo + chunk < n ? lo + chunk : n;
  for (int64_t b = lo + (threadIdx.x - lane); b < hi; b += kBS)
    ForLevels(b + lane < hi ? depth[b + lane] : -1, nlev, [&](int32_t d, uint64_t m) {
      if (lane == 0) atomicAdd(&h[d], __popcll(m));
    });
  __syncthreads();
  for (int i = threadIdx.x; i < nlev; i += kBS)
    if (h[i]) h[i] = atomicAdd(&cursor[i], h[i]);
  __syncthreads();
  for (int64_t b = lo + (threadIdx.x - lane); b < hi; b += kBS)
    ForLevels(b + lane < hi ? depth[b + lane] : -1, nlev, [&](int32_t d, uint64_t m) {
      int at = 0;
      if (lane == 0) at = atomicAdd(&h[d], __popcll(m));
      at = __builtin_amdgcn_readfirstlane(at);
      if ((m >> lane) & 1) queue[at + __popcll(LanesBelow(m))] = static_cast<int32_t>(b + lane);
    });
}

// Zeroes the level counts and bitmap words.  (There can be one level more
// than the grid has threads: the search's last, empty step counts as one.)
__global__ __launch_bounds__(kBS) void BcLevelClear(int32_t* __restrict__ counts, int nlev,
                                                    uint64_t* __restrict__ bits, int64_t words) {
  const int64_t i0 = blockIdx.x * int64_t(kBS) + threadIdx.x, stride = int64_t(gridDim.x) * kBS;
  for (int64_t i = i0; i < nlev; i += stride) counts[i] = 0;
  for (int64_t i = i0; i < words; i += stride) bits[i] = 0;
}

// Which levels hold vertices for the wavefront and hub kernels, one bit per
// level and kind: in-lists of in_min entries or more (kLongIn), out-lists of
// kWaveEdges (kWaveOut) and of kBcHubEdges (kHubOut) or more.  Most such
// vertices find their bit set already; collected per block in LDS, unless the
// levels are too many, since on few levels every block would want the same words.
enum { kLongIn, kWaveOut, kHubOut, kLevelKinds };
constexpr int kKindWords = kLevelKinds * kBucketLevels / 32;
__device__ __forceinline__ void SetBits(uint32_t* word, uint32_t bits) {
  if (bits & ~*word) atomicOr(word, bits);
}
__global__ __launch_bounds__(kBS) void BcLevelKinds(const int32_t* __restrict__ depth,
                                                    const int64_t* __restrict__ out_off,
                                                    const int64_t* __restrict__ in_off, int64_t n, int64_t in_min,
                                                    uint32_t* flags, int words) {
  __shared__ uint32_t s_flags[kKindWords];
  const bool few = kLevelKinds * words <= kKindWords;
  for (int i = threadIdx.x; few && i < kLevelKinds * words; i += kBS) s_flags[i] = 0;
  __syncthreads();
  for (int64_t v = blockIdx.x * int64_t(kBS) + threadIdx.x; v < n; v += int64_t(gridDim.x) * kBS) {
    const int32_t d = depth[v];
    const int64_t out = out_off[v + 1] - out_off[v], in = in_off[v + 1] - in_off[v];
    if (d < 0) continue;
    const bool has[kLevelKinds] = {in >= in_min, out >= kWaveEdges && out < kBcHubEdges, out >= kBcHubEdges};
#pragma unroll
    for (int kind = 0; kind < kLevelKinds; kind++) {
      if (!has[kind]) continue;
      const int at = kind * words + (d >> 5);
      if (few)
        SetBits(&s_flags[at], 1u << (d & 31));
      else
        SetBits(&flags[at], 1u << (d & 31));
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; few && i < kLevelKinds * words; i += kBS)
    if (s_flags[i]) SetBits(&flags[i], s_flags[i]);
}

__global__ __launch_bounds__(kBS) void BcClearReduce(BcCounters* c) {
  if (threadIdx.x == 0) {
    c->nred = 0;
    c->nwave = 0;
    c->nhub = 0;
    c->hub_next = 0;
  }
}

enum { kMailTail, kMailExamined, kMailValues };

__global__ __launch_bounds__(kBS) void BcPublish(BcCounters* c, unsigned long long* mb, unsigned long long seq) {
  if (threadIdx.x == 0) {
    unsigned long long vals[kMailValues];
    unsigned long long ex = 0;
    for (int i = 0; i < kStripes; i++) {
      ex += c->examined[i];
      c->examined[i] = 0;
    }
    vals[kMailTail] = static_cast<unsigned long long>(c->tail);
    vals[kMailExamined] = ex;
    c->nchunks = 0;
    c->nred = 0;
    MailPost(mb, vals, kMailValues, seq);
  }
}

template <class T>
__global__ __launch_bounds__(kBS) void BcZero(T* __restrict__ score, T* __restrict__ comp, int64_t n) {
  for (int64_t i = blockIdx.x * int64_t(kBS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBS) {
    score[i] = 0;
    if (comp) comp[i] = 0;
  }
}

// Largest score (scores are >= 0, so their bit patterns order like the
// values), then every score divided by it (bc.cc:141-148).
template <class T>
__device__ __forceinline__ T Final(const T* score, const T* comp, int64_t i);
template <>
__device__ __forceinline__ float Final(const float* score, const float* comp, int64_t i) {
  return __fadd_rn(score[i], -comp[i]);
}
template <>
__device__ __forceinline__ double Final(const double* score, const double*, int64_t i) {
  return score[i];
}

template <class T>
__global__ __launch_bounds__(kBS) void BcMax(const T* __restrict__ score, const T* __restrict__ comp, int64_t n,
                                             unsigned long long* max_bits) {
  __shared__ double s_max[kBS / kWave];
  double m = 0.0;
  for (int64_t i = blockIdx.x * int64_t(kBS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBS) {
    const double v = static_cast<double>(Final(score, comp, i));
    m = v > m ? v : m;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_xor(m, o);
    m = t > m ? t : m;
  }
  if (LaneId() == 0) s_max[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 0; w < kBS / kWave; w++) m = s_max[w] > m ? s_max[w] : m;
    atomicMax(max_bits, static_cast<unsigned long long>(__double_as_longlong(m)));
  }
}

template <class T>
__global__ __launch_bounds__(kBS) void BcNormalize(const T* __restrict__ score, const T* __restrict__ comp,
                                                   int64_t n, const unsigned long long* max_bits,
                                                   float* __restrict__ out) {
  const double mx = __longlong_as_double(static_cast<long long>(*max_bits));
  const T biggest = static_cast<T>(mx);
  for (int64_t i = blockIdx.x * int64_t(kBS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBS)
    out[i] = static_cast<float>(Final(score, comp, i) / biggest);
}

template <class T, bool kKahan>
void RunBrandes(gg_graph* g, const int32_t* roots, int k, float* scores_out, gg_stats* stats,
                const WallTimer& wt) {
  const int64_t n = g->n;
  hipStream_t st = g->stream;
  const char* tag = sizeof(T) == 4 ? "32" : "64";
  int32_t* depth = g->Scratch<int32_t>("bc.depth", n);
  BcNode<T>* node = g->Scratch<BcNode<T>>("bc.node", n);
  int32_t* queue = g->Scratch<int32_t>("bc.queue", n + 64);
  T* score = g->Scratch<T>((std::string("bc.score") + tag).c_str(), n);
  T* comp = sizeof(T) == 4 ? g->Scratch<T>("bc.comp32", n) : nullptr;  // zero unless kKahan
  int32_t* wave_list = g->Scratch<int32_t>("bc.wave_list", n + 64);
  // A vertex with kBcHubEdges successors owns that many list entries.
  int32_t* hub_list = g->Scratch<int32_t>("bc.hub_list", g->out_entries / kBcHubEdges + 64);
  float* out32 = reinterpret_cast<float*>(wave_list);  // written when no level is left to list
  unsigned long long* max_bits = g->Scratch<unsigned long long>("bc.max", 1);
  BcCounters* dc = g->Scratch<BcCounters>("bc.ctr", 1);
  // Work counters (entries read, matched in-neighbours / successors) per
  // kernel kind, for the profiled byte credits.
  enum { kWSigma, kWSigmaChunks, kWDelta, kWDeltaWave, kWDeltaHub, kWKinds };
  unsigned long long* work = g->Scratch<unsigned long long>("bc.work", kWKinds * kWorkCounters);
  int rec[kWKinds] = {-1, -1, -1, -1, -1};
  auto note = [&](int kind, int idx) {
    if (rec[kind] < 0) rec[kind] = idx;
  };
  auto wk = [&](int kind) { return work + kind * kWorkCounters; };
  // Vertices per level, after the words of BcLevelKinds.
  int32_t* lvl_counts = g->Scratch<int32_t>("bc.level_counts", kKindWords + kBucketLevels);
  int32_t* lvl_cursor = g->Scratch<int32_t>("bc.level_cursor", kBucketLevels);
  std::vector<int32_t> h_counts(kKindWords + kBucketLevels);
  const int64_t entries = g->out_entries > g->in_entries ? g->out_entries : g->in_entries;
  const bool hubs = g->max_degree >= FrontierCut::kMin, longs = g->max_degree >= kWaveEdges;
  // Chunks of a level's discovery, then of its sigma pull: for the latter, the
  // sum of ceil(d / 2^log2) over the vertices of wave_min in-edges or more.
  auto chunk_bound = [&](int64_t wave_min, int log2) {
    return std::max(FrontierCut::Bound(n, entries), (entries >> log2) + std::min(n, entries / wave_min) + 2);
  };
  EdgeChunk* chunks = longs ? g->TryScratch<EdgeChunk>("bc.chunks", chunk_bound(kWaveEdges, kSigmaChunkLog2)) : nullptr;
  const bool many_chunks = chunks != nullptr;
  if (longs && !many_chunks) chunks = g->Scratch<EdgeChunk>("bc.chunks", chunk_bound(kFewWaveEdges, kFewChunkLog2));
  const int64_t nwords = (n + 63) / 64;
  const dim3 blk(kBS);
  const dim3 grid_n(GridFor(n, kBS, g->cu_count * 32));
  const dim3 grid_c(g->cu_count * 4);
  const double N = static_cast<double>(n);
  int64_t launches = 0, levels_total = 0, reached_total = 0, examined_total = 0;
  unsigned long long mail[kMailValues];

  // Dependencies are summed in each vertex's uploaded list order (the
  // reference's successor order), also on a degree-ordered handle.
  const int32_t* fold_dst = UploadOrderLists(g);
  BeginTiming(g);
  Run(g, "bc_zero", N * sizeof(T) * 2, BcZero<T>, grid_n, blk, score, comp, n);
  Run(g, "bc_zero", 0, WorkClear, dim3(1), dim3(256), work, kWKinds * kWorkCounters);
  launches += 2;
  std::vector<int32_t> bounds;
  for (int r = 0; r < k; r++) {
    Run(g, "bc_reset_source", 4 * N, BcResetSource<T>, grid_n, blk, depth, n, roots[r], node, queue, dc);
    launches++;
    bounds.assign(1, 0);
    bounds.push_back(1);
    int32_t level = 0;
    // Forward, by DOBFS and bucketing when the levels fit the buckets.
    const BfsRun br = RunDobfs(g, roots[r], 15, 18, depth);
    launches += br.launches;
    examined_total += br.examined;
    const int nlev = static_cast<int>(br.td + br.bu + 1);
    bool bucketed = false;
    uint64_t* bits = nullptr;
    auto on_level = [&](int32_t d) {
      return OnLevel{bits ? reinterpret_cast<const uint32_t*>(bits + d * nwords) : nullptr, depth, d};
    };
    // Cut-offs of the sigma pull; level by level, with no kinds known ahead,
    // those that give fewer launches.
    const bool buckets = nlev <= kBucketLevels;
    const bool short_waves = buckets && many_chunks;
    const int64_t wave_min = short_waves ? kWaveEdges : kFewWaveEdges;
    const int chunk_log2 = short_waves ? kSigmaChunkLog2 : kFewChunkLog2;
    // Whether level d may hold vertices of a kind (BcLevelKinds, from depths of
    // nlev levels).  A kernel left out of a level that holds none saves its
    // launch and, on the side streams, a fork and join: a 500 x 500 lattice
    // (999 levels) with one vertex of 5000 leaves takes 29.7 ms, 71.4 with all
    // kernels at every level; Kronecker 20, 4 roots, 4.7 and 5.3.
    const int kind_words = (nlev + 31) / 32;
    std::vector<uint32_t> kinds;
    auto holds = [&](int kind, int32_t d) {
      return kinds.empty() || ((kinds[kind * kind_words + (d >> 5)] >> (d & 31)) & 1);
    };
    auto mark_kinds = [&](int32_t* flags) {
      Run(g, "bc_level_kinds", 20.0 * N, BcLevelKinds, dim3(GridFor(n, kBS, g->cu_count * 8)), blk, static_cast<const int32_t*>(depth),
          static_cast<const int64_t*>(g->out_off), static_cast<const int64_t*>(g->in_off), n, wave_min,
          reinterpret_cast<uint32_t*>(flags), kind_words);
      launches++;
    };
    // Path counts of level d, queue[nb, nb + nn).
    auto pull_sigma = [&](int32_t d, int32_t nb, int32_t nn) {
      note(kWSigma, Run(g, "bc_sigma", 20.0 * nn, BcSigma<T>, dim3(GridFor(nn, kBS, g->cu_count * 16)), blk,
                        static_cast<const int64_t*>(g->in_off), static_cast<const int32_t*>(g->in_dst),
                        on_level(d - 1), node, static_cast<const int32_t*>(queue), nb, nn, chunks, wave_min, chunk_log2, dc,
                        wk(kWSigma)));
      launches++;
      if (g->max_degree >= wave_min && holds(kLongIn, d)) {
        note(kWSigmaChunks,
             Run(g, "bc_sigma_chunks", 0, BcSigmaChunks<T>, dim3(g->cu_count * 8), blk,
                 static_cast<const int32_t*>(g->in_dst), on_level(d - 1), node,
                 static_cast<const EdgeChunk*>(chunks), static_cast<const BcCounters*>(dc), wk(kWSigmaChunks)));
        Run(g, "bc_clear_reduce", 0, BcClearReduce, dim3(1), blk, dc);
        launches += 2;
      }
    };
    if (buckets) {
      // (in steps of eight levels; where they do not fit, depths are tested)
      if (nlev <= kBitLevels) bits = g->TryScratch<uint64_t>("bc.level_bits", (nlev + 7) / 8 * 8 * nwords);
      const int64_t chunk = BucketChunk(n);
      const dim3 grid_b(GridFor(n, static_cast<int>(chunk)));
      // (a large graph's few levels are worth no look at every degree)
      const int nkinds = longs && (n <= kKindsVertices || nlev > kBitLevels) ? kLevelKinds * kind_words : 0;
      int32_t* counts = lvl_counts + nkinds;
      Run(g, "bc_level_count", 0, BcLevelClear, grid_n, blk, lvl_counts, nkinds + nlev, bits,
          bits ? nlev * nwords : 0);
      Run(g, "bc_level_count", 4 * N, BcLevelCount, dim3(GridFor(nwords, kBS / kWave, g->cu_count * 8)), blk,
          static_cast<const int32_t*>(depth), n, nlev, counts, bits);
      launches++;
      if (nkinds) mark_kinds(lvl_counts);
      GG_HIP(hipMemcpyAsync(h_counts.data(), lvl_counts, sizeof(int32_t) * (nkinds + nlev), hipMemcpyDeviceToHost, st));
      GG_HIP(hipStreamSynchronize(st));
      kinds.assign(h_counts.begin(), h_counts.begin() + nkinds);
      const int32_t* level_size = h_counts.data() + nkinds;
      int last = 0;
      for (int d = 0; d < nlev; d++)
        if (level_size[d]) last = d;
      bounds.assign(1, 0);
      for (int d = 0; d <= last; d++) bounds.push_back(bounds.back() + level_size[d]);
      GG_HIP(hipMemcpyAsync(lvl_cursor, bounds.data(), sizeof(int32_t) * (last + 1), hipMemcpyHostToDevice, st));
      Run(g, "bc_level_scatter", 8 * N, BcLevelScatter, grid_b, blk, static_cast<const int32_t*>(depth), n, chunk, last + 1,
          lvl_cursor, queue);
      launches += 2;
      for (int32_t d = 1; d <= last; d++) pull_sigma(d, bounds[d], bounds[d + 1] - bounds[d]);
      level = last;
      bucketed = true;
    } else {
      // Too deep for the buckets: the top-down discovery, level by level
      // (the BFS above only cost its own time; reset its outputs).
      Run(g, "bc_reset_source", 4 * N, BcResetSource<T>, grid_n, blk, depth, n, roots[r], node, queue, dc);
      launches++;
    }
    while (!bucketed) {
      const int32_t qb = bounds[bounds.size() - 2], qn = bounds.back() - qb;
      const int idx = Run(g, "bc_discover", 8.0 * qn, BcDiscover, dim3(GridFor(qn, kBS, g->cu_count * 8)), blk,
                          static_cast<const int64_t*>(g->out_off), static_cast<const int32_t*>(g->out_dst),
                          depth, queue, qb, qn, level + 1, dc,
                          hubs ? chunks : static_cast<EdgeChunk*>(nullptr));
      launches++;
      if (hubs) {
        Run(g, "bc_discover_chunks", 0, BcDiscoverChunks, grid_c, blk, static_cast<const int32_t*>(g->out_dst),
            depth, queue, level + 1, dc, static_cast<const EdgeChunk*>(chunks));
        launches++;
      }
      const unsigned long long seq = MailNext(g);
      Run(g, "bc_publish", 0, BcPublish, dim3(1), blk, dc, g->mail_dev, seq);
      launches++;
      MailWait(g, seq, mail, kMailValues);
      CreditBytes(g, idx, 4.0 * mail[kMailExamined]);
      examined_total += static_cast<int64_t>(mail[kMailExamined]);
      const int32_t tail = static_cast<int32_t>(mail[kMailTail]);
      if (tail == bounds.back()) break;
      const int32_t nb = bounds.back(), nn = tail - nb;
      bounds.push_back(tail);
      pull_sigma(level + 1, nb, nn);
      level++;
    }
    if (!bucketed && longs) {
      int32_t* flags = wave_list;  // not listed in yet; 3 bits a level, at most n + 1 levels
      Run(g, "bc_level_kinds", 0, BcLevelClear, dim3(GridFor(kLevelKinds * kind_words, kBS)), blk, flags,
          kLevelKinds * kind_words, static_cast<uint64_t*>(nullptr), int64_t(0));
      mark_kinds(flags);
      launches++;
      kinds.resize(kLevelKinds * kind_words);
      GG_HIP(hipMemcpyAsync(kinds.data(), flags, sizeof(uint32_t) * kinds.size(), hipMemcpyDeviceToHost, st));
      GG_HIP(hipStreamSynchronize(st));
    }
    reached_total += bounds.back();
    levels_total += level + 1;
    // Backward: deepest level first; delta of level d reads level d + 1.
    for (int32_t d = level; d >= 0; d--) {
      const int32_t qb = bounds[d], qn = bounds[d + 1] - bounds[d];
      // (below the deepest level nothing is marked: no bitmap, no depth)
      const OnLevel next = d < level ? on_level(d + 1) : OnLevel{nullptr, depth, d + 1};
      auto delta = [&] {
        note(kWDelta, Run(g, "bc_delta", (16.0 + 2 * sizeof(T) + 8.0) * qn, BcDelta<T, kKahan>,
                          dim3(GridFor(qn, kBS, g->cu_count * 16)), blk, static_cast<const int64_t*>(g->out_off),
                          fold_dst, next, node, score, comp, static_cast<const int32_t*>(queue), qb, qn, wk(kWDelta)));
        launches++;
      };
      const bool waves = longs && holds(kWaveOut, d), hubs = g->max_degree >= kBcHubEdges && holds(kHubOut, d);
      if (!waves && !hubs) {
        delta();
      } else {
        // The three kernels write disjoint vertices and only read level
        // d + 1, so they run on three streams; all finish before the lists
        // are cleared.  A level below kSideLevel is over sooner than the
        // second fork costs.
        const bool side_wave = waves && qn >= kSideLevel;
        Run(g, "bc_delta_lists", 0, BcDeltaLists, dim3(GridFor(qn, kListTile, g->cu_count * 8)), blk,
            static_cast<const int64_t*>(g->out_off), static_cast<const int32_t*>(queue), qb, qn, wave_list, hub_list,
            dc);
        if (hubs || side_wave) {
          EnsureSideStream(g);
          GG_HIP(hipEventRecord(g->ev_fork, st));
        }
        if (hubs) {
          GG_HIP(hipStreamWaitEvent(g->side, g->ev_fork, 0));
          note(kWDeltaHub,
               RunOn(g, g->side, "bc_delta_hub", 0, BcDeltaHub<T, kKahan>, dim3(g->cu_count * kBcHubGrid), dim3(kBcHubBS),
                     static_cast<const int64_t*>(g->out_off), fold_dst, next, node, score, comp,
                     static_cast<const int32_t*>(hub_list), dc, wk(kWDeltaHub)));
          GG_HIP(hipEventRecord(g->ev_join, g->side));
          launches++;
        }
        if (waves) {
          hipStream_t ws = side_wave ? g->side2 : st;
          if (side_wave) GG_HIP(hipStreamWaitEvent(ws, g->ev_fork, 0));
          note(kWDeltaWave,
               RunOn(g, ws, "bc_delta_wave", 0, BcDeltaWave<T, kKahan>,
                     dim3(GridFor(qn, kBS / kWave, g->cu_count * 8)), blk, static_cast<const int64_t*>(g->out_off),
                     fold_dst, next, node, score, comp, static_cast<const int32_t*>(wave_list),
                     static_cast<const BcCounters*>(dc), wk(kWDeltaWave)));
          if (side_wave) GG_HIP(hipEventRecord(g->ev_join2, ws));
          launches++;
        }
        delta();
        if (hubs) GG_HIP(hipStreamWaitEvent(st, g->ev_join, 0));
        if (side_wave) GG_HIP(hipStreamWaitEvent(st, g->ev_join2, 0));
        Run(g, "bc_clear_reduce", 0, BcClearReduce, dim3(1), blk, dc);
        launches += 2;
      }
    }
  }
  GG_HIP(hipMemsetAsync(max_bits, 0, sizeof(unsigned long long), st));
  Run(g, "bc_max", N * sizeof(T) * 2, BcMax<T>, dim3(GridFor(n, kBS, g->cu_count * 4)), blk,
      static_cast<const T*>(score), static_cast<const T*>(comp), n, max_bits);
  Run(g, "bc_normalize", N * (sizeof(T) * 2 + 4), BcNormalize<T>, grid_n, blk, static_cast<const T*>(score),
      static_cast<const T*>(comp), n, static_cast<const unsigned long long*>(max_bits), out32);
  launches += 2;
  GG_HIP(hipGetLastError());
  if (g->profile) {
    // Bytes beyond the per-vertex parts credited at launch: per list entry
    // its id and the neighbour's depth (8 B; its level bit comes from cache);
    // per matched in-neighbour its sigma (8 B); per successor its sigma and
    // delta (8 + sizeof(T) B).
    const std::vector<unsigned long long> w = ReadWork(g, work, kWKinds);
    for (int kind = 0; kind < kWKinds; kind++) {
      const double per_match = kind <= kWSigmaChunks ? 8.0 : 8.0 + sizeof(T);
      CreditBytes(g, rec[kind], 8.0 * w[2 * kind] + per_match * w[2 * kind + 1]);
    }
  }
  FinishTiming(g, stats, wt);
  g->ws.Spare("bc.level_bits");
  g->ws.Spare("bc.chunks");
  if (scores_out) CopyOutVertexF32(g, out32, scores_out);
  if (stats) {
    stats->total_ms = wt.ms();
    stats->iterations = levels_total;
    stats->reached = reached_total;
    stats->edges_examined = examined_total;
    stats->launches = launches;
  }
}

}  // namespace
}  // namespace gg

using namespace gg;

extern "C" int gg_bc(gg_graph* g, const int32_t* roots, int k, int mode, float* scores, gg_stats* stats) {
  return Guard([&] {
    WallTimer wt;
    StatsReset(stats);
    GG_REQUIRE(g != nullptr, GG_EINVAL, "null graph");
    GG_REQUIRE(!g->weighted, GG_ENOTSUP, "BC needs an unweighted graph upload");
    GG_REQUIRE(k >= 0 && (k == 0 || roots != nullptr), GG_EINVAL, "bad root list");
    GG_REQUIRE(mode == GG_BC_FP32 || mode == GG_BC_FP64 || mode == GG_BC_FP32_KAHAN, GG_EINVAL,
               "unknown precision mode");
    for (int i = 0; i < k; i++) GG_REQUIRE(roots[i] >= 0 && roots[i] < g->n, GG_EINVAL, "root out of range");
    GG_HIP(hipSetDevice(g->device));
    std::vector<int32_t> mapped(roots, roots + k);
    for (int32_t& r : mapped) r = DeviceVertex(g, r);
    roots = mapped.data();
    if (mode == GG_BC_FP32)
      RunBrandes<float, false>(g, roots, k, scores, stats, wt);
    else if (mode == GG_BC_FP32_KAHAN)
      RunBrandes<float, true>(g, roots, k, scores, stats, wt);
    else
      RunBrandes<double, false>(g, roots, k, scores, stats, wt);
  });
}
