// Load-balanced expansion of a vertex frontier over its CSR edges.
//
// One 256-thread block takes a tile of 256 frontier vertices and visits all
// their edges so that a hub with millions of edges and a vertex with three
// cost about the same per edge:
//   0. vertices with >= MinFor edges are cut into chunks of at most kMax
//      edges appended to a chunk list, which a second kernel (ExpandChunks)
//      spreads over the whole grid.  Frontiers use FrontierCut: neighbouring
//      frontier entries of a degree-ordered graph have similar degrees, so
//      with a higher cut-off one tile can hold 256 vertices of thousands of
//      edges and outlast the rest of its launch (Kronecker 22, SSSP: 1.7 ms at
//      4096, 0.5 ms at 512); of a small frontier, whose tiles leave most of
//      the chip idle, shorter lists are spread too (40 k vertices of 400 close
//      neighbours: BFS 33 ms at 512, 5.3 at 256, SSSP 55 and 9.3).  Passes over
//      all vertices use WholeCut: fewer chunks;
//   1. the rest form one flat range of edges (block prefix sum over their
//      edge counts); each thread takes kExpandEdges of them per step, one
//      per kExpandBS, and finds an edge's vertex by binary search in LDS.
// The visitor is called as op.Visit(u, payload, edge_index, valid) with
// arrays of kExpandEdges, by every lane of a wavefront together.  It loads
// for all its edges before it acts on the first, so a wavefront has several
// dependent-load chains in flight; padding edges (valid[k] == false) name
// edge 0, which may be loaded but not acted on; a wavefront all of padding
// edges does not call it.  op.StepEnd(edges) follows each step of that many
// edges, called by the whole block.  The flat range itself needs no barrier:
// with one edge per thread and two barriers per 256 edges, and vertices of
// 256 to 4095 edges taken by the whole block one after the other, the
// single-root SSSP relaxations of Kronecker 22 took 7.9 instead of 5.3 ms.
#pragma once

#include <algorithm>

#include "gg_common.h"

namespace gg {

constexpr int kExpandBS = 256;
constexpr int kExpandEdges = 4;  // edges per thread and step
constexpr int kStepEdges = kExpandBS * kExpandEdges;

// Which vertices go to the chunk list and how long their chunks are.
template <int kMinEdges, int kMaxEdges>
struct ChunkCut {
  static constexpr int kMin = kMinEdges, kMax = kMaxEdges;
  // Upper bound on the chunks of one expansion in which every vertex appears
  // at most once: sum(ceil(deg / kMax)) <= E / kMax + #{deg >= kMin}.
  static int64_t Bound(int64_t n, int64_t entries) {
    const int64_t big = entries / kMin < n ? entries / kMin : n;
    return entries / kMax + big + 2;
  }
};
// The cut-off follows the frontier's size: kMin in one of few vertices.
struct FrontierCut {
  static constexpr int kMin = 256, kMinLarge = 512, kMax = kStepEdges;
  static constexpr int64_t kFew = 4096;
  __host__ __device__ static int MinFor(int64_t vertices) { return vertices <= kFew ? kMin : kMinLarge; }
  static int64_t Bound(int64_t n, int64_t entries) {
    return ChunkCut<kMinLarge, kMax>::Bound(n, entries) + std::min(kFew, entries / kMin);
  }
};
// Of a pass over a whole graph: lists of kMax entries or more.  A few thousand
// vertices of hundreds of entries fill a few tiles, so relabelling spreads
// lists of MinFor (4096 vertices of 2000 entries: the copy 1.10 ms with kMax,
// 0.03 with 256; 16 k of 1600: 1.31 and 0.17).  Components link them no faster
// so: more threads meet at the same roots (Shiloach-Vishkin, 40 k vertices of
// 400 close neighbours: 0.42 ms, 0.80 with 256).
struct WholeCut : ChunkCut<4096, 4096> {
  static constexpr int64_t kFew = 1 << 18, kDense = 128;
  static int MinFor(int64_t n, int64_t entries) { return n <= kFew && entries >= kDense * n ? 256 : kMin; }
  static int64_t BoundFor(int64_t n, int64_t entries) {
    return MinFor(n, entries) < kMin ? ChunkCut<256, kMax>::Bound(n, entries) : Bound(n, entries);
  }
};

struct EdgeChunk {
  int64_t beg, end;
  int32_t u, payload;
};

struct ExpandShared {
  int scan[kExpandBS / kWave];
  int pre[kExpandBS];  // first flat position of each vertex
  int32_t u[kExpandBS];
  int32_t payload[kExpandBS];
  int64_t beg[kExpandBS];
};

// Expands one tile.  (u, payload, beg, end) describe this thread's vertex
// (beg == end for threads without one).  Must be called by all threads of
// the block.  Vertices of chunk_min edges or more (the same in every tile) go
// to the chunk list; chunks == nullptr disables it (the tile's edges must then
// number below 2^31).  Threads from nv on have no vertex: the owner
// search of a frontier's last, small tile is that much shorter (SSSP of 2^18
// vertices with close neighbours, a few hundred in a bucket: 463 -> 453 ms).
template <class Cut, class Op>
__device__ __forceinline__ void ExpandTile(ExpandShared& sh, int32_t u, int32_t payload,
                                           int64_t beg, int64_t end, Op& op,
                                           EdgeChunk* chunks, int32_t* nchunks, int chunk_min,
                                           int nv = kExpandBS) {
  const int tid = threadIdx.x, wave_first = __builtin_amdgcn_readfirstlane(tid);
  // 0. Hubs: hand their edges to the grid-wide chunk kernel, one reservation
  // per wavefront.
  if (chunks) {
    const int nc = end - beg >= chunk_min ? static_cast<int>((end - beg + Cut::kMax - 1) / Cut::kMax) : 0;
    if (__ballot(nc > 0)) {
      const int upto = WaveInclusiveScan(nc);
      int base = 0;
      if (LaneId() == kWave - 1) base = atomicAdd(nchunks, upto);
      base = __builtin_amdgcn_readlane(base, kWave - 1) + upto - nc;
      for (int c = 0; c < nc; c++) {
        const int64_t cb = beg + int64_t(c) * Cut::kMax;
        const int64_t ce = cb + Cut::kMax < end ? cb + Cut::kMax : end;
        chunks[base + c] = EdgeChunk{cb, ce, u, payload};
      }
      if (nc) beg = end;
    }
  }
  // 1. Everything else, flat.
  int total = 0;
  sh.pre[tid] = BlockExclusiveScan<kExpandBS>(static_cast<int>(end - beg), &total, sh.scan);
  sh.u[tid] = u;
  sh.payload[tid] = payload;
  sh.beg[tid] = beg;
  int top = kExpandBS / 2;  // the owner search's first step
  while (top >= nv) top >>= 1;
  __syncthreads();
  for (int base = 0; base < total; base += kStepEdges) {
    int32_t eu[kExpandEdges], ep[kExpandEdges];
    int64_t e[kExpandEdges];
    bool valid[kExpandEdges];
    int at[kExpandEdges];  // the last vertex starting at or before the edge: the one that owns it
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++) at[k] = 0;
    for (int step = top; step > 0; step >>= 1) {
#pragma unroll
      for (int k = 0; k < kExpandEdges; k++)
        if (sh.pre[at[k] + step] <= base + k * kExpandBS + tid) at[k] += step;
    }
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++) {
      const int j = base + k * kExpandBS + tid;
      valid[k] = j < total;
      eu[k] = sh.u[at[k]];
      ep[k] = sh.payload[at[k]];
      e[k] = valid[k] ? sh.beg[at[k]] + (j - sh.pre[at[k]]) : 0;
    }
    if (base + wave_first < total) op.Visit(eu, ep, e, valid);
    op.StepEnd(total - base < kStepEdges ? total - base : kStepEdges);
  }
  __syncthreads();
}

// Visits the edges of every chunk emitted by ExpandTile with the same Cut.
// Work items are steps of kStepEdges edges, spread over the grid; a block's
// next chunk is read while it works on the current one.  Must be called by
// all threads of the block.
template <class Cut, class Op>
__device__ __forceinline__ void ExpandChunks(const EdgeChunk* __restrict__ chunks, int32_t nchunks,
                                             Op& op) {
  constexpr int kSteps = Cut::kMax / kStepEdges;
  const int wave_first = __builtin_amdgcn_readfirstlane(threadIdx.x);
  static_assert(kSteps * kStepEdges == Cut::kMax, "chunks are whole steps");
  const int64_t items = int64_t(nchunks) * kSteps;
  int64_t it = blockIdx.x;
  if (it >= items) return;
  EdgeChunk next = chunks[it / kSteps];
  while (it < items) {
    const EdgeChunk ch = next;
    const int64_t first = ch.beg + (it % kSteps) * kStepEdges + threadIdx.x;
    it += gridDim.x;
    if (it < items) next = chunks[it / kSteps];
    const int64_t left = ch.end - (first - threadIdx.x);
    if (left <= 0) continue;  // a short last chunk
    int32_t eu[kExpandEdges], ep[kExpandEdges];
    int64_t e[kExpandEdges];
    bool valid[kExpandEdges];
#pragma unroll
    for (int k = 0; k < kExpandEdges; k++) {
      valid[k] = first + k * kExpandBS < ch.end;
      eu[k] = ch.u;
      ep[k] = ch.payload;
      e[k] = valid[k] ? first + k * kExpandBS : 0;
    }
    if (wave_first < left) op.Visit(eu, ep, e, valid);
    op.StepEnd(left < kStepEdges ? static_cast<int>(left) : kStepEdges);
  }
}

// A block's output queue staged in LDS: wavefronts append with LDS atomics,
// the block flushes once with one global atomic.  Entries that do not fit
// go straight to global memory.
template <int CAP>
struct LdsQueue {
  int count;  // entries reserved; may exceed CAP
  int32_t base;
  int32_t items[CAP];
};

template <int CAP>
__device__ __forceinline__ void LdsQueueInit(LdsQueue<CAP>& q) {
  if (threadIdx.x == 0) q.count = 0;
  __syncthreads();
}

// K pushes per lane for one reservation: every active lane of the wavefront
// calls it together.
template <int CAP, int K>
__device__ __forceinline__ void LdsQueuePushMany(LdsQueue<CAP>& q, const bool (&take)[K], const int32_t (&v)[K],
                                                 int32_t* gout, int32_t* gtail) {
  uint64_t m[K];
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < K; k++) {
    m[k] = __ballot(take[k]);
    cnt += __popcll(m[k]);
  }
  if (cnt == 0) return;
  const bool leader = LanesBelow(__ballot(true)) == 0;  // the first active lane
  int base = 0;
  if (leader) base = atomicAdd(&q.count, cnt);
  base = __builtin_amdgcn_readfirstlane(base);
  const int fit = base >= CAP ? 0 : CAP - base;
  int gbase = 0;
  if (cnt > fit) {
    if (leader) gbase = atomicAdd(gtail, cnt - fit);
    gbase = __builtin_amdgcn_readfirstlane(gbase);
  }
  int rank0 = 0;
#pragma unroll
  for (int k = 0; k < K; k++) {
    if (take[k]) {
      const int rank = rank0 + __popcll(LanesBelow(m[k]));
      if (rank < fit)
        q.items[base + rank] = v[k];
      else
        gout[gbase + rank - fit] = v[k];
    }
    rank0 += __popcll(m[k]);
  }
}

// Wave-wide: every active lane of the wavefront calls it together.
template <int CAP>
__device__ __forceinline__ void LdsQueuePush(LdsQueue<CAP>& q, bool take, int32_t v, int32_t* gout,
                                             int32_t* gtail) {
  const uint64_t m = __ballot(take);
  if (m == 0) return;
  const int lane = LaneId();
  const int leader = __ffsll(static_cast<unsigned long long>(m)) - 1;
  const int cnt = __popcll(m);
  int base = 0;
  if (lane == leader) base = atomicAdd(&q.count, cnt);
  base = __shfl(base, leader);
  const int fit = CAP - base > 0 ? CAP - base : 0;
  const int over = cnt > fit ? cnt - fit : 0;
  int gbase = 0;
  if (over && lane == leader) gbase = atomicAdd(gtail, over);
  gbase = __shfl(gbase, leader);
  if (take) {
    const int rank = __popcll(LanesBelow(m));
    if (rank < fit)
      q.items[base + rank] = v;
    else
      gout[gbase + rank - fit] = v;
  }
}

// Block-wide: all threads call it (synchronises).
template <int CAP>
__device__ __forceinline__ void LdsQueueFlush(LdsQueue<CAP>& q, int32_t* gout, int32_t* gtail) {
  __syncthreads();
  const int cnt = q.count < CAP ? q.count : CAP;
  if (threadIdx.x == 0) q.base = cnt ? atomicAdd(gtail, cnt) : 0;
  __syncthreads();
  for (int i = threadIdx.x; i < cnt; i += blockDim.x) gout[q.base + i] = q.items[i];
}

// Block-wide, after a step that pushed at most `pushed` entries; `most` is
// what the queue can hold since it was last looked at.  Empties the queue
// while a whole step still fits; the barriers that a look takes are left out
// while it surely does.  A queue that overflows
// pushes through one global counter, an atomic per wavefront, which the chip
// takes one after another (SSSP on Kronecker 22, largest launch: 2.0 ms
// against 0.6).
template <int CAP>
__device__ __forceinline__ void LdsQueueMakeRoom(LdsQueue<CAP>& q, int32_t* gout, int32_t* gtail, int& most,
                                                 int pushed) {
  static_assert(CAP >= 2 * kStepEdges, "room for a step while half full");
  most += pushed;
  if (most <= CAP - kStepEdges) return;  // the same in all threads
  __syncthreads();
  most = q.count;
  __syncthreads();  // read by all before anyone pushes again
  if (most <= CAP - kStepEdges) return;
  most = 0;
  LdsQueueFlush(q, gout, gtail);
  __syncthreads();
  if (threadIdx.x == 0) q.count = 0;
  __syncthreads();
}

// Block-aggregated append: one atomic per block.  All threads of the block
// call it together; `sh` needs kExpandBS/64 + 1 ints.
template <class T>
__device__ __forceinline__ void BlockAppend(bool take, T value, T* out, int32_t* tail, int* sh) {
  const int lane = LaneId(), wid = threadIdx.x / kWave;
  const uint64_t m = __ballot(take);
  if (lane == 0) sh[wid] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int total = 0;
    for (int w = 0; w < kExpandBS / kWave; w++) {
      const int c = sh[w];
      sh[w] = total;
      total += c;
    }
    sh[kExpandBS / kWave] = total ? atomicAdd(tail, total) : 0;
  }
  __syncthreads();
  if (take) out[sh[kExpandBS / kWave] + sh[wid] + __popcll(LanesBelow(m))] = value;
  __syncthreads();
}

}  // namespace gg
