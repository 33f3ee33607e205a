// Batched path-segment back-propagation on gfx950: the training samples of
// many recorded paths (PathSegmentDataStorage::prepareSamples,
// data/PathSegmentDataStorage.h:160-315, applied to each path), written as
// PGLSampleData records, surface and volume apart, in the order the
// per-path calls would append them to one sample storage.
//
// One thread per vertex, 256 consecutive vertices per workgroup (a tile).
// The tile's vertices, and the rest of the path its last vertex belongs to
// (up to 64 more), are first copied to LDS with coalesced loads, together
// with the offsets of the tile's paths; each vertex's thread then finds its
// path in LDS, redoes the path's backward distance walk from the last vertex
// down to its own (the exact sequence of float operations of the serial
// walk) and its own contribution (path_samples.h) reading LDS, and stores its
// record and a packed surface | volume << 32 flag.  A path reaching beyond
// the staged vertices is read from global memory.  The first path of every
// tile is found beforehand, one thread per tile.  An inclusive scan of the
// flags gives every record its place: the records of earlier paths, plus
// those of the same path at later vertices (the walk emits vertex n-2 first).
// Outputs with room for every vertex are written by one pass over the vertices
// instead (k_path_fused, below); these launches remain for smaller outputs,
// for paths of more than 64 vertices and for the caller that may not allocate.
#pragma clang fp contract(off)
#include <hip/hip_runtime.h>

#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <string>

#include "kernels.h"
#include "path_samples.h"

namespace pglgpu {

namespace {

constexpr int kPathThreads = 256;
constexpr uint32_t kNoPath = 0xffffffffu;

// the path holding vertex v: the last p with offsets[p] <= v
__device__ __forceinline__ uint32_t path_of(const uint32_t* __restrict__ offsets, uint32_t numPaths, uint32_t v) {
  uint32_t lo = 0, hi = numPaths;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (offsets[mid] <= v) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ void k_path_clear(unsigned long long* __restrict__ totals) {
  if (threadIdx.x < 3) totals[threadIdx.x] = 0ull;
}

__global__ void __launch_bounds__(kPathThreads) k_path_check(const uint32_t* __restrict__ offsets, uint32_t numPaths,
                                                             uint32_t numSegments,
                                                             unsigned long long* __restrict__ totals) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= numPaths) return;
  if (offsets[p] > offsets[p + 1] || offsets[p + 1] > numSegments) totals[2] = 1ull;
}

constexpr uint32_t kStage = kPathThreads + 64;  // staged vertices of a tile
constexpr uint32_t kTileOffsets = 512;           // path offsets of a tile kept in LDS
constexpr uint32_t kStepBuckets = 64;            // walk lengths >= 63 share the last bucket

// tileFirst[t] = path of vertex t * kPathThreads, tileFirst[numTiles] = path
// of the last vertex (numSegments >= 1)
__global__ void __launch_bounds__(kPathThreads) k_path_tiles(const uint32_t* __restrict__ offsets, uint32_t numPaths,
                                                             uint32_t numSegments, uint32_t numTiles,
                                                             uint32_t* __restrict__ tileFirst) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > numTiles) return;
  tileFirst[t] = path_of(offsets, numPaths, t < numTiles ? t * kPathThreads : numSegments - 1);
}

// the last p in [0, count) with offs[p] <= v (0 if none)
__device__ __forceinline__ uint32_t tile_path(const uint32_t* offs, uint32_t count, uint32_t v) {
  uint32_t lo = 0, hi = count;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (offs[mid] <= v) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ void __launch_bounds__(kPathThreads) k_path_vertex(const PathVertex* __restrict__ segs, uint32_t numSegments,
                                                              const uint32_t* __restrict__ offsets, uint32_t numPaths,
                                                              const uint32_t* __restrict__ tileFirst,
                                                              PathSampleOptions o, PathSample* __restrict__ records,
                                                              unsigned long long* __restrict__ flags,
                                                              uint32_t* __restrict__ pathOf) {
  __shared__ PathVertex stage[kStage];
  __shared__ uint32_t offs[kTileOffsets];
  __shared__ uint32_t stageEnd;
  __shared__ uint32_t hist[kStepBuckets];
  __shared__ uint32_t vb[kPathThreads], ve[kPathThreads], vq[kPathThreads];
  __shared__ uint16_t order[kPathThreads];
  const uint32_t tid = threadIdx.x, t0 = blockIdx.x * kPathThreads;
  const uint32_t t1 = min(t0 + kPathThreads, numSegments);
  const uint32_t v = t0 + tid;
  // the tile's paths p0 .. p1 (monotone offsets); their offsets p0 .. p1 + 1
  const uint32_t p0 = tileFirst[blockIdx.x];
  const uint32_t p1 = max(p0, min(tileFirst[blockIdx.x + 1], numPaths - 1));
  const uint32_t np = p1 - p0 + 2;
  const bool inLds = np <= kTileOffsets;
  if (inLds)
    for (uint32_t i = tid; i < np; i += kPathThreads) offs[i] = offsets[p0 + i];
  if (tid == 0) stageEnd = t1;
  __syncthreads();
  uint32_t q = kNoPath, b = 0, e = 0;
  if (v < t1) {
    q = inLds ? p0 + tile_path(offs, np - 1, v) : path_of(offsets, numPaths, v);
    b = inLds ? offs[q - p0] : offsets[q];
    e = inLds ? offs[q - p0 + 1] : offsets[q + 1];
    // the tile's last vertex extends the staged range to the end of its path
    if (v + 1 == t1 && e > t1 && e <= numSegments) stageEnd = min(e, t0 + kStage);
  }
  __syncthreads();
  const uint32_t nStage = stageEnd - t0;
  {
    // 8-byte words (the vertex alignment); every thread issues all its loads
    // before its first store, so a tile pays one memory latency
    constexpr uint32_t kWords = (uint32_t)(sizeof(PathVertex) / 8);
    constexpr uint32_t kIt = (kStage * kWords + kPathThreads - 1) / kPathThreads;
    const uint2* src = reinterpret_cast<const uint2*>(segs + t0);
    uint2* dst = reinterpret_cast<uint2*>(stage);
    const uint32_t words = nStage * kWords;
    uint2 tmp[kIt];
#pragma unroll
    for (uint32_t k = 0; k < kIt; k++) {
      const uint32_t i = tid + k * kPathThreads;
      if (i < words) tmp[k] = src[i];
    }
#pragma unroll
    for (uint32_t k = 0; k < kIt; k++) {
      const uint32_t i = tid + k * kPathThreads;
      if (i < words) dst[i] = tmp[k];
    }
  }
  // a vertex's walk takes e - v - 1 steps: the tile's vertices are handed to
  // the threads in decreasing order of that length (counting sort in LDS), so
  // that the lanes of a wave take about the same number of steps
  const bool valid = v < t1 && b <= v && v < e && e <= numSegments;
  const uint32_t steps = valid && v + 1 < e ? e - v - 1 : 0u;
  const uint32_t key = kStepBuckets - 1 - min(steps, kStepBuckets - 1);
  if (tid < kStepBuckets) hist[tid] = 0u;
  vb[tid] = b;
  ve[tid] = e;
  vq[tid] = valid ? q : kNoPath;
  __syncthreads();
  const uint32_t rank = v < t1 ? atomicAdd(&hist[key], 1u) : 0u;
  __syncthreads();
  if (tid < kStepBuckets) {  // exclusive prefix of the bucket counts (one wave)
    const uint32_t c = hist[tid];
    uint32_t x = c;
#pragma unroll
    for (int d = 1; d < (int)kStepBuckets; d <<= 1) {
      const uint32_t y = __shfl_up(x, d, (int)kStepBuckets);
      if ((int)tid >= d) x += y;
    }
    hist[tid] = x - c;
  }
  __syncthreads();
  if (v < t1) order[hist[key] + rank] = (uint16_t)tid;
  __syncthreads();
  if (v >= t1) return;
  // this thread's vertex (the order within a bucket varies; each record does not)
  const uint32_t w = order[tid], u = t0 + w;
  const uint32_t ub = vb[w], ue = ve[w], uq = vq[w];
  unsigned long long flag = 0ull;
  if (uq != kNoPath) {
    PathSample s;
    bool ok = false;
    if (u + 1 < ue) {  // vertices n-1 (the last of a path) yield no sample
      // the walk reads vertices u .. e-1 only: vertex u is index 0 of the suffix
      if (ue <= t0 + nStage) ok = path_vertex_sample(stage + w, (int)(ue - u), 0, o, s);
      else ok = path_vertex_sample(segs + u, (int)(ue - u), 0, o, s);
    }
    if (ok) {
      records[u] = s;
      flag = (s.flags & 2u) ? (1ull << 32) : 1ull;
    }
  }
  (void)ub;
  flags[u] = flag;
  pathOf[u] = uq;
}

__global__ void k_path_totals(const unsigned long long* __restrict__ incl, uint32_t numSegments,
                              unsigned long long* __restrict__ totals) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const unsigned long long t = numSegments ? incl[numSegments - 1] : 0ull;
    totals[0] = t & 0xffffffffull;
    totals[1] = t >> 32;
  }
}

__global__ void __launch_bounds__(kPathThreads) k_path_scatter(const PathSample* __restrict__ records,
                                                               const unsigned long long* __restrict__ flags,
                                                               const uint32_t* __restrict__ pathOf,
                                                               const unsigned long long* __restrict__ incl,
                                                               const uint32_t* __restrict__ offsets,
                                                               uint32_t numSegments, PathSample* __restrict__ surfOut,
                                                               PathSample* __restrict__ volOut) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < numSegments; v += stride) {
    const unsigned long long f = flags[v];
    if (!f) continue;
    const uint32_t p = pathOf[v];
    const uint32_t b = offsets[p], e = offsets[p + 1];
    const unsigned long long before = b > 0 ? incl[b - 1] : 0ull;  // records of earlier paths
    const unsigned long long last = incl[e - 1], mine = incl[v];
    const int hi = (f >> 32) ? 32 : 0;
    // records of earlier paths + those of this path at later vertices
    const uint32_t pos = (uint32_t)(before >> hi) + ((uint32_t)(last >> hi) - (uint32_t)(mine >> hi));
    if (hi) volOut[pos] = records[v]; else surfOut[pos] = records[v];
  }
}

// ---- the same records in one pass over the vertices
//
// A tile is the paths that begin at its 256 vertices, so that every record of
// a path, and with it the reversed order within the path, is known to one
// block; the records go straight to their final places.  The place of a tile's
// first record is the sum of the counts of all tiles before it: each tile
// publishes its counts, the first block adds them up, and a tile's records,
// held in registers, are written once its successor in the same block has
// published its own.  Blocks take tiles in increasing order from a counter, so
// every tile that one waits for is held by a block that is already running and
// itself waits for lower tiles only.
//
// 136 bytes per vertex come in and 40 per record go out, and the tiles of a
// compute unit are few (45 KB of LDS each); so a block reads its next tile
// into registers while it works on the current one.  6.0M vertices in 1M
// paths: 320 us, 2.6 TB/s of vertices (the counting launches and their scatter
// 515 us); 12k vertices in 3001 paths: 34 us with both launches and the wait,
// 74 us before.  What bounds a tile's 10 us is latency: 4 us are the longest
// wave's walk, 3 the waits for the staged words and for earlier tiles' counts;
// the vector units are busy a third of the time, LDS conflicts a fifth.

constexpr uint32_t kReadAhead = 271;  // vertices of a tile read ahead: 18 8-byte words per thread
constexpr uint32_t kAheadWords = 18;
constexpr uint32_t kVertexWords8 = (uint32_t)(sizeof(PathVertex) / 8);
constexpr uint32_t kVertexWords4 = (uint32_t)(sizeof(PathVertex) / 4);
// paths of a tile taken one by one; with more of them, most of them empty (rays
// that left the scene), every vertex finds its own by bisection: 500k empty
// paths in one tile of 12k vertices took 450 us one by one, 29 by bisection;
// 5000 take 29 and 28
constexpr uint32_t kTilePaths = 2048;
constexpr uint32_t kMaskWords = 16;  // bit mask of a tile's vertices, a word per lane of a row
static_assert(kMaskWords > kStage / 32, "counts of the bits before any vertex and before the end");
static_assert(kReadAhead * kVertexWords8 <= kAheadWords * kPathThreads, "a tile's vertices are read by one pass");
static_assert(kFusedPathLength + kPathThreads <= kStage, "a tile's last path ends in the staged vertices");
// words of PathVertex that carry something else inside a tile: the pad and the
// region pointer hold the distance to the next vertex and the factor of the
// length carried on, the first of the directionOut words the record's tail
constexpr uint32_t kWordReciprocal = 31, kWordDistance = 32, kWordFactor = 33, kWordTail = 6;

// Division of the three throughputs by a survival probability, the same result
// as the divisions themselves: with the reciprocal refined once (one per
// vertex), the quotient is refined by two exact remainders.  Only in ranges
// where no step can over- or underflow; elsewhere, and for negative numbers,
// the plain division (kept reciprocal 0).
constexpr float kSmallDivided = 0x1p-60f, kLargeDivided = 0x1p60f;
__device__ __forceinline__ float survival_reciprocal(float rr) {
  if (!(rr >= kSmallDivided && rr <= 0x1p20f)) return 0.0f;
  const float y = __builtin_amdgcn_rcpf(rr);
  return fmaf(fmaf(-rr, y, 1.0f), y, y);
}
__device__ __forceinline__ void survive(const PathStep& v, float t[3]) {
  const float rr = v.survival, y = v.reciprocal;
  const uint32_t b0 = __float_as_uint(t[0]), b1 = __float_as_uint(t[1]), b2 = __float_as_uint(t[2]);
  const uint32_t hi = max(max(b0, b1), b2), lo = min(min(b0 - 1u, b1 - 1u), b2 - 1u);  // zero is in range
  if (y != 0.0f && hi <= __float_as_uint(kLargeDivided) && lo >= __float_as_uint(kSmallDivided) - 1u) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      float q = t[k] * y;
      q = fmaf(fmaf(-rr, q, t[k]), y, q);
      t[k] = fmaf(fmaf(-rr, q, t[k]), y, q);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 3; k++) t[k] /= rr;
  }
}

// a tile's word and base: surface count | volume count << 31, and this once known
constexpr unsigned long long kTileKnown = 1ull << 63;

// One thread per path (and one more): malformed or long paths, and the first
// path of every tile (the first that begins at or after the tile's first
// vertex; tileFirst[numTiles] = numPaths).  Clears the tiles' words.
__global__ void __launch_bounds__(kPathThreads) k_path_index(const uint32_t* __restrict__ offsets, uint32_t numPaths,
                                                             uint32_t numSegments, uint32_t numTiles,
                                                             uint32_t* __restrict__ tileFirst,
                                                             unsigned long long* __restrict__ tileWord,
                                                             FusedPathControl* __restrict__ control, uint32_t epoch) {
  const uint32_t i0 = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (uint32_t t = i0; t < 2 * numTiles; t += stride) tileWord[t] = 0ull;  // and the bases behind them
  if (i0 == 0) control->ticket = 0u;
  for (uint32_t p = i0; p <= numPaths; p += stride) {
    uint32_t last = numTiles;
    if (p < numPaths) {
      const uint32_t a = offsets[p], b = offsets[p + 1];
      if (a > b || b > numSegments) control->bad = epoch;
      else if (b - a > kFusedPathLength) control->general = epoch;
      last = min(a / kPathThreads, numTiles);
    }
    // the tiles whose first vertex lies after the previous path's and not after this one's
    const uint32_t first = p > 0 ? offsets[p - 1] / kPathThreads + 1 : 0u;
    if (last >= first && last - first > 64u) control->general = epoch;  // many vertices of no path
    else
      for (uint32_t t = first; t <= last; t++) tileFirst[t] = p;
  }
}

// inclusive sums over 16 lanes (a row) and over the wave, all lanes active
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add(uint32_t x) {
  return x + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t row_scan(uint32_t x) {
  x = dpp_add<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  return dpp_add<0x118, 0xf>(x);
}
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  x = row_scan(x);
  x = dpp_add<0x142, 0xa>(x);  // the last lane of the row before, then of the first half
  return dpp_add<0x143, 0xc>(x);
}

struct alignas(4) RecordPiece {  // a fifth of a record (records are aligned to 4 bytes)
  uint32_t a, b;
};

// The running sums, by one wave: 8 tiles per lane and pass, as far as tiles
// have published their counts.  A wave of its own, as tiles that add up the
// counts before them themselves read some 800 words each (all blocks reach
// that point about together): 12 us of every tile's 20, and 20 of 28 with all
// those words in flight at once.
constexpr uint32_t kScanTiles = 8;
__device__ void path_tile_sums(const unsigned long long* tileWord, unsigned long long* tileBase, uint32_t numTiles,
                               uint32_t lane, unsigned long long* totals) {
  unsigned long long sum = 0ull;
  uint32_t done = 0;
  while (done < numTiles) {
    unsigned long long w[kScanTiles];
    const uint32_t t = done + lane * kScanTiles;
#pragma unroll
    for (uint32_t k = 0; k < kScanTiles; k++)
      w[k] = t + k < numTiles ? __hip_atomic_load(tileWord + t + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
    uint32_t ready = 0;
    unsigned long long own = 0ull;
#pragma unroll
    for (uint32_t k = 0; k < kScanTiles; k++) {
      const bool r = ready == k && (w[k] & kTileKnown);
      ready += r ? 1u : 0u;
      w[k] = r ? w[k] & ~kTileKnown : 0ull;
      own += w[k];
    }
    const unsigned long long stuck = __ballot(ready < kScanTiles);
    const uint32_t stop = stuck ? (uint32_t)__ffsll((long long)stuck) - 1u : 63u;  // the last lane of this pass
    unsigned long long incl = lane <= stop ? own : 0ull;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long y = __shfl_up(incl, d, 64);
      if ((int)lane >= d) incl += y;
    }
    unsigned long long at = sum + incl - own;
#pragma unroll
    for (uint32_t k = 0; k < kScanTiles; k++) {
      if (lane <= stop && k < ready)
        __hip_atomic_store(tileBase + t + k, kTileKnown | at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      at += w[k];
    }
    sum += __shfl(incl, 63, 64);
    const uint32_t step = stop * kScanTiles + __shfl(ready, (int)stop, 64);
    done += step;
    if (step == 0) __builtin_amdgcn_s_sleep(2);
  }
  if (lane == 0) {
    totals[0] = sum & 0x7fffffffull;
    totals[1] = sum >> 31;
    totals[2] = totals[3] = 0ull;
  }
}

__global__ void __launch_bounds__(kPathThreads, 3)
    k_path_fused(const PathVertex* __restrict__ segs, uint32_t numSegments, const uint32_t* __restrict__ offsets,
                 uint32_t numPaths, const uint32_t* __restrict__ tileFirst, uint32_t numTiles, PathSampleOptions o,
                 RecordPiece* __restrict__ surfOut, RecordPiece* __restrict__ volOut, unsigned long long* tileWord,
                 FusedPathControl* control, uint32_t epoch, unsigned long long* totals) {
  __shared__ __align__(16) uint32_t stage[kStage * kVertexWords4];
  __shared__ uint32_t span[kStage];  // per vertex: first | end << 16 of its path, 0 for none
  __shared__ uint32_t hist[kStepBuckets];
  __shared__ uint32_t mask[2][kMaskWords];
  __shared__ uint16_t order[kStage];
  __shared__ uint32_t ticket;
  __shared__ unsigned long long heldBase;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  if (tid == 0) ticket = atomicAdd(&control->ticket, 1u);
  __syncthreads();
  // the first ticket is the summing block's
  uint32_t tile = __builtin_amdgcn_readfirstlane(ticket) - 1u;
  unsigned long long* tileBase = tileWord + numTiles;
  const bool bad = control->bad == epoch, general = control->general == epoch;
  if (bad || general) {  // nothing is written
    if (tile == ~0u && tid == 0) {
      totals[0] = totals[1] = 0ull;
      totals[2] = bad ? 1ull : 0ull;
      totals[3] = 1ull;
    }
    return;
  }
  if (tile == ~0u) {
    if (tid < 64) path_tile_sums(tileWord, tileBase, numTiles, lane, totals);
    return;
  }
  uint2 ahead[kAheadWords];
  const auto readAhead = [&](uint32_t t) {
    const uint32_t v0 = t * kPathThreads;
    const uint2* src = reinterpret_cast<const uint2*>(segs + v0);
    const uint32_t words = min(kReadAhead, numSegments - v0) * kVertexWords8;
#pragma unroll
    for (uint32_t k = 0; k < kAheadWords; k++) ahead[k] = src[min(tid + k * kPathThreads, words - 1)];
  };
  // the records of the block's last tile, in pieces, until their place is known
  constexpr uint32_t kHeld = (kStage * 5 + kPathThreads - 1) / kPathThreads;
  RecordPiece held[kHeld];
  uint32_t heldTile = 0, heldS = 0, heldAll = 0;
  const auto heldPlace = [&]() {
    return __hip_atomic_load(tileBase + heldTile, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const auto writeHeld = [&](unsigned long long base) {
    if (heldAll == 0) return;
    while (!(base & kTileKnown)) {
      __builtin_amdgcn_s_sleep(1);
      base = heldPlace();
    }
    base &= ~kTileKnown;
    RecordPiece* surf = surfOut + (base & 0x7fffffffull) * 5;
    RecordPiece* volu = volOut + (base >> 31) * 5 - heldS;
#pragma unroll
    for (uint32_t k = 0; k < kHeld; k++) {
      if (k * kPathThreads >= heldAll) break;
      const uint32_t i = tid + k * kPathThreads;
      RecordPiece* to = i < heldS ? surf : volu;
      if (i < heldAll) to[i] = held[k];
    }
  };
  // the tile's paths, the end of the last one, the thread's first path
  uint32_t p0 = 0, p1 = 0, last = 0, begin = 0, end = 0;
  const auto readPaths = [&](uint32_t first, uint32_t past) {
    p0 = first;
    p1 = past;
    last = offsets[past];
    begin = offsets[min(first + tid, numPaths)];
    end = offsets[min(first + tid + 1, numPaths)];
  };
  if (tile < numTiles) {
    readPaths(tileFirst[tile], tileFirst[tile + 1]);
    readAhead(tile);
  }
  while (tile < numTiles) {
    const uint32_t t0 = tile * kPathThreads;
    const uint32_t np = p1 - p0, staged = np ? last - t0 : 0u;
    {
      // (words past the end of the vertices were read as the last one)
      uint2* dst = reinterpret_cast<uint2*>(stage);
#pragma unroll
      for (uint32_t k = 0; k < kAheadWords; k++) {
        const uint32_t i = tid + k * kPathThreads;
        if ((k + 1) * kPathThreads <= kReadAhead * kVertexWords8 || i < kReadAhead * kVertexWords8) dst[i] = ahead[k];
      }
      if (staged > kReadAhead) {
        const uint2* src = reinterpret_cast<const uint2*>(segs + t0);
        for (uint32_t i = kReadAhead * kVertexWords8 + tid; i < staged * kVertexWords8; i += kPathThreads) dst[i] = src[i];
      }
    }
    for (uint32_t i = tid; i < kStage; i += kPathThreads) span[i] = 0u;
    if (tid < kStepBuckets) hist[tid] = 0u;
    if (tid < 2 * kMaskWords) (&mask[0][0])[tid] = 0u;
    __syncthreads();
    // every vertex learns its path's first and end
    if (np <= kTilePaths) {
      for (uint32_t i = tid; i < np; i += kPathThreads) {
        const uint32_t b = (i < kPathThreads ? begin : offsets[p0 + i]) - t0;
        const uint32_t e = (i < kPathThreads ? end : offsets[p0 + i + 1]) - t0;
        for (uint32_t w = b; w < e; w++) span[w] = b | (e << 16);
      }
    } else {
      for (uint32_t w = tid; w < staged; w += kPathThreads) {
        const uint32_t p = p0 + path_of(offsets + p0, np, t0 + w);
        const uint32_t b = offsets[p] - t0, e = offsets[p + 1] - t0;
        if (b <= w && w < e) span[w] = b | (e << 16);
      }
    }
    if (tid == kPathThreads - 1) ticket = atomicAdd(&control->ticket, 1u);
    __syncthreads();
    const uint32_t next = __builtin_amdgcn_readfirstlane(ticket) - 1u;
    uint32_t nextFirst = 0, nextPast = 0;
    if (next < numTiles) {
      readAhead(next);
      nextFirst = tileFirst[next];
      nextPast = tileFirst[next + 1];
    }
    // the length each vertex adds to a walk, and the vertices that can yield a
    // record, in decreasing order of their walk (counting sort)
    uint32_t key[2], rank[2];
#pragma unroll
    for (uint32_t r = 0; r < 2; r++) {
      const uint32_t w = tid + r * kPathThreads;
      key[r] = kStepBuckets;
      if (w >= kStage) continue;
      const uint32_t e = span[w] >> 16;
      if (w + 1 >= e) continue;
      const PathVertex* c = reinterpret_cast<const PathVertex*>(stage) + w;
      float carried;
      float* words = reinterpret_cast<float*>(stage + w * kVertexWords4);
      words[kWordDistance] = path_edge(c[0], c[1], carried);
      words[kWordFactor] = carried;
      words[kWordReciprocal] = survival_reciprocal(c->russianRouletteProbability);
      if (!path_vertex_records(c[0])) continue;
      key[r] = kStepBuckets - min(e - w - 1, kStepBuckets);
      rank[r] = atomicAdd(&hist[key[r]], 1u);
    }
    __syncthreads();
    const uint32_t count = hist[lane];
    const uint32_t incl = wave_scan(count);
    const uint32_t active = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
#pragma unroll
    for (uint32_t r = 0; r < 2; r++) {
      if (r == 1 && tid >= 64u) break;  // whole waves
      const uint32_t before = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(key[r] * 4u), (int)(incl - count));
      if (key[r] < kStepBuckets) order[before + rank[r]] = (uint16_t)(tid + r * kPathThreads);
    }
    __syncthreads();
    // (the waves' shares differ in length and rotate from tile to tile; the one
    // with the shortest walks also asks for the place of the held records;
    // it must not wait for the place before the tile's own counts
    // are out, or all tiles would wait in one chain)
    const uint32_t at = (tid + 64u * tile) & (kPathThreads - 1);
    for (uint32_t i = at; i < active; i += kPathThreads) {
      const uint32_t w = order[i], e = span[w] >> 16;
      const PathVertex* seg = reinterpret_cast<const PathVertex*>(stage) + w;
      const float* words = reinterpret_cast<const float*>(stage);
      float lastDistance = 0.0f, distance = 0.0f;
#pragma unroll 4
      for (uint32_t k = e - 1; k-- > w;)
        distance = path_carry(words[k * kVertexWords4 + kWordDistance], words[k * kVertexWords4 + kWordFactor],
                              o.maxDistance, lastDistance);
      PathSample s;
      if (path_vertex_record(seg, (int)(e - w), 0, distance, o, s, survive)) {
        // position and directionIn lead the vertex as they lead the record
        uint32_t* tail = stage + w * kVertexWords4 + kWordTail;
        tail[0] = __float_as_uint(s.weight);
        tail[1] = __float_as_uint(s.pdf);
        tail[2] = __float_as_uint(s.distance);
        tail[3] = s.flags;
        atomicOr(&mask[s.flags ? 1 : 0][w >> 5], 1u << (w & 31u));
      }
    }
    if (at >= kPathThreads - 64) {
      unsigned long long base = heldPlace();
      for (int k = 0; k < 2 && !(base & kTileKnown); k++) base = heldPlace();
      if (lane == 0) heldBase = base;
    }
    __syncthreads();
    // counts before each word of the masks: surface in the first row of lanes, volume in the second
    const uint32_t ones = (uint32_t)__popc((&mask[0][0])[lane & 31u]);
    const uint32_t incl2 = row_scan(ones), pre = incl2 - ones;
    const uint32_t numS = (uint32_t)__builtin_amdgcn_readlane((int)incl2, 15);
    const uint32_t numV = (uint32_t)__builtin_amdgcn_readlane((int)incl2, 31);
    if (tid == 0)
      __hip_atomic_store(tileWord + tile, kTileKnown | (unsigned long long)numS | ((unsigned long long)numV << 31),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    writeHeld(heldBase);
    if (next < numTiles) readPaths(nextFirst, nextPast);
    // records in their order: those of the paths before, then those of the
    // path's later vertices
#pragma unroll
    for (uint32_t r = 0; r < 2; r++) {
      const uint32_t w = tid + r * kPathThreads;
      if (r == 1 && tid >= 64u) break;  // whole waves
      const uint32_t se = span[w], b = se & 0xffffu, e = se >> 16;
      const bool vol = (mask[1][w >> 5] >> (w & 31u)) & 1u, sur = (mask[0][w >> 5] >> (w & 31u)) & 1u;
      const uint32_t row = vol ? kMaskWords : 0u;
      const auto prefix = [&](uint32_t x) {
        const uint32_t at = row + (x >> 5);
        return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(at * 4u), (int)pre) +
               (uint32_t)__popc((&mask[0][0])[at] & ((1u << (x & 31u)) - 1u));
      };
      const uint32_t pos = prefix(b) + (prefix(e) - prefix(w + 1));
      if (vol || sur) order[(vol ? numS : 0u) + pos] = (uint16_t)w;
    }
    __syncthreads();
    const RecordPiece* pieces = reinterpret_cast<const RecordPiece*>(stage);
    heldTile = tile;
    heldS = numS * 5u;
    heldAll = (numS + numV) * 5u;
    if (heldAll) {
#pragma unroll
      for (uint32_t k = 0; k < kHeld; k++) {
        if (k * kPathThreads >= heldAll) break;
        const uint32_t i = min(tid + k * kPathThreads, heldAll - 1u), j = i / 5u;
        held[k] = pieces[order[j] * kVertexWords8 + (i - j * 5u)];
      }
    }
    tile = next;
    __syncthreads();  // the records are read before the next tile is staged
  }
  writeHeld(heldPlace());
}

// ---- records routed by their EInsideVolume flag (SampleDataStorage.h:72-90):
// flag = surface | volume << 32 per record, inclusive scan, stable scatter
__global__ void __launch_bounds__(kPathThreads) k_route_flags(const PathSample* __restrict__ recs, uint32_t n,
                                                              unsigned long long* __restrict__ flags) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    flags[i] = (recs[i].flags & 2u) ? (1ull << 32) : 1ull;
}

__global__ void __launch_bounds__(kPathThreads) k_route_scatter(const PathSample* __restrict__ recs,
                                                                const unsigned long long* __restrict__ incl,
                                                                uint32_t n, PathSample* __restrict__ surfOut,
                                                                PathSample* __restrict__ volOut) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const PathSample r = recs[i];
    const unsigned long long c = incl[i];
    if (r.flags & 2u) volOut[(uint32_t)(c >> 32) - 1u] = r;
    else surfOut[(uint32_t)(c & 0xffffffffull) - 1u] = r;
  }
}

uint32_t path_grid(uint32_t n) {
  const uint32_t blocks = (n + kPathThreads - 1) / kPathThreads;
  return blocks < 65536u ? (blocks ? blocks : 1u) : 65536u;
}

}  // namespace

void launch_path_fused(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets, uint32_t numPaths,
                       const PathSampleOptions& o, PathSample* surfOut, PathSample* volOut, uint32_t* tileFirst,
                       unsigned long long* tileWord, FusedPathControl* control, uint32_t epoch, uint32_t numCUs,
                       unsigned long long* totals, hipStream_t s) {
  const uint32_t numTiles = (numSegments + kPathThreads - 1) / kPathThreads;
  hipLaunchKernelGGL(k_path_index, dim3(path_grid(numPaths + 1)), dim3(kPathThreads), 0, s, offsets, numPaths,
                     numSegments, numTiles, tileFirst, tileWord, control, epoch);
  hipLaunchKernelGGL(k_path_fused, dim3(std::min(numTiles, 3 * numCUs - 1) + 1), dim3(kPathThreads), 0, s, segs, numSegments,
                     offsets, numPaths, tileFirst, numTiles, o, reinterpret_cast<RecordPiece*>(surfOut),
                     reinterpret_cast<RecordPiece*>(volOut), tileWord, control, epoch, totals);
}

size_t path_scan_temp_bytes(uint32_t numSegments) {
  size_t bytes = 0;
  const unsigned long long* in = nullptr;
  unsigned long long* out = nullptr;
  PGL_KERNEL_CHECK(hipcub::DeviceScan::InclusiveSum(nullptr, bytes, in, out, (int)numSegments));
  return bytes;
}

size_t path_tile_words(uint32_t numSegments) { return (numSegments + kPathThreads - 1) / kPathThreads + 1; }

void launch_path_records(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets, uint32_t numPaths,
                         const PathSampleOptions& o, PathSample* records, unsigned long long* flags, uint32_t* pathOf,
                         uint32_t* tileFirst, unsigned long long* incl, void* scanTemp, size_t scanBytes,
                         bool checked, unsigned long long* totals, hipStream_t s) {
  if (!checked) hipLaunchKernelGGL(k_path_clear, dim3(1), dim3(64), 0, s, totals);
  if (numPaths == 0 || numSegments == 0) return;
  if (!checked)
    hipLaunchKernelGGL(k_path_check, dim3((numPaths + kPathThreads - 1) / kPathThreads), dim3(kPathThreads), 0, s,
                       offsets, numPaths, numSegments, totals);
  const uint32_t numTiles = (numSegments + kPathThreads - 1) / kPathThreads;
  hipLaunchKernelGGL(k_path_tiles, dim3(numTiles / kPathThreads + 1), dim3(kPathThreads), 0, s, offsets, numPaths,
                     numSegments, numTiles, tileFirst);
  hipLaunchKernelGGL(k_path_vertex, dim3(numTiles), dim3(kPathThreads), 0, s, segs, numSegments, offsets, numPaths,
                     tileFirst, o, records, flags, pathOf);
  PGL_KERNEL_CHECK(hipcub::DeviceScan::InclusiveSum(scanTemp, scanBytes, flags, incl, (int)numSegments, s));
  hipLaunchKernelGGL(k_path_totals, dim3(1), dim3(64), 0, s, incl, numSegments, totals);
}

void launch_path_scatter(const PathSample* records, const unsigned long long* flags, const uint32_t* pathOf,
                         const unsigned long long* incl, const uint32_t* offsets, uint32_t numSegments,
                         PathSample* surfOut, PathSample* volOut, hipStream_t s) {
  if (numSegments == 0) return;
  hipLaunchKernelGGL(k_path_scatter, dim3(path_grid(numSegments)), dim3(kPathThreads), 0, s, records, flags, pathOf,
                     incl, offsets, numSegments, surfOut, volOut);
}

void launch_route_count(const PathSample* recs, uint32_t n, unsigned long long* flags, unsigned long long* incl,
                        void* scanTemp, size_t scanBytes, unsigned long long* totals, hipStream_t s) {
  hipLaunchKernelGGL(k_path_clear, dim3(1), dim3(64), 0, s, totals);
  if (n == 0) return;
  hipLaunchKernelGGL(k_route_flags, dim3(path_grid(n)), dim3(kPathThreads), 0, s, recs, n, flags);
  PGL_KERNEL_CHECK(hipcub::DeviceScan::InclusiveSum(scanTemp, scanBytes, flags, incl, (int)n, s));
  hipLaunchKernelGGL(k_path_totals, dim3(1), dim3(64), 0, s, incl, n, totals);
}

void launch_route_scatter(const PathSample* recs, const unsigned long long* incl, uint32_t n, PathSample* surfOut,
                          PathSample* volOut, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_route_scatter, dim3(path_grid(n)), dim3(kPathThreads), 0, s, recs, incl, n, surfOut, volOut);
}

// ---- the variant that allocates nothing
//
// Its scratch (records, flags, their scan, path of each vertex, tile table,
// scan temporary storage, totals) is carved from one file-scope device array
// of a fixed size; each GPU holds its own copy for the life of the process.
// Host code reaches it only through the address hipGetSymbolAddress returns
// on that device.

namespace {

constexpr size_t na_align(size_t b) { return (b + 255) & ~size_t(255); }
constexpr size_t kNaRecords = 0;
constexpr size_t kNaFlags = kNaRecords + na_align(size_t(kNoAllocMaxVertices) * sizeof(PathSample));
constexpr size_t kNaIncl = kNaFlags + na_align(size_t(kNoAllocMaxVertices) * 8);
constexpr size_t kNaPathOf = kNaIncl + na_align(size_t(kNoAllocMaxVertices) * 8);
constexpr size_t kNaTiles = kNaPathOf + na_align(size_t(kNoAllocMaxVertices) * 4);
constexpr size_t kNaTotals = kNaTiles + na_align(size_t(kNoAllocMaxVertices / kPathThreads + 1) * 4);
constexpr size_t kNaScan = kNaTotals + 256;
constexpr size_t kNaScanBytes = size_t(1) << 18;  // the scan's temporary storage (checked at set-up)
constexpr size_t kNaBytes = kNaScan + kNaScanBytes;
static_assert(kNaBytes == kNoAllocScratchBytes, "scratch layout and its declared size differ");
constexpr int kNaMaxDevices = 64;

}  // namespace

static __device__ __align__(256) unsigned char scratch[kNaBytes];

// this device's copy of scratch, looked up once per device (with it current)
static unsigned char* noalloc_scratch() {
  static std::mutex lock;
  static unsigned char* ptr[kNaMaxDevices] = {};
  int dev = 0;
  PGL_KERNEL_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kNaMaxDevices) throw std::runtime_error("openpgl_amd: device index out of range");
  std::lock_guard<std::mutex> g(lock);
  if (!ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      throw std::runtime_error(std::string("openpgl_amd: hipGetSymbolAddress(scratch) failed: ") +
                               hipGetErrorString(e));
    if (path_scan_temp_bytes(kNoAllocMaxVertices) > kNaScanBytes)
      throw std::runtime_error("openpgl_amd: the path scan needs more temporary storage than the static scratch holds");
    ptr[dev] = static_cast<unsigned char*>(p);
  }
  return ptr[dev];
}

void path_prepare_noalloc(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets, uint32_t numPaths,
                          const PathSampleOptions& o, PathSample* surfOut, size_t surfCap, PathSample* volOut,
                          size_t volCap, size_t& numSurf, size_t& numVol, hipStream_t s) {
  numSurf = numVol = 0;
  if (numSegments > kNoAllocMaxVertices)
    throw std::runtime_error("openpgl_amd: the allocation-free path batch takes at most " +
                             std::to_string(kNoAllocMaxVertices) + " vertices per call (got " +
                             std::to_string(numSegments) + ")");
  unsigned char* base = noalloc_scratch();
  const uint32_t n = numPaths ? numSegments : 0;
  PathSample* records = reinterpret_cast<PathSample*>(base + kNaRecords);
  unsigned long long* flags = reinterpret_cast<unsigned long long*>(base + kNaFlags);
  unsigned long long* incl = reinterpret_cast<unsigned long long*>(base + kNaIncl);
  uint32_t* pathOf = reinterpret_cast<uint32_t*>(base + kNaPathOf);
  uint32_t* tiles = reinterpret_cast<uint32_t*>(base + kNaTiles);
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(base + kNaTotals);
  const size_t scanBytes = path_scan_temp_bytes(n > 0 ? n : 1u);
  if (scanBytes > kNaScanBytes) throw std::runtime_error("openpgl_amd: path scan storage exceeds the static scratch");
  launch_path_records(segs, n, offsets, numPaths, o, records, flags, pathOf, tiles, incl, base + kNaScan, scanBytes,
                      false, totals, s);
  unsigned long long t[3] = {0ull, 0ull, 0ull};
  PGL_KERNEL_CHECK(hipMemcpyAsync(t, totals, sizeof(t), hipMemcpyDeviceToHost, s));
  PGL_KERNEL_CHECK(hipStreamSynchronize(s));
  if (t[2]) throw std::runtime_error("openpgl_amd: path offsets must be non-decreasing and within the segments");
  numSurf = (size_t)t[0];
  numVol = (size_t)t[1];
  if (numSurf > surfCap || numVol > volCap)
    throw std::runtime_error("openpgl_amd: path samples exceed the output capacity (" + std::to_string(numSurf) +
                             " surface, " + std::to_string(numVol) + " volume)");
  if (numSurf == 0 && numVol == 0) return;
  launch_path_scatter(records, flags, pathOf, incl, offsets, n, surfOut, volOut, s);
  PGL_KERNEL_CHECK(hipStreamSynchronize(s));
}

}  // namespace pglgpu
