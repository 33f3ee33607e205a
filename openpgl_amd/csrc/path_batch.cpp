// Host side of the batched path-segment back-propagation (kernels_path.hip).
#include "path_batch.h"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace pglgpu {

static_assert(sizeof(PathSample) == kSampleRecordBytes, "PathSample is the 40-byte PGLSampleData record");

PathSampleBatch::PathSampleBatch() {
  PGL_HIP_CHECK(hipStreamCreate(&stream_));
  hTotals_.coherent = true;
}

PathSampleBatch::~PathSampleBatch() {
  (void)hipStreamSynchronize(stream_);
  (void)hipStreamDestroy(stream_);
}

void PathSampleBatch::count(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets, uint32_t numPaths,
                            const PathSampleOptions& o, bool checked) {
  offsets_ = offsets;
  numSegments_ = numPaths ? numSegments : 0;
  hTotals_.ensure(32);
  const size_t V = std::max<size_t>(numSegments_, 1);
  records_.ensure(V * sizeof(PathSample));
  flags_.ensure(V * 8);
  incl_.ensure(V * 8);
  pathOf_.ensure(V * 4);
  tiles_.ensure(path_tile_words((uint32_t)V) * 4);
  const size_t scanBytes = path_scan_temp_bytes(std::max<uint32_t>(numSegments_, 1));
  scanTemp_.ensure(std::max<size_t>(scanBytes, 16));
  launch_path_records(segs, numSegments_, offsets, numPaths, o, records_.as<PathSample>(),
                      flags_.as<unsigned long long>(), pathOf_.as<uint32_t>(), tiles_.as<uint32_t>(),
                      incl_.as<unsigned long long>(), scanTemp_.p, scanBytes, checked,
                      (unsigned long long*)hTotals_.dev, stream_);
}

void PathSampleBatch::scatter(PathSample* surfOut, PathSample* volOut) {
  launch_path_scatter(records_.as<PathSample>(), flags_.as<unsigned long long>(), pathOf_.as<uint32_t>(),
                      incl_.as<unsigned long long>(), offsets_, numSegments_, surfOut, volOut, stream_);
}

bool PathSampleBatch::totals(size_t& numSurf, size_t& numVol) {
  PGL_HIP_CHECK(hipStreamSynchronize(stream_));
  const unsigned long long* t = hTotals_.as<unsigned long long>();
  if (t[2]) throw std::runtime_error("openpgl_amd: path offsets must be non-decreasing and within the segments");
  numSurf = (size_t)t[0];
  numVol = (size_t)t[1];
  return t[3] == 0;
}

void PathSampleBatch::fused(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets, uint32_t numPaths,
                            const PathSampleOptions& o, PathSample* surfOut, PathSample* volOut, size_t& numSurf,
                            size_t& numVol) {
  numSurf = numVol = 0;
  if (numPaths == 0 || numSegments == 0) return;
  const size_t tiles = path_tile_words(numSegments);
  tiles_.ensure(tiles * 4);
  tileWords_.ensure(tiles * 16);
  hTotals_.ensure(32);
  if (!control_.p) {
    int dev = 0, cus = 0;
    PGL_HIP_CHECK(hipGetDevice(&dev));
    PGL_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    numCUs_ = (uint32_t)cus;
    control_.ensure(sizeof(FusedPathControl));
    PGL_HIP_CHECK(hipMemsetAsync(control_.p, 0, sizeof(FusedPathControl), stream_));
  }
  if (++epoch_ == 0) epoch_ = 1;
  launch_path_fused(segs, numSegments, offsets, numPaths, o, surfOut, volOut, tiles_.as<uint32_t>(),
                    tileWords_.as<unsigned long long>(), control_.as<FusedPathControl>(), epoch_, numCUs_,
                    (unsigned long long*)hTotals_.dev, stream_);
  if (totals(numSurf, numVol)) return;
  // Paths that the pass leaves: the counting launches.  The offsets are checked
  // and every record has room, so the scatter follows without a wait, which
  // makes up for the launches that found them: 12k vertices with one path of 65
  // take 73 us (91 with a check and a wait of their own, 76 by the counting
  // launches alone), 5.4M vertices with one 450 (468, 441 to 447), 1.5M with 1 %
  // of the paths of 65 to 200 vertices 470 (490, 498).
  count(segs, numSegments, offsets, numPaths, o, true);
  scatter(surfOut, volOut);
  totals(numSurf, numVol);
}

void PathSampleBatch::prepare(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets,
                              uint32_t numPaths, const PathSampleOptions& o, PathSample* surfOut, size_t surfCap,
                              PathSample* volOut, size_t volCap, size_t& numSurf, size_t& numVol) {
  if (surfCap >= numSegments && volCap >= numSegments && numSegments <= kFusedPathVertices)
    return fused(segs, numSegments, offsets, numPaths, o, surfOut, volOut, numSurf, numVol);
  count(segs, numSegments, offsets, numPaths, o, false);
  totals(numSurf, numVol);
  if (numSurf > surfCap || numVol > volCap)
    throw std::runtime_error("openpgl_amd: path samples exceed the output capacity (" + std::to_string(numSurf) +
                             " surface, " + std::to_string(numVol) + " volume)");
  if (numSurf == 0 && numVol == 0) return;
  scatter(surfOut, volOut);
  PGL_HIP_CHECK(hipStreamSynchronize(stream_));
}

void PathSampleBatch::prepareOwned(const PathVertex* segs, uint32_t numSegments, const uint32_t* offsets,
                                   uint32_t numPaths, const PathSampleOptions& o, const PathSample*& surf,
                                   size_t& numSurf, const PathSample*& vol, size_t& numVol) {
  const int b = next_;
  const size_t room = numPaths ? numSegments : 0;
  if (numSegments <= kFusedPathVertices && acquireOwned(b, room, room, true)) {
    fused(segs, numSegments, offsets, numPaths, o, out_[b][0].as<PathSample>(), out_[b][1].as<PathSample>(), numSurf,
          numVol);
  } else {
    count(segs, numSegments, offsets, numPaths, o, false);
    totals(numSurf, numVol);
    acquireOwned(b, numSurf, numVol);
    if (numSurf || numVol) {
      scatter(out_[b][0].as<PathSample>(), out_[b][1].as<PathSample>());
      PGL_HIP_CHECK(hipStreamSynchronize(stream_));
    }
  }
  next_ = 1 - next_;
  surf = out_[b][0].as<PathSample>();
  vol = out_[b][1].as<PathSample>();
  lastBuffer_ = b;
}

bool PathSampleBatch::acquireOwned(int b, size_t numSurf, size_t numVol, bool optional) {
  // the buffer's previous consumers (the gathers of an earlier update) must be done with it
  for (int k = 0; k < 2; k++)
    if (pendingRelease_[b][k]) {
      PGL_HIP_CHECK(hipStreamWaitEvent(stream_, released_[b][k], 0));
      pendingRelease_[b][k] = false;
    }
  const size_t ns = std::max<size_t>(numSurf, 1), nv = std::max<size_t>(numVol, 1);
  const bool refuse = optional && failNextFull;
  if (optional) failNextFull = false;
  if (refuse || out_[b][0].bytes < ns * sizeof(PathSample) || out_[b][1].bytes < nv * sizeof(PathSample))
    PGL_HIP_CHECK(hipStreamSynchronize(stream_));  // a reallocation frees memory the wait above protects
  if (!optional) {
    out_[b][0].ensure(ns * sizeof(PathSample));
    out_[b][1].ensure(nv * sizeof(PathSample));
    return true;
  }
  if (!refuse && out_[b][0].tryEnsure(ns * sizeof(PathSample)) && out_[b][1].tryEnsure(nv * sizeof(PathSample)))
    return true;
  out_[b][0].release();
  out_[b][1].release();
  return false;
}

void PathSampleBatch::routeOwned(const PathSample* recs, uint32_t n, const PathSample*& surf, size_t& numSurf,
                                 const PathSample*& vol, size_t& numVol) {
  const int b = next_;
  next_ = 1 - next_;
  totals_.ensure(24);
  hTotals_.ensure(32);
  const size_t V = std::max<size_t>(n, 1);
  flags_.ensure(V * 8);
  incl_.ensure(V * 8);
  const size_t scanBytes = path_scan_temp_bytes((uint32_t)V);
  scanTemp_.ensure(std::max<size_t>(scanBytes, 16));
  launch_route_count(recs, n, flags_.as<unsigned long long>(), incl_.as<unsigned long long>(), scanTemp_.p,
                     scanBytes, totals_.as<unsigned long long>(), stream_);
  PGL_HIP_CHECK(hipMemcpyAsync(hTotals_.p, totals_.p, 24, hipMemcpyDeviceToHost, stream_));
  PGL_HIP_CHECK(hipStreamSynchronize(stream_));
  const unsigned long long* t = hTotals_.as<unsigned long long>();
  numSurf = (size_t)t[0];
  numVol = (size_t)t[1];
  acquireOwned(b, numSurf, numVol);
  surf = out_[b][0].as<PathSample>();
  vol = out_[b][1].as<PathSample>();
  if (n) {
    launch_route_scatter(recs, incl_.as<unsigned long long>(), n, out_[b][0].as<PathSample>(),
                         out_[b][1].as<PathSample>(), stream_);
    PGL_HIP_CHECK(hipStreamSynchronize(stream_));
  }
  lastBuffer_ = b;
}

void PathSampleBatch::setReleased(hipEvent_t surfaceDone, hipEvent_t volumeDone) {
  const int b = lastBuffer_;
  released_[b][0] = surfaceDone;
  released_[b][1] = volumeDone;
  pendingRelease_[b][0] = surfaceDone != nullptr;
  pendingRelease_[b][1] = volumeDone != nullptr;
}

}  // namespace pglgpu
