// ljg_stage.h -- sizes of the pinned staging buffer and of a download's chunks (no HIP needed).
#pragma once

#include <cstddef>

namespace ljg {

// A context's staging buffer is pinned inside the call that first needs it, at up to 0.4 ms per MiB where the pages
// are new, so it is no larger than it has to be: the bytes wanted to the next 64 KiB, and half as much again as
// the buffer it replaces (a context whose systems grow does not pin for each of them), at most kRingBytes (uploads
// that go through it are smaller).
constexpr size_t kRingBytes = 8u << 20;
constexpr size_t kStageStep = 64u << 10;
inline size_t stage_capacity(size_t wanted, size_t had) {
  size_t cap = wanted > had + had / 2 ? wanted : had + had / 2;
  cap = (cap + kStageStep - 1) / kStageStep * kStageStep;
  if (cap > kRingBytes) cap = kRingBytes;
  return cap > wanted ? cap : wanted;
}

// Doubles per chunk of a download of `total`: an eighth, at least 256 KiB, where a chunk's transfer takes as long as
// its launch, at most 1 MiB, so that the ring holds eight.
constexpr size_t kMinChunk = (256u << 10) / sizeof(double), kMaxChunk = (1u << 20) / sizeof(double);
inline size_t download_chunk(size_t total) {
  const size_t eighth = (total + 7) / 8;
  return eighth < kMinChunk ? kMinChunk : eighth > kMaxChunk ? kMaxChunk : eighth;
}

}  // namespace ljg
