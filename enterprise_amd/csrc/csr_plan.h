// Which sorted constructions take the partition of csr_msd.h, and its leaf
// bits and passes (host code without HIP, included by csr_msd.h).
#pragma once

#include <algorithm>
#include <cstdint>

namespace ent {

constexpr int kPart2Threads = 512, kPart2Items = 8;  // second partition pass (csr_msd.h)
constexpr int kPart2Tile = kPart2Threads * kPart2Items;
constexpr int kHistBits = 15;      // leaf counters one block holds (128 KiB of LDS)
constexpr int kMaxLeafBits = 16;
constexpr int kChunk = 16384;      // largest leaf sorted whole; chunk of a merged one
constexpr int kLeafTarget = 4096;  // mean records per leaf aimed at
constexpr unsigned kEmitStep = 256;  // records a wavefront of k_emit takes at a time

// Records are numbered in 32 bits. The kernels step past the last one by less
// than a tile (kPart2Tile, kEmitStep) and round a leaf's size up to chunks, so
// the partition stops a chunk short of 2^32; what is left of the accepted
// sizes takes the radix sort, which numbers in 64 bits.
constexpr int64_t kMsdMaxRecords = INT64_C(0xFFFFFFFF) - kChunk;

struct MsdPlan {
  int cb, b, b1, b2, rem;
  int nb;     // histogram blocks
  int halves; // ranges of kHistBits-bit counters
};

// Leaf bits and partition passes for sorted rows without weights: `records`
// records of ne tuples, row and column of cb bits. False for more than
// kMsdMaxRecords, and when the rest of a key would not fit 32 bits (n above
// 2^24): those builds take the radix sort.
inline bool msd_plan(int64_t records, int64_t ne, int cb, MsdPlan *p) {
  p->cb = cb;
  const int least = std::max(0, 2 * cb - 32), most = std::min(cb, kMaxLeafBits);
  if (least > most || records > kMsdMaxRecords) return false;
  int b = 0;
  while (b < most && (records >> b) > kLeafTarget) ++b;
  p->b = std::max(b, least);
  p->b1 = std::min(p->b, 8);
  p->b2 = p->b - p->b1;
  p->rem = 2 * cb - p->b;
  p->nb = int(std::min<int64_t>(256, (ne + (1 << 14) - 1) >> 14));
  p->halves = p->b > kHistBits ? 2 : 1;
  return true;
}

}  // namespace ent
