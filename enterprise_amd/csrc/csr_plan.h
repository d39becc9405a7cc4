// Which sorted constructions take the partition of csr_msd.h, and its leaf
// bits and passes (host code without HIP, included by csr_msd.h).
//
// The partition pays as long as few records lie in leaves above kChunk, which
// are merged from sorted chunks, one pass over them for each doubling. Device
// times in ms of the partition and of the radix sort, and the merge passes
// times the share of the records they move:
//
//   134 M records, 16,384 rows       1.9  4.4   0
//                  4,096             3.0  4.3   2
//                  1,024             4.5  3.7   4
//                  256               4.6  3.6   6
//                  16                6.1  2.8  10
//                  2                 4.7  2.0  13
//     half of them in one row of 2^16  7.7  5.0   6.5
//     5% in one row of 2^16            3.9  5.1   0.5
//   67 M, all in one row of 2^16     5.2  2.6  13
//   8.4 M, 256 rows                  0.21 0.29  2
//          64                        0.23 0.22  4
//          16                        0.28 0.22  6
//
// so the radix sort takes what would be merged more than kMergeLimit times on
// average. Few rows are seen from the sizes alone; one long row by the host
// once the leaves are counted, while the first partition pass runs, and only
// from kSwitchRecords on: below, the whole call takes less than 0.6 ms in
// either form.
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

constexpr int64_t kMergeLimit = 3;
constexpr int64_t kSwitchRecords = 1 << 24;

// Merge passes of a leaf of `size` records.
inline int merge_passes(int64_t size) {
  int passes = 0;
  while ((int64_t(kChunk) << passes) < size) ++passes;
  return passes;
}

// Whether leaves above kChunk that hold `merged` records, the largest of them
// max_size, are better sorted by radix. Every pass moves all of them.
inline bool merges_too_much(int64_t records, int64_t merged, int64_t max_size) {
  return merged * merge_passes(max_size) > kMergeLimit * records;
}

struct MsdPlan {
  int cb, b, b1, b2, rem;
  int nb;     // histogram blocks
  int halves; // ranges of kHistBits-bit counters
};

// Leaf bits and partition passes for sorted rows without weights: `records`
// records of ne tuples, row and column of cb bits. False for more than
// kMsdMaxRecords, when the rest of a key would not fit 32 bits (n above
// 2^24), and when the mean leaf is eight chunks or more (the largest is larger
// still: four merge passes): those builds take the radix sort.
inline bool msd_plan(int64_t records, int64_t ne, int cb, MsdPlan *p) {
  p->cb = cb;
  const int least = std::max(0, 2 * cb - 32), most = std::min(cb, kMaxLeafBits);
  if (least > most || records > kMsdMaxRecords) return false;
  int b = 0;
  while (b < most && (records >> b) > kLeafTarget) ++b;
  if ((records >> b) >= 8 * kChunk) return false;
  p->b = std::max(b, least);
  p->b1 = std::min(p->b, 8);
  p->b2 = p->b - p->b1;
  p->rem = 2 * cb - p->b;
  p->nb = int(std::min<int64_t>(256, (ne + (1 << 14) - 1) >> 14));
  p->halves = p->b > kHistBits ? 2 : 1;
  return true;
}

}  // namespace ent
