// Sorted CSR rows from edge tuples without weights: a most-significant-digit
// partition of the records into leaves of a few thousand, each sorted in LDS
// (included by csr_build.hip).
//
// A record is (row, col), cb bits each (cb = bits of n - 1). The top `b` row
// bits choose its leaf; what is left of the key, (row low bits, col), is
// rem = 2 cb - b <= 32 bits and travels as one 32-bit word from the last
// partition pass on:
//
//   k_msd_hist    per-block histograms of the leaf digit (LDS)
//   k_msd_reduce  their sum, and the list of each sort kernel's leaves
//   k_scan        leaf offsets
//   k_msd_part1/2 tuples -> 64-bit keys by the first b1 bits (LDS-staged
//                 tiles, so a bucket's records leave in runs), then 64-bit
//                 keys -> 32-bit leaf keys by the next b2; one pass when
//                 b <= 8
//   k_leaf_bins   a leaf of at most kChunk records sorted in LDS, in place
//   k_leaf_sort, k_chunk_sort   the same by radix passes, where bins are crowded
//   k_leaf_merge  leaves above kChunk: their sorted chunks merged
//   k_scan, k_emit  duplicates dropped, columns and offsets out
//
// The sorts also count the records each emission tile keeps (the duplicates
// are seen there), so emission reads the keys once.
//
// Bound: passes over the records. 134 M records (R-MAT 22 tuples, both
// directions): 2.5 ms a call, against 7.0 ms for the six-pass
// least-significant-digit sort of 45-bit keys that the other forms take.
#pragma once

#include "csr_plan.h"

namespace ent {
namespace {

// Threads and records per thread of the partition passes (a tile of keys
// staged in LDS each). R-MAT 22, 134 M records: the first pass takes 400 us
// with 16,384 records a tile, 490 with 8,192 and 680 with 4,096 (its 256
// buckets get longer runs); the second, to 128 leaves a bucket, 450 us with
// 4,096 (four blocks fit a CU) and 570 with 8,192.
constexpr int kPart1Threads = 1024, kPart1Items = 16;
constexpr int kMaxFan = 256;                          // buckets of one partition pass
constexpr int kHistThreads = 1024;
constexpr int kLeafItems = 16;     // records per thread of the leaf sorts
constexpr int kLeafClasses = 3;    // leaves of at most 4096, 8192, 16384 records: 256, 512, 1024 threads
constexpr int kLeafSmall = 4096;
constexpr int kGroups = 256;       // key ranges a leaf's bins are spread over
constexpr unsigned kBinMax = 64;   // a bin of more records sends its leaf to k_leaf_sort
constexpr int kScanThreads = 1024;
constexpr int kScanItems = 32;
constexpr int kMergeTile = 2048;
constexpr int kMergeThreads = 256;
constexpr int kEmitThreads = 256;
constexpr int kEmitShift = 10;     // a wavefront emits 1024 consecutive records
constexpr unsigned kEmitTile = 1u << kEmitShift;

struct Chunk {
  unsigned start, size;         // records of this chunk
  unsigned leaf_start, leaf_end;
};

// Counters the reduce pass leaves for the host and the later kernels.
struct MsdCounts {
  unsigned leaves[kLeafClasses];  // leaves by sort class
  unsigned crowded[2];            // leaves, chunks left to the radix sort
  unsigned chunks;                // chunks of the leaves above kChunk
  unsigned max_size;              // largest leaf
  unsigned merged;                // records of the leaves above kChunk
};

// The (up to two) valid records of tuple i: bit 0 (u, v), bit 1 (v, u).
__device__ __forceinline__ int tuple_records(const BuildShape &s, unsigned u, unsigned v) {
  const unsigned n = unsigned(s.n);
  if (u >= n || v >= n || (s.no_loops && u == v)) return 0;
  return s.rev ? 3 : 1;
}

// Block histograms; also zeroes the counters of the later kernels.
__global__ __launch_bounds__(kHistThreads) void k_msd_hist(BuildShape s, MsdPlan p, const int *src, const int *dst,
                                                           unsigned *hist, MsdCounts *mc, unsigned *tile_cnt,
                                                           unsigned tiles, unsigned long long *ngaps) {
  extern __shared__ unsigned h[];
  if (blockIdx.y == 0) {
    const unsigned g = blockIdx.x * kHistThreads + threadIdx.x;
    for (unsigned i = g; i < tiles; i += gridDim.x * kHistThreads) tile_cnt[i] = 0;
    if (g < sizeof(MsdCounts) / 4) reinterpret_cast<unsigned *>(mc)[g] = 0;
    if (g == 0) *ngaps = 0;
  }
  const int nc = 1 << min(p.b, kHistBits);
  const unsigned base = unsigned(blockIdx.y) << kHistBits;
  for (int i = threadIdx.x; i < nc; i += kHistThreads) h[i] = 0;
  __syncthreads();
  const int sh = p.cb - p.b;
  auto add = [&](unsigned row) {
    const unsigned d = (row >> sh) - base;
    if (d < unsigned(nc)) atomicAdd(&h[d], 1u);
  };
  const long long nt = (long long)gridDim.x * kHistThreads;
  long long i = (long long)blockIdx.x * kHistThreads + threadIdx.x;
  // Four tuples per step keep eight loads in flight.
  for (; i + 3 * nt < s.ne; i += 4 * nt) {
    unsigned u[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u[j] = unsigned(src[i + j * nt]);
      v[j] = unsigned(dst[i + j * nt]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = tuple_records(s, u[j], v[j]);
      if (r & 1) add(u[j]);
      if (r & 2) add(v[j]);
    }
  }
  for (; i < s.ne; i += nt) {
    const unsigned u = unsigned(src[i]), v = unsigned(dst[i]);
    const int r = tuple_records(s, u, v);
    if (r & 1) add(u);
    if (r & 2) add(v);
  }
  __syncthreads();
  unsigned *out = hist + ((long long)blockIdx.x << p.b) + base;
  for (int k = threadIdx.x; k < nc; k += kHistThreads) out[k] = h[k];
}

// counts[leaf] = its records; lists the leaves each sort kernel takes
// (lists[c << b ...] for class c). A leaf above kChunk is listed as chunks of
// kChunk records (offsets within the leaf; k_chunk_place adds the leaf's
// start once it is known). 64 leaves per block; each wavefront sums a
// quarter of the blocks' histograms, eight loads in flight per lane.
__global__ __launch_bounds__(256) void k_msd_reduce(MsdPlan p, const unsigned *hist, unsigned *counts,
                                                    unsigned *lists, Chunk *chunks, MsdCounts *mc) {
  __shared__ unsigned part[4][kWave];
  const int wid = threadIdx.x / kWave, lane = lane_id();
  const unsigned leaf = blockIdx.x * kWave + lane, nl = 1u << p.b;
  unsigned x = 0;
  if (leaf < nl) {
    int k = wid;
    for (; k + 28 < p.nb; k += 32) {
      unsigned y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = hist[((long long)(k + 4 * j) << p.b) + leaf];
#pragma unroll
      for (int j = 0; j < 8; ++j) x += y[j];
    }
    for (; k < p.nb; k += 4) x += hist[((long long)k << p.b) + leaf];
  }
  part[wid][lane] = x;
  __syncthreads();
  if (wid) return;
  const unsigned c = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
  if (leaf < nl) counts[leaf] = c;
  unsigned top = 0;
#pragma unroll
  for (int k = 0; k < kLeafClasses; ++k) {
    const unsigned cap = unsigned(kLeafSmall) << k;
    const bool in = c > top && c <= cap;
    top = cap;
    const unsigned long long m = __ballot(in);
    if (!m) continue;
    unsigned at = 0;
    if (lane == 0) at = atomicAdd(&mc->leaves[k], unsigned(__popcll(m)));
    at = unsigned(__shfl(int(at), 0)) + unsigned(mask_rank(m));
    if (in) lists[((unsigned long long)k << p.b) + at] = leaf;
  }
  if (c > unsigned(kChunk)) {
    const unsigned k = (c + kChunk - 1) / kChunk;
    const unsigned at = atomicAdd(&mc->chunks, k);
    for (unsigned j = 0; j < k; ++j)
      chunks[at + j] = Chunk{j * kChunk, min(unsigned(kChunk), c - j * kChunk), leaf, 0u};
    atomicMax(&mc->max_size, c);
    atomicAdd(&mc->merged, c);
  }
}

// Replaces a chunk's leaf number by the leaf's range.
__global__ __launch_bounds__(256) void k_chunk_place(const MsdCounts *mc, const unsigned *off, Chunk *chunks) {
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < mc->chunks; i += gridDim.x * 256) {
    Chunk c = chunks[i];
    const unsigned leaf = c.leaf_start;
    c.leaf_start = off[leaf];
    c.leaf_end = off[leaf + 1];
    c.start += c.leaf_start;
    chunks[i] = c;
  }
}

// Exclusive sums of cnt[0 .. n) into off[0 .. n] (off[n] = total), by one
// block of 16 wavefronts with kScanItems coalesced rows of 64 entries each in
// flight (32,768 entries a step; n is at most some 100,000 at the benchmark
// sizes). With cur1, also the partition cursors: cur2 = off,
// cur1[q] = off[q << b2].
__global__ __launch_bounds__(kScanThreads) void k_scan(const unsigned *cnt, unsigned *off, unsigned n, unsigned *cur1,
                                                       unsigned *cur2, int b2) {
  __shared__ unsigned part[kScanThreads / kWave];
  const int wid = threadIdx.x / kWave, lane = lane_id();
  unsigned run = 0;
  for (unsigned base = 0; base < n; base += kScanThreads * kScanItems) {
    const unsigned i0 = base + unsigned(wid) * kWave * kScanItems + lane;
    unsigned x[kScanItems], t = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) x[j] = i0 + j * kWave < n ? cnt[i0 + j * kWave] : 0u;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {  // x[j] becomes its inclusive sum within the wavefront's entries
      x[j] = t + unsigned(wave_incl_scan(int(x[j])));
      t = unsigned(wave_read(int(x[j]), kWave - 1));
    }
    if (lane == 0) part[wid] = t;
    __syncthreads();
    unsigned before = run, all = 0;
#pragma unroll
    for (int k = 0; k < kScanThreads / kWave; ++k) {
      const unsigned y = part[k];
      if (k < wid) before += y;
      all += y;
    }
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
      const unsigned i = i0 + j * kWave;
      unsigned e = unsigned(__shfl_up(int(x[j]), 1));
      if (lane == 0) e = j ? unsigned(wave_read(int(x[j ? j - 1 : 0]), kWave - 1)) : 0u;
      e += before;
      if (i < n) {
        off[i] = e;
        if (cur1) {
          cur2[i] = e;
          if ((i & ((1u << b2) - 1)) == 0) cur1[i >> b2] = e;
        }
      }
    }
    run += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) off[n] = run;
}

// One staged tile of a partition pass: item(j, key) gives the thread's j-th
// record (false: none), key -> bucket (key >> shift) & (fan - 1), out[...] =
// Out(key & mask). A bucket's records of the tile leave LDS as one run.
template <int T, int I>
struct PartSmem {
  unsigned long long stage[T * I];
  unsigned cnt[kMaxFan], loc[kMaxFan], gb[kMaxFan];
  unsigned part[kMaxFan / kWave];
};

template <int T, int I, class Out, class Item>
__device__ __forceinline__ void part_tile(PartSmem<T, I> &sm, int shift, int fan, unsigned long long mask,
                                          unsigned *cursor, Out *out, Item item) {
  const int t = threadIdx.x;
  for (int k = t; k < kMaxFan; k += T) sm.cnt[k] = 0;
  __syncthreads();
  unsigned long long key[I];
  int rank[I];
#pragma unroll
  for (int j = 0; j < I; ++j) {
    const bool in = item(j, key[j]);
    rank[j] = in ? int(atomicAdd(&sm.cnt[(key[j] >> shift) & (fan - 1)], 1u)) : -1;
  }
  __syncthreads();
  unsigned c = 0, incl = 0;
  if (t < kMaxFan) {
    c = sm.cnt[t];
    incl = unsigned(wave_incl_scan(int(c)));
    if (lane_id() == kWave - 1) sm.part[t / kWave] = incl;
  }
  __syncthreads();
  if (t < kMaxFan) {
    unsigned before = 0;
    for (int k = 0; k < t / kWave; ++k) before += sm.part[k];
    sm.loc[t] = before + incl - c;
    sm.gb[t] = c ? atomicAdd(&cursor[t], c) : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < I; ++j)
    if (rank[j] >= 0) sm.stage[sm.loc[(key[j] >> shift) & (fan - 1)] + unsigned(rank[j])] = key[j];
  unsigned total = 0;
#pragma unroll
  for (int k = 0; k < kMaxFan / kWave; ++k) total += sm.part[k];
  __syncthreads();
  for (unsigned i = t; i < total; i += T) {
    const unsigned long long k = sm.stage[i];
    const unsigned d = unsigned(k >> shift) & unsigned(fan - 1);
    out[sm.gb[d] + (i - sm.loc[d])] = Out(k & mask);
  }
}

// First pass: tuples to buckets of the first b1 key bits.
template <class Out>
__global__ __launch_bounds__(kPart1Threads) void k_msd_part1(BuildShape s, MsdPlan p, const int *src, const int *dst,
                                                            unsigned *cursor, Out *out) {
  __shared__ PartSmem<kPart1Threads, kPart1Items> sm;
  const int per = s.rev ? kPart1Items / 2 : kPart1Items;
  const long long t0 = (long long)blockIdx.x * per * kPart1Threads + threadIdx.x;
  unsigned u[kPart1Items], v[kPart1Items];
#pragma unroll
  for (int j = 0; j < kPart1Items; ++j) {
    const long long i = t0 + (long long)j * kPart1Threads;
    const bool in = j < per && i < s.ne;
    u[j] = in ? unsigned(src[i]) : ~0u;
    v[j] = in ? unsigned(dst[i]) : ~0u;
  }
  const unsigned long long mask = sizeof(Out) == 8 ? ~0ull : (1ull << p.rem) - 1;
  part_tile<kPart1Threads, kPart1Items, Out>(sm, 2 * p.cb - p.b1, 1 << p.b1, mask, cursor, out, [&](int j, unsigned long long &key) {
    // With the reverse entries, item 2i is (u, v) and item 2i + 1 is (v, u).
    const bool back = s.rev && (j & 1);
    const unsigned a = s.rev ? u[j / 2] : u[j], c = s.rev ? v[j / 2] : v[j];
    key = ((unsigned long long)(back ? c : a) << p.cb) | (back ? a : c);
    return ((tuple_records(s, a, c) >> (back ? 1 : 0)) & 1) != 0;
  });
}

// Second pass: a tile of one first-pass bucket to its leaves.
__global__ __launch_bounds__(kPart2Threads) void k_msd_part2(MsdPlan p, const unsigned long long *in,
                                                            const unsigned *off, unsigned *cursor, unsigned *out) {
  __shared__ PartSmem<kPart2Threads, kPart2Items> sm;
  __shared__ unsigned first[kMaxFan + 1];
  __shared__ int bucket;
  const int t = threadIdx.x, fan1 = 1 << p.b1;
  unsigned c = 0, incl = 0;
  if (t < kMaxFan) {
    if (t < fan1) c = (off[(t + 1) << p.b2] - off[t << p.b2] + kPart2Tile - 1) / kPart2Tile;
    incl = unsigned(wave_incl_scan(int(c)));
    if (lane_id() == kWave - 1) sm.part[t / kWave] = incl;
  }
  if (t == 0) bucket = -1;
  __syncthreads();
  if (t < kMaxFan) {
    unsigned before = 0;
    for (int k = 0; k < t / kWave; ++k) before += sm.part[k];
    first[t] = before + incl - c;
    if (blockIdx.x >= first[t] && blockIdx.x < first[t] + c) bucket = t;
  }
  __syncthreads();
  const int q = bucket;
  if (q < 0) return;  // past the last tile
  const unsigned e = off[(q + 1) << p.b2];
  const unsigned s0 = off[q << p.b2] + (blockIdx.x - first[q]) * kPart2Tile;
  __syncthreads();  // sm.part is written again
  part_tile<kPart2Threads, kPart2Items, unsigned>(sm, 2 * p.cb - p.b, 1 << p.b2, (1ull << p.rem) - 1, cursor + ((long long)q << p.b2), out,
                      [&](int j, unsigned long long &key) {
                        const unsigned i = s0 + unsigned(j) * kPart2Threads + unsigned(t);
                        const bool ok = i < e;
                        key = ok ? in[i] : 0ull;
                        return ok;
                      });
}

// Adds to tcnt[tile - tile0] the kept records of a wavefront, tile = pos >>
// kEmitShift. Every lane of the wavefront calls it.
__device__ __forceinline__ void count_kept(unsigned *tcnt, unsigned tile0, unsigned pos, bool kept) {
  const unsigned tile = (pos >> kEmitShift) - tile0;
  unsigned long long m = __ballot(kept);
  while (m) {
    const unsigned t = unsigned(wave_read(int(tile), __ffsll((long long)m) - 1));
    const unsigned long long same = __ballot(kept && tile == t) & m;
    if (lane_id() == 0) atomicAdd(&tcnt[t], unsigned(__popcll(same)));
    m &= ~same;
  }
}

constexpr int kLeafTiles = (kChunk >> kEmitShift) + 2;  // emission tiles a leaf of kChunk records can touch

// One leaf of at most T * kLeafItems records, sorted in place by spreading
// its records over as many bins as it has records: the key's top 8 bits give
// one of kGroups ranges, whose records are counted; a range of c records gets
// c bins, evenly over the rest of the key. Bins then hold one or two records
// where the columns of a row are spread evenly (relabelled ids), and a
// record's place is its bin's start plus the smaller records of the bin. A
// leaf with a bin above kBinMax is left for k_leaf_sort.
//
// Bound: LDS operations, about ten per record (two counter updates, one
// scatter, the bin's bounds and its few records), against about 45 vector
// instructions per radix digit and record group for the ballot ranking of
// k_leaf_sort.
template <int T>
struct BinSmem {
  unsigned exch[T * kLeafItems];
  uint4 bins[T * kLeafItems / 8 + 1];  // 16-bit counters, then 16-bit starts, in pairs
  unsigned group[kGroups];  // record counts, then first bin | count << 16
  unsigned part[T / kWave];
  unsigned tcnt[kLeafTiles];
  int crowded;
};

// Work: the leaves of list (off[leaf] on, sorted in place), or, with chunks,
// the chunks themselves from src to dst. What is crowded is listed by leaf or
// chunk number.
template <int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T < 1024 ? 6 : 4))) void k_leaf_bins(MsdPlan p, int dedup, const unsigned *list, const Chunk *chunks,
                                                 const unsigned *nlist, const unsigned *off, const unsigned *src,
                                                 unsigned *dst, unsigned *tile_cnt, unsigned *crowded,
                                                 unsigned *ncrowded) {
  __shared__ BinSmem<T> sm;
  const int t = threadIdx.x, wid = t / kWave, lane = lane_id();
  const unsigned n = *nlist;
  unsigned *bins = reinterpret_cast<unsigned *>(sm.bins);
  auto start_of = [&](unsigned b) { return int((bins[b >> 1] >> ((b & 1) * 16)) & 0xFFFFu); };
  const int low = max(p.rem - 8, 0);                   // key bits below the group
  const int up = low ? 32 - low : 0;                   // ... moved to the top of a word
  for (unsigned li = blockIdx.x; li < n; li += gridDim.x) {
    const unsigned item = chunks ? li : list[li];
    const unsigned first = chunks ? chunks[li].start : off[item];
    const int size = chunks ? int(chunks[li].size) : int(off[item + 1] - first);
    unsigned key[kLeafItems];
#pragma unroll
    for (int j = 0; j < kLeafItems; ++j) {
      const int i = j * T + t;
      key[j] = i < size ? src[first + unsigned(i)] : 0u;
    }
    for (int k = t; k < kGroups; k += T) sm.group[k] = 0;
    for (int k = t; k < T * kLeafItems / 8 + 1; k += T) sm.bins[k] = make_uint4(0u, 0u, 0u, 0u);
    if (t < kLeafTiles) sm.tcnt[t] = 0;
    if (t == 0) sm.crowded = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLeafItems; ++j)
      if (j * T + t < size) atomicAdd(&sm.group[key[j] >> low], 1u);
    __syncthreads();
    unsigned c = 0, incl = 0;
    if (t < kGroups) {
      c = sm.group[t];
      incl = unsigned(wave_incl_scan(int(c)));
      if (lane == kWave - 1) sm.part[wid] = incl;
    }
    __syncthreads();
    if (t < kGroups) {
      unsigned before = incl - c;
      for (int k = 0; k < wid; ++k) before += sm.part[k];
      sm.group[t] = before | (c << 16);
    }
    __syncthreads();
    auto bin_of = [&](unsigned k) {
      const unsigned g = sm.group[k >> low];
      return (g & 0xFFFFu) + (up ? __umulhi(k << up, g >> 16) : 0u);
    };
    unsigned bin[kLeafItems];  // bin | rank among its records << 16
    bool over = false;
#pragma unroll
    for (int j = 0; j < kLeafItems; ++j) {
      bin[j] = 0;
      if (j * T + t < size) {
        const unsigned b = bin_of(key[j]), sh = (b & 1) * 16;
        const unsigned r = (atomicAdd(&bins[b >> 1], 1u << sh) >> sh) & 0xFFFFu;
        over |= r >= kBinMax;
        bin[j] = b | (r << 16);
      }
    }
    if (over) sm.crowded = 1;
    __syncthreads();
    if (sm.crowded) {  // the whole block
      if (t == 0) crowded[atomicAdd(ncrowded, 1u)] = item;
      __syncthreads();
      continue;
    }
    // Thread t turns the counts of bins 16 t .. 16 t + 15 into starts.
    uint4 w0 = sm.bins[2 * t], w1 = sm.bins[2 * t + 1];
    unsigned w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
    unsigned sum = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const unsigned a = w[k] & 0xFFFFu, b = w[k] >> 16;
      w[k] = sum | ((sum + a) << 16);
      sum += a + b;
    }
    const unsigned inc = unsigned(wave_incl_scan(int(sum)));
    if (lane == kWave - 1) sm.part[wid] = inc;
    __syncthreads();
    unsigned before = inc - sum;
    for (int k = 0; k < wid; ++k) before += sm.part[k];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] += before | (before << 16);
    sm.bins[2 * t] = make_uint4(w[0], w[1], w[2], w[3]);
    sm.bins[2 * t + 1] = make_uint4(w[4], w[5], w[6], w[7]);
    if (t == 0) bins[T * kLeafItems / 2] = unsigned(size);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLeafItems; ++j)
      if (j * T + t < size) sm.exch[start_of(bin[j] & 0xFFFFu) + int(bin[j] >> 16)] = key[j];
    __syncthreads();
    const unsigned tile0 = first >> kEmitShift;
#pragma unroll 4
    for (int j = 0; j < kLeafItems; ++j) {
      const int i = j * T + t;
      if (i - lane >= size) break;  // the whole wavefront
      bool kept = false;
      unsigned pos = first;
      if (i < size) {
        const unsigned k = sm.exch[i];
        const unsigned b = bin_of(k);
        const int s0 = start_of(b), s1 = start_of(b + 1);
        int at = s0;
        bool dup = false;
        for (int q = s0; q < s1; ++q) {
          const unsigned y = sm.exch[q];
          const bool eq = y == k && q < i;
          dup |= eq;
          at += (y < k || eq) ? 1 : 0;
        }
        pos = first + unsigned(at);
        dst[pos] = k;
        kept = !dup;
      }
      if (dedup) count_kept(sm.tcnt, tile0, pos, kept);
    }
    __syncthreads();
    if (dedup && t < kLeafTiles && sm.tcnt[t]) atomicAdd(&tile_cnt[tile0 + t], sm.tcnt[t]);
    __syncthreads();
  }
}

// Sorts src[start .. start + size) by the low `rem` bits into dst (the same
// place or another buffer). Lane l of wavefront w holds positions
// w * 64 * items + 64 j + l; each pass ranks a digit of at most 8 bits per
// wavefront (ballot matching, one LDS counter row per wavefront), scans the
// counters and exchanges the keys through LDS. Keys of ~0 pad the last
// wavefronts: they carry the largest digit in every pass and stay behind.
template <int T, int ITEMS>
struct LeafSmem {
  unsigned exch[T * ITEMS];
  unsigned short cnt[T / kWave][kMaxFan];
  unsigned part[kMaxFan / kWave];
  unsigned tcnt[kLeafTiles];
};

template <int T, int ITEMS>
__device__ __forceinline__ void leaf_sort(LeafSmem<T, ITEMS> &sm, const unsigned *src, unsigned *dst, unsigned start,
                                          int size, int rem, unsigned *tile_cnt) {
  constexpr int W = T / kWave;
  const int t = threadIdx.x, wid = t / kWave, lane = lane_id();
  const int items = (size + T - 1) / T;
  const int p0 = wid * kWave * items + lane;
  unsigned key[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int i = p0 + j * kWave;
    key[j] = j < items && i < size ? src[start + unsigned(i)] : ~0u;
  }
  const int passes = (rem + 7) / 8;
  int shift = 0;
  for (int ps = 0; ps < passes; ++ps) {
    const int bits = (rem - shift + passes - ps - 1) / (passes - ps);
    const unsigned dm = (1u << bits) - 1;
    for (int k = t; k < W * kMaxFan / 2; k += T) reinterpret_cast<unsigned *>(sm.cnt)[k] = 0;
    __syncthreads();
    int rank[ITEMS];
    volatile unsigned short *cw = sm.cnt[wid];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (j < items) {
        const unsigned d = (key[j] >> shift) & dm;
        unsigned long long m = ~0ull;
        for (int bit = 0; bit < bits; ++bit) {
          const bool one = (d >> bit) & 1;
          const unsigned long long bal = __ballot(one);
          m &= one ? bal : ~bal;
        }
        const int below = mask_rank(m);
        const int old = cw[d];
        rank[j] = old + below;
        wave_sync();
        if (below == 0) cw[d] = (unsigned short)(old + __popcll(m));
        wave_sync();
      }
    }
    __syncthreads();
    // Thread d < 256 turns digit d's per-wavefront counts into first
    // positions.
    unsigned tot = 0, incl = 0;
    if (t < kMaxFan) {
      for (int w = 0; w < W; ++w) {
        const unsigned x = sm.cnt[w][t];
        sm.cnt[w][t] = (unsigned short)tot;
        tot += x;
      }
      incl = unsigned(wave_incl_scan(int(tot)));
      if (lane == kWave - 1) sm.part[wid] = incl;
    }
    __syncthreads();
    if (t < kMaxFan) {
      unsigned base = incl - tot;
      for (int k = 0; k < wid; ++k) base += sm.part[k];
      for (int w = 0; w < W; ++w) sm.cnt[w][t] = (unsigned short)(sm.cnt[w][t] + base);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (j < items) sm.exch[sm.cnt[wid][(key[j] >> shift) & dm] + rank[j]] = key[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (j < items) key[j] = sm.exch[p0 + j * kWave];
    shift += bits;
  }
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int i = p0 + j * kWave;
    if (j < items && i < size) dst[start + unsigned(i)] = key[j];
  }
  // sm.exch holds the sorted records.
  if (tile_cnt) {
    const unsigned tile0 = start >> kEmitShift;
    for (int k = t; k < kLeafTiles; k += T) sm.tcnt[k] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const int i = p0 + j * kWave;
      if (j < items)
        count_kept(sm.tcnt, tile0, start + unsigned(i < size ? i : 0),
                   i < size && (i == 0 || sm.exch[i - 1] != key[j]));
    }
    __syncthreads();
    for (int k = t; k < kLeafTiles; k += T)
      if (sm.tcnt[k]) atomicAdd(&tile_cnt[tile0 + unsigned(k)], sm.tcnt[k]);
  }
  __syncthreads();
}

// Leaves of at most T * ITEMS records whose bins were crowded.
template <int T, int ITEMS>
__global__ __launch_bounds__(T) void k_leaf_sort(MsdPlan p, int dedup, const unsigned *list, const unsigned *nlist,
                                                 const unsigned *off, unsigned *keys, unsigned *tile_cnt) {
  __shared__ LeafSmem<T, ITEMS> sm;
  const unsigned n = *nlist;
  for (unsigned i = blockIdx.x; i < n; i += gridDim.x) {
    const unsigned leaf = list[i], s = off[leaf];
    leaf_sort<T, ITEMS>(sm, keys, keys, s, int(off[leaf + 1] - s), p.rem, dedup ? tile_cnt : nullptr);
  }
}

template <int T, int ITEMS>
__global__ __launch_bounds__(T) void k_chunk_sort(MsdPlan p, const Chunk *chunks, const unsigned *list,
                                                  const unsigned *nlist, const unsigned *src, unsigned *dst) {
  __shared__ LeafSmem<T, ITEMS> sm;
  const unsigned n = *nlist;
  for (unsigned i = blockIdx.x; i < n; i += gridDim.x) {
    const Chunk c = chunks[list[i]];
    leaf_sort<T, ITEMS>(sm, src, dst, c.start, int(c.size), p.rem, nullptr);
  }
}

// Records of a[0 .. na) among the first d outputs of merging a and b[0 .. nb)
// (a first among equals).
__device__ __forceinline__ unsigned merge_split(const unsigned *a, unsigned na, const unsigned *b, unsigned nb,
                                                unsigned d) {
  unsigned lo = d > nb ? d - nb : 0u, hi = min(d, na);
  while (lo < hi) {
    const unsigned mid = (lo + hi) >> 1;
    if (a[mid] <= b[d - 1 - mid]) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// One merge pass over the leaves above kChunk: pairs of runs of `run` records
// (a multiple of kChunk), kMergeTile outputs per block. With tile_cnt (the
// last pass of a build that drops duplicates) it counts the kept records.
__global__ __launch_bounds__(kMergeThreads) void k_leaf_merge(const Chunk *chunks, const unsigned *src, unsigned *dst,
                                                              unsigned long long run, unsigned *tile_cnt) {
  __shared__ unsigned buf[kMergeTile], outb[kMergeTile];
  __shared__ unsigned split[2];
  __shared__ unsigned tcnt[(kMergeTile >> kEmitShift) + 1];
  if (threadIdx.x <= (kMergeTile >> kEmitShift)) tcnt[threadIdx.x] = 0;
  const Chunk c = chunks[blockIdx.x];
  const unsigned t0 = blockIdx.y * kMergeTile;
  if (t0 >= c.size) return;
  const unsigned long long leaf = c.leaf_start, end = c.leaf_end;
  const unsigned long long pair = leaf + (c.start - leaf) / (2 * run) * (2 * run);
  const unsigned long long mid = min(pair + run, end), stop = min(pair + 2 * run, end);
  const unsigned *a = src + pair, *b = src + mid;
  const unsigned na = unsigned(mid - pair), nb = unsigned(stop - mid);
  const unsigned d0 = unsigned(c.start - pair) + t0;
  const unsigned cnt = min(unsigned(kMergeTile), c.size - t0);
  if (threadIdx.x % kWave == 0 && threadIdx.x < 2 * kWave)
    split[threadIdx.x / kWave] = merge_split(a, na, b, nb, threadIdx.x ? d0 + cnt : d0);
  __syncthreads();
  const unsigned a0 = split[0], ta = split[1] - a0, b0 = d0 - a0, tb = cnt - ta;
  for (unsigned i = threadIdx.x; i < cnt; i += kMergeThreads) buf[i] = i < ta ? a[a0 + i] : b[b0 + i - ta];
  __syncthreads();
  constexpr unsigned kPer = kMergeTile / kMergeThreads;
  const unsigned o = threadIdx.x * kPer;
  if (o < cnt) {
    unsigned i = merge_split(buf, ta, buf + ta, tb, o), j = o - i;
    for (unsigned k = o; k < min(o + kPer, cnt); ++k)
      outb[k] = j >= tb || (i < ta && buf[i] <= buf[ta + j]) ? buf[i++] : buf[ta + j++];
  }
  __syncthreads();
  const unsigned o0 = c.start + t0, tile0 = o0 >> kEmitShift;
  for (unsigned i = threadIdx.x; i < cnt; i += kMergeThreads) dst[o0 + i] = outb[i];
  if (!tile_cnt) return;
  // The record before the tile is the larger of the last ones taken.
  unsigned before = 0;
  if (a0) before = a[a0 - 1];
  if (b0) before = max(before, b[b0 - 1]);
  for (unsigned i0 = 0; i0 < cnt; i0 += kMergeThreads) {
    const unsigned i = i0 + threadIdx.x;
    const bool in = i < cnt;
    const bool kept = in && (i ? outb[i - 1] != outb[i] : d0 == 0 || before != outb[0]);
    count_kept(tcnt, tile0, o0 + (in ? i : 0u), kept);
  }
  __syncthreads();
  if (threadIdx.x <= (kMergeTile >> kEmitShift) && tcnt[threadIdx.x])
    atomicAdd(&tile_cnt[tile0 + threadIdx.x], tcnt[threadIdx.x]);
}

// Leaf of record i: the last l with off[l] <= i (64-way search, all lanes
// with the same i).
__device__ __forceinline__ int leaf_of(const unsigned *off, int b, unsigned i) {
  int lo = 0;
  for (int len = 1 << b; len > 1;) {
    const int st = max(1, len >> 6), k = lane_id() * st;
    const int c = __popcll(__ballot(k < len && off[lo + k] <= i));
    lo += (c - 1) * st;
    len = st;
  }
  return lo;
}

// The same for a lane's own i, within [lo, hi].
__device__ __forceinline__ int leaf_between(const unsigned *off, int lo, int hi, unsigned i) {
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Emission: each wavefront takes a tile of kEmitTile consecutive sorted
// records, drops those equal to their predecessor (dedup), writes the others'
// columns at their ranks and the offsets of the rows that start (or, empty,
// would start) there.
__global__ __launch_bounds__(kEmitThreads) void k_emit(BuildShape s, MsdPlan p, const unsigned *keys,
                                                       const unsigned *off, const unsigned *tile_off, unsigned tiles,
                                                       long long *beg, int *adj, Gap *gaps,
                                                       unsigned long long *ngaps) {
  const unsigned nrec = off[1u << p.b];
  if (nrec == 0) {  // no row: every offset is zero
    const long long nt = (long long)gridDim.x * kEmitThreads;
    for (long long v = (long long)blockIdx.x * kEmitThreads + threadIdx.x; v <= s.n; v += nt) beg[v] = 0;
    return;
  }
  const int lane = lane_id();
  const unsigned tile = blockIdx.x * (kEmitThreads / kWave) + threadIdx.x / kWave;
  if (tile >= tiles || ((unsigned long long)tile << kEmitShift) >= nrec) return;
  const unsigned first = tile << kEmitShift;
  const unsigned last = unsigned(min((unsigned long long)first + kEmitTile, (unsigned long long)nrec));
  const unsigned m = s.dedup ? tile_off[tiles] : nrec;
  unsigned base = s.dedup ? tile_off[tile] : first;
  const int lo = leaf_of(off, p.b, first ? first - 1 : 0), hi = leaf_of(off, p.b, last - 1);
  const int rsh = p.cb - p.b;  // row = leaf << rsh | key >> cb
  const unsigned colmask = unsigned((1ull << p.cb) - 1);
  auto row_of = [&](int leaf, unsigned key) {
    return (unsigned(leaf) << rsh) | unsigned((unsigned long long)key >> p.cb);
  };
  unsigned carry = first ? keys[first - 1] : 0u;
  int carry_row = first ? int(row_of(lo, carry)) : -1;
  constexpr int kStep = kEmitStep / kWave;  // loads in flight
  for (unsigned i0 = first; i0 < last; i0 += kStep * kWave) {
    unsigned key[kStep];
#pragma unroll
    for (int j = 0; j < kStep; ++j) {
      const unsigned long long i = (unsigned long long)i0 + unsigned(j * kWave + lane);
      key[j] = i < last ? keys[i] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kStep; ++j) {
      const unsigned long long i = (unsigned long long)i0 + unsigned(j * kWave + lane);
      const bool in = i < last;
      const int row = in ? int(row_of(leaf_between(off, lo, hi, unsigned(i)), key[j])) : 0;
      unsigned pk = unsigned(__shfl_up(int(key[j]), 1));
      int prow = __shfl_up(row, 1);
      if (lane == 0) {
        pk = carry;
        prow = carry_row;
      }
      carry = unsigned(wave_read(int(key[j]), kWave - 1));
      carry_row = wave_read(row, kWave - 1);
      const bool kept = in && !(s.dedup && prow == row && ((pk ^ key[j]) & colmask) == 0);
      const unsigned long long km = __ballot(kept);
      const unsigned pos = base + unsigned(mask_rank(km));
      base += unsigned(__popcll(km));
      if (kept) {
        adj[pos] = int(key[j] & colmask);
        if (row != prow) fill_rows(beg, (long long)prow + 1, (long long)row + 1, pos, gaps, ngaps);
        if (pos == m - 1) fill_rows(beg, (long long)row + 1, (long long)s.n + 1, m, gaps, ngaps);
      }
    }
  }
}

}  // namespace
}  // namespace ent
