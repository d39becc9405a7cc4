// Edge list to CSR on the device, behind include/ent_convert.h. The
// reference builds its CSR on the host, tuple by tuple, in file order
// (tuple_text_to_binary_csr/tuple_text_to_bin.cpp:190-248); this file
// sorts one record per stored entry.
//
// Sorted rows without weights, the form that the searches use, take the
// partition of csr_msd.h, as long as csr_plan.h's rules hold. Every other
// form, and what those rules leave out (n above 2^24, few or very long rows,
// record counts next to 2^32), gives each entry a 64-bit record and
// radix-sorts the records:
//
//   record r (tuple i = r / 2 with ENT_CSR_REVERSE, else i = r; the odd
//   record of a reversed tuple is (dst, src)):
//     input order : key = row                      (stable sort keeps tuple order)
//     sorted rows : key = row << cb | col          (cb = bits of n)
//   a dropped self-loop gets row = n and sorts behind every row.
//
// There, sorted rows without weights sort the keys alone; the others carry the
// record index (u32) to fetch the column and weight afterwards. Then, per
// tile of 4096 sorted records: the count of kept records (real row, and with
// dedup a key unlike its predecessor's), a scan of the tile counts, and one
// assembly pass that writes each kept record at its rank: its column and
// weight, and beg_pos at the row boundaries.
//
// HBM traffic per record of that form: the radix sort's passes over 8-byte keys
// (and 4-byte indices), one pass per 8 key bits; the record and assembly
// kernels read the tuples once and write the CSR once.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

#include "ent_bfs.h"
#include "ent_common.h"
#include "ent_convert.h"
#include "ent_device.h"
#include "ent_internal.h"

namespace ent {
namespace {

constexpr int kBuildBlock = 256;

// Bits needed for the values 0..x.
int bits_for(uint64_t x) {
  int b = 1;
  while (b < 64 && (uint64_t(1) << b) <= x) ++b;
  return b;
}

struct BuildShape {
  long long ne, records;
  int n, rev, no_loops, sorted, dedup, cb;
};

__device__ __forceinline__ void record_entry(const BuildShape &s, const int *src, const int *dst, long long r,
                                             long long &tuple, unsigned long long &row, unsigned long long &col) {
  tuple = s.rev ? r >> 1 : r;
  const bool back = s.rev && (r & 1);
  const int u = src[tuple], v = dst[tuple];
  row = (unsigned long long)(back ? v : u);
  col = (unsigned long long)(back ? u : v);
  if (s.no_loops && u == v) row = (unsigned long long)s.n;
}

__global__ __launch_bounds__(kBuildBlock) void k_records(BuildShape s, const int *src, const int *dst,
                                                         unsigned long long *keys, unsigned *idx) {
  for (long long r = (long long)blockIdx.x * kBuildBlock + threadIdx.x; r < s.records;
       r += (long long)gridDim.x * kBuildBlock) {
    long long t;
    unsigned long long row, col;
    record_entry(s, src, dst, r, t, row, col);
    keys[r] = s.sorted ? (row << s.cb) | (row == (unsigned long long)s.n ? 0ull : col) : row;
    if (idx) idx[r] = unsigned(r);
  }
}

// A run of empty rows too long for one thread: beg[v0 .. v1) = val.
struct Gap {
  long long v0, v1, val;
};
constexpr int kGapCap = 1 << 16;
constexpr long long kGapSerial = 256;  // longest run a thread fills itself

// Sets beg[v] = val for v in [v0, v1): by this thread when the run is
// short, else listed for k_fill_gaps (or by this thread if the list is full).
__device__ __forceinline__ void fill_rows(long long *beg, long long v0, long long v1, long long val, Gap *gaps,
                                          unsigned long long *ngaps) {
  if (v1 - v0 > kGapSerial) {
    const unsigned long long g = atomicAdd(ngaps, 1ull);
    if (g < (unsigned long long)kGapCap) {
      gaps[g] = Gap{v0, v1, val};
      return;
    }
  }
  for (long long v = v0; v < v1; ++v) beg[v] = val;
}

// Tiles of kTile sorted records, one block each. Record i is kept when its
// row is a real row (< n) and, with dedup, its key differs from record
// i - 1's (records of a dropped loop sort last, behind every kept one).
constexpr int kTileItems = 16;
constexpr long long kTile = (long long)kBuildBlock * kTileItems;

__device__ __forceinline__ bool record_kept(const BuildShape &s, const unsigned long long *keys, long long i,
                                            int shift) {
  const unsigned long long k = keys[i];
  if ((k >> shift) >= (unsigned long long)s.n) return false;
  return !s.dedup || i == 0 || keys[i - 1] != k;
}

__global__ __launch_bounds__(kBuildBlock) void k_tile_count(BuildShape s, const unsigned long long *keys,
                                                            unsigned long long *tile_cnt) {
  const int shift = s.sorted ? s.cb : 0;
  const long long t0 = (long long)blockIdx.x * kTile;
  int c = 0;
#pragma unroll 4
  for (int j = 0; j < kTileItems; ++j) {
    const long long i = t0 + (long long)j * kBuildBlock + threadIdx.x;
    if (i < s.records) c += record_kept(s, keys, i, shift) ? 1 : 0;
  }
  __shared__ int part[kBuildBlock / kWave];
  const int w = wave_sum(c);
  if (lane_id() == 0) part[threadIdx.x / kWave] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int k = 0; k < kBuildBlock / kWave; ++k) t += (unsigned long long)part[k];
    tile_cnt[blockIdx.x] = t;
  }
}

// Writes each kept record at its rank (tile_off[tile] + rank in the tile):
// its column and weight, and beg for the rows from the previous record's row
// (exclusive) to its own (inclusive) when its row starts there; the last kept
// record also fills beg for the rows after it, up to n. tile_off has
// ntiles + 1 entries (the last is m); beg is zero beforehand (for m = 0).
__global__ __launch_bounds__(kBuildBlock) void k_tile_assemble(BuildShape s, const unsigned long long *keys,
                                                               const unsigned *idx,
                                                               const unsigned long long *tile_off, const int *src,
                                                               const int *dst, const int *w_in, long long *beg,
                                                               int *adj, int *w_out, Gap *gaps,
                                                               unsigned long long *ngaps) {
  const int shift = s.sorted ? s.cb : 0;
  const unsigned long long colmask = (1ull << s.cb) - 1;
  const long long t0 = (long long)blockIdx.x * kTile;
  const long long m = (long long)tile_off[gridDim.x];
  long long base = (long long)tile_off[blockIdx.x];
  const int wid = threadIdx.x / kWave, lane = lane_id();
  __shared__ int wcnt[kBuildBlock / kWave];
  for (int j = 0; j < kTileItems; ++j) {
    const long long i = t0 + (long long)j * kBuildBlock + threadIdx.x;
    const bool kp = i < s.records && record_kept(s, keys, i, shift);
    const unsigned long long bal = __ballot(kp);
    if (lane == 0) wcnt[wid] = __popcll(bal);
    __syncthreads();
    long long pos = base + mask_rank(bal);
    long long step = 0;
    for (int k = 0; k < kBuildBlock / kWave; ++k) {
      if (k < wid) pos += wcnt[k];
      step += wcnt[k];
    }
    if (kp) {
      const unsigned long long key = keys[i];
      const long long row = (long long)(key >> shift);
      // Clamped: ids outside [0, n) (unchecked on the device form) cannot
      // send beg writes out of range.
      const long long prev = i == 0 ? -1 : (long long)min(keys[i - 1] >> shift, (unsigned long long)s.n);
      if (row != prev) fill_rows(beg, prev + 1, row + 1, pos, gaps, ngaps);
      if (pos == m - 1) fill_rows(beg, row + 1, (long long)s.n + 1, m, gaps, ngaps);
      if (idx) {
        long long t;
        unsigned long long r, col;
        record_entry(s, src, dst, (long long)idx[i], t, r, col);
        adj[pos] = int(col);
        if (w_out) w_out[pos] = w_in[t];
      } else {
        adj[pos] = int(key & colmask);
      }
    }
    base += step;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBuildBlock) void k_fill_gaps(const Gap *gaps, const unsigned long long *ngaps,
                                                           long long *beg) {
  const long long ng = (long long)min(*ngaps, (unsigned long long)kGapCap);
  for (long long g = blockIdx.x; g < ng; g += gridDim.x) {
    const Gap x = gaps[g];
    for (long long v = x.v0 + threadIdx.x; v < x.v1; v += kBuildBlock) beg[v] = x.val;
  }
}

}  // namespace
}  // namespace ent

#include "csr_msd.h"

namespace ent {
namespace {

int grid_for(long long items, int cus) {
  return int(std::max<long long>(1, std::min<long long>((long long)cus * 16, (items + kBuildBlock - 1) / kBuildBlock)));
}

struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) ignore(hipFree(p));
  }
  int alloc(int device, size_t bytes, const char *what) {
    if (device_malloc(device, &p, std::max<size_t>(bytes, 16)) != hipSuccess) {
      ignore(hipGetLastError());
      p = nullptr;
      return set_error(ENT_ENOMEM, "hipMalloc of %zu bytes (%s) failed", bytes, what);
    }
    return ENT_OK;
  }
  template <class T>
  T *as() const {
    return static_cast<T *>(p);
  }
};

// What one construction needs on a device: a stream, two events and a block
// of scratch memory. The calls take no handle, so the last idle context of
// each device waits here for the next one: allocating and freeing the scratch
// costs 0.6 ms a call at 1.6 GB, and the driver's clearing of freed memory
// stalls calls in a row for 10 to 1,000 ms. Bounded: one context per device,
// of at most kIdleBytes; concurrent calls make their own. Given back by
// ent_csr_release_scratch, when a library allocation fails and when a graph
// handle of the device is freed. A call takes it only once its own buffers are
// allocated, so that they can still have its memory.
constexpr size_t kIdleBytes = size_t(4) << 30;

struct BuildContext {
  int device = 0, cus = 0;
  hipStream_t stream = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr, e_counts = nullptr;
  struct Host {  // pinned
    long long m;
    MsdCounts counts;
  } *host = nullptr;
  void *mem = nullptr;
  size_t bytes = 0;
  BuildContext *next = nullptr;  // of the idle ones

  ~BuildContext() {
    if (hipSetDevice(device) != hipSuccess) return;
    if (e0) ignore(hipEventDestroy(e0));
    if (e1) ignore(hipEventDestroy(e1));
    if (e_counts) ignore(hipEventDestroy(e_counts));
    if (host) ignore(hipHostFree(host));
    if (stream) ignore(hipStreamDestroy(stream));
    if (mem) ignore(hipFree(mem));
  }
  int init(int dev) {
    device = dev;
    HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    HIP_TRY(hipEventCreateWithFlags(&e_counts, hipEventDisableTiming));
    HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&host), sizeof(Host), hipHostMallocDefault));
    HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    return ENT_OK;
  }
  int reserve(size_t want) {
    if (want <= bytes) return ENT_OK;
    if (mem) ignore(hipFree(mem));
    mem = nullptr;
    bytes = 0;
    if (device_malloc(device, &mem, want) != hipSuccess) {
      ignore(hipGetLastError());
      mem = nullptr;
      return set_error(ENT_ENOMEM, "hipMalloc of %zu bytes (construction scratch) failed", want);
    }
    bytes = want;
    return ENT_OK;
  }
};

std::mutex g_idle_mu;
// Never destroyed: the runtime may be gone when static objects are.
BuildContext *g_idle = nullptr;

// A call's hold on a context. The stream is drained before the context is
// idle again, also after an error.
struct ContextLease {
  std::unique_ptr<BuildContext> c;
  int take(int device) {
    {
      std::lock_guard<std::mutex> lk(g_idle_mu);
      for (BuildContext **p = &g_idle; *p; p = &(*p)->next)
        if ((*p)->device == device) {
          c.reset(*p);
          *p = c->next;
          c->next = nullptr;
          return ENT_OK;
        }
    }
    c.reset(new (std::nothrow) BuildContext());
    if (!c) return set_error(ENT_ENOMEM, "out of host memory");
    return c->init(device);
  }
  ~ContextLease() { give(); }
  void give() {
    std::unique_ptr<BuildContext> c = std::move(this->c);
    if (!c) return;
    if (!c->stream || !c->host || hipStreamSynchronize(c->stream) != hipSuccess || c->bytes > kIdleBytes) return;
    std::unique_ptr<BuildContext> other;  // freed behind the lock
    std::lock_guard<std::mutex> lk(g_idle_mu);
    BuildContext **p = &g_idle;
    while (*p && (*p)->device != c->device) p = &(*p)->next;
    if (*p) {  // another call came back first: keep the larger block
      if ((*p)->bytes >= c->bytes) {
        other = std::move(c);
        return;
      }
      other.reset(*p);
      c->next = other->next;
    }
    *p = c.release();
  }
};

// Offsets of a scratch block, 256-byte aligned.
struct Carver {
  size_t at = 0;
  size_t take(size_t bytes) {
    const size_t o = at;
    at += (std::max<size_t>(bytes, 16) + 255) / 256 * 256;
    return o;
  }
};

// Sorted rows without weights by partition (csr_msd.h). plan() sizes the
// scratch, run() queues the kernels.
struct MsdBuild {
  MsdPlan p;
  unsigned tiles = 0;
  size_t o_wide = 0, o_keys = 0, o_mc = 0, o_counts = 0, o_off = 0, o_cur1 = 0, o_cur2 = 0, o_lists = 0, o_crowded = 0,
         o_crowded2 = 0, o_chunks = 0, o_tc = 0, o_to = 0, o_hist = 0;

  void plan(const BuildShape &s, Carver &cv) {
    const size_t R = size_t(s.records), L = size_t(1) << p.b;
    tiles = unsigned((s.records + kEmitTile - 1) >> kEmitShift);
    o_keys = cv.take(4 * R);
    // 64-bit keys between the passes; afterwards the merge buffer.
    o_wide = cv.take(p.b2 ? 8 * R : R > size_t(kChunk) ? 4 * R : 0);
    o_mc = cv.take(sizeof(MsdCounts));
    o_counts = cv.take(4 * L);
    o_off = cv.take(4 * (L + 1));
    o_cur1 = cv.take(4 * kMaxFan);
    o_cur2 = cv.take(4 * L);
    o_lists = cv.take(4 * L * kLeafClasses);
    o_crowded = cv.take(4 * L);
    o_chunks = cv.take(sizeof(Chunk) * (2 * (R / kChunk) + 1));
    o_crowded2 = cv.take(4 * (2 * (R / kChunk) + 1));
    o_tc = cv.take(4 * size_t(tiles));
    o_to = cv.take(4 * (size_t(tiles) + 1));
    o_hist = cv.take(4 * L * size_t(p.nb));
  }

  template <int T>
  void sort_class(int k, hipStream_t stream, int cus, const BuildShape &s, const unsigned *lists, MsdCounts *mc,
                  const unsigned *off, unsigned *k32, unsigned *tile_cnt, unsigned *crowded) const {
    if (k && s.records <= (long long)kLeafSmall << (k - 1)) return;
    // Blocks that fit the LDS at once (27, 51 and 99 KB each).
    const unsigned grid = std::min(1u << p.b, unsigned(cus) * (k == 0 ? 6u : k == 1 ? 3u : 1u));
    hipLaunchKernelGGL(k_leaf_bins<T>, dim3(grid), dim3(T), 0, stream, p, s.dedup, lists + (size_t(k) << p.b),
                       nullptr, &mc->leaves[k], off, k32, k32, tile_cnt, crowded, &mc->crowded[0]);
  }

  // With `radix`, a build whose leaves would be merged too much ends behind the
  // first partition pass, with *radix set: the caller sorts the tuples.
  int run(BuildContext &c, const BuildShape &s, const int *src, const int *dst, long long *beg, int *adj, Gap *gaps,
          unsigned long long *ngaps, bool *radix) const {
    char *base = static_cast<char *>(c.mem);
    auto u = [&](size_t o) { return reinterpret_cast<unsigned *>(base + o); };
    unsigned *k32 = u(o_keys), *counts = u(o_counts), *off = u(o_off), *cur1 = u(o_cur1), *cur2 = u(o_cur2),
             *lists = u(o_lists), *crowded = u(o_crowded), *tile_cnt = u(o_tc), *tile_off = u(o_to), *hist = u(o_hist);
    unsigned long long *k64 = reinterpret_cast<unsigned long long *>(base + o_wide);
    MsdCounts *mc = reinterpret_cast<MsdCounts *>(base + o_mc);
    Chunk *chunks = reinterpret_cast<Chunk *>(base + o_chunks);
    hipStream_t stream = c.stream;
    const unsigned L = 1u << p.b;
    const size_t hist_lds = size_t(4) << std::min(p.b, kHistBits);
    // The attribute belongs to the function, not to this launch: always the
    // largest, whatever another thread builds meanwhile.
    HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_msd_hist), hipFuncAttributeMaxDynamicSharedMemorySize,
                                4 << kHistBits));
    hipLaunchKernelGGL(k_msd_hist, dim3(unsigned(p.nb), unsigned(p.halves)), dim3(kHistThreads), hist_lds, stream, s,
                       p, src, dst, hist, mc, tile_cnt, tiles, ngaps);
    hipLaunchKernelGGL(k_msd_reduce, dim3((L + kWave - 1) / kWave), dim3(256), 0, stream, p, hist, counts, lists,
                       chunks, mc);
    if (s.records > kChunk) {
      HIP_TRY(hipMemcpyAsync(&c.host->counts, mc, sizeof(MsdCounts), hipMemcpyDeviceToHost, stream));
      HIP_TRY(hipEventRecord(c.e_counts, stream));
    }
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(kScanThreads), 0, stream, counts, off, L, cur1, cur2, p.b2);
    const long long per = (s.rev ? kPart1Items / 2 : kPart1Items) * (long long)kPart1Threads;
    const unsigned t1 = unsigned((s.ne + per - 1) / per);
    if (p.b2)
      hipLaunchKernelGGL(k_msd_part1<unsigned long long>, dim3(t1), dim3(kPart1Threads), 0, stream, s, p, src, dst,
                         cur1, k64);
    else
      hipLaunchKernelGGL(k_msd_part1<unsigned>, dim3(t1), dim3(kPart1Threads), 0, stream, s, p, src, dst, cur1, k32);
    MsdCounts h{};
    if (radix) {
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipEventSynchronize(c.e_counts));
      h = c.host->counts;
      if ((*radix = merges_too_much(s.records, h.merged, h.max_size))) return ENT_OK;
    }
    if (p.b2) {
      const unsigned t2 = unsigned(s.records / kPart2Tile) + (1u << p.b1);
      hipLaunchKernelGGL(k_msd_part2, dim3(t2), dim3(kPart2Threads), 0, stream, p, k64, off, cur2, k32);
    }
    sort_class<256>(0, stream, c.cus, s, lists, mc, off, k32, tile_cnt, crowded);
    sort_class<512>(1, stream, c.cus, s, lists, mc, off, k32, tile_cnt, crowded);
    sort_class<1024>(2, stream, c.cus, s, lists, mc, off, k32, tile_cnt, crowded);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL((k_leaf_sort<1024, kLeafItems>), dim3(std::min(L, unsigned(c.cus) * 2)), dim3(1024), 0, stream,
                       p, s.dedup, crowded, &mc->crowded[0], off, k32, tile_cnt);
    HIP_TRY(hipGetLastError());
    if (s.records > kChunk) {
      // The copy was queued before the partition passes, so the device is
      // still busy with them when the host has it.
      if (!radix) {
        HIP_TRY(hipEventSynchronize(c.e_counts));
        h = c.host->counts;
      }
      if (h.chunks) {
        // The number of merge passes follows from the largest leaf; the
        // sorted chunks go where it leaves the result in k32.
        unsigned *other = reinterpret_cast<unsigned *>(k64);
        const int passes = merge_passes(h.max_size);
        hipLaunchKernelGGL(k_chunk_place, dim3(std::min((h.chunks + 255) / 256, 1024u)), dim3(256), 0, stream, mc, off,
                           chunks);
        unsigned *from = (passes & 1) ? other : k32, *to = (passes & 1) ? k32 : other;
        unsigned *crowded_chunks = u(o_crowded2);
        hipLaunchKernelGGL(k_leaf_bins<1024>, dim3(std::min(h.chunks, unsigned(c.cus))), dim3(1024), 0, stream, p, 0,
                           nullptr, chunks, &mc->chunks, off, k32, from, nullptr, crowded_chunks, &mc->crowded[1]);
        hipLaunchKernelGGL((k_chunk_sort<1024, kLeafItems>), dim3(std::min(h.chunks, unsigned(c.cus) * 2)),
                           dim3(1024), 0, stream, p, chunks, crowded_chunks, &mc->crowded[1], k32, from);
        for (int i = 0; i < passes; ++i) {
          hipLaunchKernelGGL(k_leaf_merge, dim3(h.chunks, kChunk / kMergeTile), dim3(kMergeThreads), 0, stream, chunks,
                             from, to, (unsigned long long)kChunk << i,
                             s.dedup && i == passes - 1 ? tile_cnt : nullptr);
          std::swap(from, to);
        }
        HIP_TRY(hipGetLastError());
      }
    }
    if (s.dedup)
      hipLaunchKernelGGL(k_scan, dim3(1), dim3(kScanThreads), 0, stream, tile_cnt, tile_off, tiles, nullptr, nullptr,
                         0);
    hipLaunchKernelGGL(k_emit, dim3((tiles + 3) / 4), dim3(kEmitThreads), 0, stream, s, p, k32, off, tile_off, tiles,
                       beg, adj, gaps, ngaps);
    HIP_TRY(hipGetLastError());
    return ENT_OK;
  }
};

// Every other form: a least-significant-digit radix sort of 64-bit keys, with
// the record index where rows keep the tuples' order or carry weights.
struct RadixBuild {
  bool keys_only = false;
  int kbits = 0;
  long long ntiles = 1;
  size_t o_k0 = 0, o_k1 = 0, o_i0 = 0, o_i1 = 0, o_tiles = 0, o_tmp = 0, sort_bytes = 0, scan_bytes = 0;

  int plan(const BuildShape &s, int bits, bool weights, hipStream_t stream, Carver &cv) {
    const size_t R = size_t(s.records);
    keys_only = s.sorted && !weights;
    kbits = bits;
    ntiles = std::max<long long>(1, (s.records + kTile - 1) / kTile);
    o_k0 = cv.take(8 * R);
    o_k1 = cv.take(8 * R);
    o_i0 = cv.take(keys_only ? 0 : 4 * R);
    o_i1 = cv.take(keys_only ? 0 : 4 * R);
    o_tiles = cv.take(8 * size_t(2 * ntiles + 1));
    // Scratch for the sort and the scan of tile counts.
    rocprim::double_buffer<unsigned long long> kb(nullptr, nullptr);
    rocprim::double_buffer<unsigned> vb(nullptr, nullptr);
    unsigned long long *none = nullptr;
    if (keys_only)
      HIP_TRY(rocprim::radix_sort_keys(nullptr, sort_bytes, kb, R, 0u, unsigned(kbits), stream));
    else
      HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort_bytes, kb, vb, R, 0u, unsigned(kbits), stream));
    HIP_TRY(rocprim::inclusive_scan(nullptr, scan_bytes, none, none, size_t(ntiles),
                                    rocprim::plus<unsigned long long>(), stream));
    o_tmp = cv.take(std::max(sort_bytes, scan_bytes));
    return ENT_OK;
  }

  int run(BuildContext &c, const BuildShape &s, const int *src, const int *dst, const int *w_in, long long *beg,
          int *adj, int *w_out, Gap *gaps, unsigned long long *ngaps) const {
    hipStream_t stream = c.stream;
    // beg starts at zero: with no kept record nothing else writes it.
    HIP_TRY(hipMemsetAsync(ngaps, 0, 8, stream));
    HIP_TRY(hipMemsetAsync(beg, 0, 8 * size_t(s.n + 1ll), stream));
    const size_t R = size_t(s.records);
    if (!R) return ENT_OK;
    char *base = static_cast<char *>(c.mem);
    auto u64 = [&](size_t o) { return reinterpret_cast<unsigned long long *>(base + o); };
    auto u32 = [&](size_t o) { return reinterpret_cast<unsigned *>(base + o); };
    rocprim::double_buffer<unsigned long long> kb(u64(o_k0), u64(o_k1));
    rocprim::double_buffer<unsigned> vb(u32(o_i0), u32(o_i1));
    void *tmp = base + o_tmp;
    hipLaunchKernelGGL(k_records, dim3(grid_for(s.records, c.cus)), dim3(kBuildBlock), 0, stream, s, src, dst,
                       kb.current(), keys_only ? nullptr : vb.current());
    HIP_TRY(hipGetLastError());
    size_t tb = sort_bytes;
    if (keys_only)
      HIP_TRY(rocprim::radix_sort_keys(tmp, tb, kb, R, 0u, unsigned(kbits), stream));
    else
      HIP_TRY(rocprim::radix_sort_pairs(tmp, tb, kb, vb, R, 0u, unsigned(kbits), stream));
    // Kept records per tile, their running sum, then every kept record at its
    // rank.
    unsigned long long *tile_cnt = u64(o_tiles), *tile_off = tile_cnt + ntiles;
    HIP_TRY(hipMemsetAsync(tile_cnt, 0, 8 * size_t(2 * ntiles + 1), stream));
    hipLaunchKernelGGL(k_tile_count, dim3(unsigned(ntiles)), dim3(kBuildBlock), 0, stream, s, kb.current(), tile_cnt);
    HIP_TRY(hipGetLastError());
    tb = scan_bytes;
    HIP_TRY(rocprim::inclusive_scan(tmp, tb, tile_cnt, tile_off + 1, size_t(ntiles),
                                    rocprim::plus<unsigned long long>(), stream));
    hipLaunchKernelGGL(k_tile_assemble, dim3(unsigned(ntiles)), dim3(kBuildBlock), 0, stream, s, kb.current(),
                       keys_only ? nullptr : vb.current(), tile_off, src, dst, w_in, beg, adj, w_out, gaps, ngaps);
    HIP_TRY(hipGetLastError());
    return ENT_OK;
  }
};

// The whole construction on the context's stream; w_in/w_out may be null.
int build_csr(BuildContext &c, long long n, long long ne, const int *src, const int *dst,
              const int *w_in, int flags, long long *beg, int *adj, long long adj_cap, int *w_out,
              long long *m_out, ent_build_stats *st) {
  if (n < 0 || n > INT32_MAX || ne < 0) return set_error(ENT_EINVAL, "bad sizes n=%lld ne=%lld", n, ne);
  if (flags & ~(ENT_CSR_REVERSE | ENT_CSR_NO_LOOPS | ENT_CSR_SORT | ENT_CSR_DEDUP))
    return set_error(ENT_EINVAL, "unknown flags 0x%x", flags);
  BuildShape s{};
  s.ne = ne;
  s.rev = (flags & ENT_CSR_REVERSE) != 0;
  s.records = ne * (s.rev ? 2 : 1);
  s.n = int(n);
  s.no_loops = (flags & ENT_CSR_NO_LOOPS) != 0;
  s.dedup = (flags & ENT_CSR_DEDUP) != 0;
  s.sorted = s.dedup || (flags & ENT_CSR_SORT) != 0;
  s.cb = bits_for(uint64_t(std::max<long long>(n - 1, 0)));
  if (s.records >= (1ll << 32)) return set_error(ENT_EINVAL, "%lld records: at most 2^32 - 1", s.records);
  if (adj_cap < s.records) return set_error(ENT_EINVAL, "adjacency capacity %lld < %lld records", adj_cap, s.records);
  const int kbits = s.sorted ? s.cb + bits_for(uint64_t(n)) : bits_for(uint64_t(n));
  if (kbits > 64) return set_error(ENT_EINVAL, "key of %d bits", kbits);
  Carver cv;
  const size_t o_cnt = cv.take(16), o_gaps = cv.take(sizeof(Gap) * kGapCap);
  MsdBuild msd;
  RadixBuild radix;
  const bool part = s.records && s.sorted && !w_in && msd_plan(s.records, s.ne, s.cb, &msd.p);
  int rc = ENT_OK;
  // A large build by partition may turn to the radix sort, in the same scratch.
  bool turn = part && s.records >= kSwitchRecords, turned = false;
  Carver cr = cv;
  if (part) msd.plan(s, cv);
  if ((!part || turn) && (rc = radix.plan(s, kbits, w_in != nullptr, c.stream, cr))) return rc;
  if (!part) cv = cr;
  if (turn && c.reserve(std::max(cv.at, cr.at))) {
    clear_error();
    turn = false;  // no room for that
  }
  if ((rc = c.reserve(cv.at))) return rc;
  char *mem = static_cast<char *>(c.mem);
  unsigned long long *ngaps = reinterpret_cast<unsigned long long *>(mem + o_cnt);
  Gap *gaps = reinterpret_cast<Gap *>(mem + o_gaps);
  hipStream_t stream = c.stream;
  HIP_TRY(hipEventRecord(c.e0, stream));
  if (part && (rc = msd.run(c, s, src, dst, beg, adj, gaps, ngaps, turn ? &turned : nullptr))) return rc;
  if ((!part || turned) && (rc = radix.run(c, s, src, dst, w_in, beg, adj, w_out, gaps, ngaps))) return rc;
  hipLaunchKernelGGL(k_fill_gaps, dim3(c.cus * 4), dim3(kBuildBlock), 0, stream, gaps, ngaps, beg);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(c.e1, stream));
  HIP_TRY(hipMemcpyAsync(&c.host->m, beg + n, 8, hipMemcpyDeviceToHost, stream));
  HIP_TRY(hipStreamSynchronize(stream));
  const long long m = c.host->m;
  *m_out = m;
  if (st) {
    std::memset(st, 0, sizeof *st);
    st->records = s.records;
    st->m = m;
    st->key_bits = kbits;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, c.e0, c.e1) == hipSuccess) st->device_ms = ms;
  }
  return ENT_OK;
}

// Tuple ids are checked on the host: the kernels index rows by them.
int check_tuples(int64_t n, int64_t ne, const int32_t *src, const int32_t *dst) {
  if (n < 0 || n > INT32_MAX || ne < 0) return set_error(ENT_EINVAL, "bad sizes n=%lld ne=%lld", (long long)n, (long long)ne);
  std::atomic<int64_t> bad{-1};
  parallel_for(ne, 1 << 16, [&](int64_t b, int64_t e) {
    for (int64_t i = b; i < e; ++i)
      if (src[i] < 0 || src[i] >= n || dst[i] < 0 || dst[i] >= n) {
        bad.store(i);
        return;
      }
  });
  const int64_t i = bad.load();
  if (i >= 0)
    return set_error(ENT_EINVAL, "tuple %lld (%d, %d) outside [0, %lld)", (long long)i, src[i], dst[i], (long long)n);
  return ENT_OK;
}

// Device buffers for host tuples (and weights), and the CSR built of them.
struct HostBuild {
  DevBuf s, d, w, beg, adj, w_out;
  int alloc(int device, int64_t n, int64_t ne, int64_t records, bool weights) {
    int rc;
    if ((rc = s.alloc(device, 4 * size_t(ne), "tuples")) || (rc = d.alloc(device, 4 * size_t(ne), "tuples")) ||
        (rc = beg.alloc(device, 8 * size_t(n + 1), "offsets")) ||
        (rc = adj.alloc(device, 4 * size_t(records), "adjacency")))
      return rc;
    if (weights && ((rc = w.alloc(device, 4 * size_t(ne), "weights")) ||
                    (rc = w_out.alloc(device, 4 * size_t(records), "weights"))))
      return rc;
    return ENT_OK;
  }
  int upload(hipStream_t stream, int64_t ne, const int32_t *src, const int32_t *dst, const int32_t *weight) {
    if (ne) {
      HIP_TRY(hipMemcpyAsync(s.p, src, 4 * size_t(ne), hipMemcpyHostToDevice, stream));
      HIP_TRY(hipMemcpyAsync(d.p, dst, 4 * size_t(ne), hipMemcpyHostToDevice, stream));
      if (weight) HIP_TRY(hipMemcpyAsync(w.p, weight, 4 * size_t(ne), hipMemcpyHostToDevice, stream));
    }
    return ENT_OK;
  }
};

}  // namespace

void build_give_back(int device) {
  std::unique_ptr<BuildContext> c;  // freed behind the lock
  std::lock_guard<std::mutex> lk(g_idle_mu);
  for (BuildContext **p = &g_idle; *p; p = &(*p)->next)
    if ((*p)->device == device) {
      c.reset(*p);
      *p = c->next;
      return;  // there is one per device
    }
}

}  // namespace ent

using namespace ent;

extern "C" {

int ent_csr_release_scratch(int32_t device) {
  clear_error();
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess) {
    ignore(hipGetLastError());
    ndev = 0;
  }
  if (device < 0 || device >= ndev) return set_error(ENT_EINVAL, "device %d of %d", device, ndev);
  build_give_back(device);
  return ENT_OK;
}

// For tests, not in the public headers: bytes of scratch kept idle on `device`.
int64_t ent_internal_scratch_bytes(int32_t device) {
  std::lock_guard<std::mutex> lk(g_idle_mu);
  for (const BuildContext *c = g_idle; c; c = c->next)
    if (c->device == device) return int64_t(c->bytes);
  return 0;
}

int ent_csr_build_device(int32_t device, int64_t n, int64_t ne, const int32_t *src_dev, const int32_t *dst_dev,
                         int32_t flags, int64_t *beg_pos_dev, int32_t *adj_dev, int64_t adj_capacity,
                         int64_t *m_out, ent_build_stats *st) {
  clear_error();
  if (!beg_pos_dev || !m_out || (ne > 0 && (!src_dev || !dst_dev || !adj_dev)))
    return set_error(ENT_EINVAL, "NULL argument");
  HIP_TRY(hipSetDevice(device));
  ContextLease ctx;
  int rc = ctx.take(device);
  if (rc) return rc;
  long long m = 0;
  rc = build_csr(*ctx.c, n, ne, src_dev, dst_dev, nullptr, flags, reinterpret_cast<long long *>(beg_pos_dev), adj_dev,
                 adj_capacity, nullptr, &m, st);
  if (rc) return rc;
  *m_out = m;
  return ENT_OK;
}

int ent_csr_build(int32_t device, int64_t n, int64_t ne, const int32_t *src, const int32_t *dst,
                  const int32_t *weight, int32_t flags, ent_csr *out, int32_t **weight_out, ent_build_stats *st) {
  clear_error();
  if (!out || (ne > 0 && (!src || !dst))) return set_error(ENT_EINVAL, "NULL argument");
  int rc = check_tuples(n, ne, src, dst);
  if (rc) return rc;
  std::memset(out, 0, sizeof *out);
  if (weight_out) *weight_out = nullptr;
  HIP_TRY(hipSetDevice(device));
  const int64_t records = ne * ((flags & ENT_CSR_REVERSE) ? 2 : 1);
  HostBuild hb;
  ContextLease ctx;
  if ((rc = hb.alloc(device, n, ne, records, weight != nullptr)) || (rc = ctx.take(device))) return rc;
  hipStream_t stream = ctx.c->stream;
  long long m = 0;
  if ((rc = hb.upload(stream, ne, src, dst, weight)) ||
      (rc = build_csr(*ctx.c, n, ne, hb.s.as<int>(), hb.d.as<int>(), hb.w.as<int>(), flags, hb.beg.as<long long>(),
                      hb.adj.as<int>(), records, hb.w_out.as<int>(), &m, st)))
    return rc;
  int64_t *beg = static_cast<int64_t *>(std::malloc(8 * size_t(n + 1)));
  int32_t *adj = static_cast<int32_t *>(std::malloc(4 * size_t(std::max<long long>(m, 1))));
  int32_t *wh = weight_out && weight ? static_cast<int32_t *>(std::malloc(4 * size_t(std::max<long long>(m, 1)))) : nullptr;
  auto fail = [&](int code) {
    std::free(beg);
    std::free(adj);
    std::free(wh);
    return code;
  };
  if (!beg || !adj || (weight_out && weight && !wh))
    return fail(set_error(ENT_ENOMEM, "out of host memory (%lld entries)", m));
  hipError_t e = hipMemcpyAsync(beg, hb.beg.p, 8 * size_t(n + 1), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess && m) e = hipMemcpyAsync(adj, hb.adj.p, 4 * size_t(m), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess && wh && m) e = hipMemcpyAsync(wh, hb.w_out.p, 4 * size_t(m), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return fail(set_error(ENT_EDEVICE, "copy of the CSR to the host failed: %s", hipGetErrorString(e)));
  out->n = n;
  out->m = m;
  out->beg_pos = beg;
  out->adj = adj;
  if (weight_out) *weight_out = wh;
  return ENT_OK;
}

int ent_graph_upload_edges(const int32_t *src, const int32_t *dst, int64_t n, int64_t ne, int32_t flags,
                           int32_t device, int32_t upload_flags, ent_graph **out) {
  clear_error();
  if (!out) return set_error(ENT_EINVAL, "out is NULL");
  *out = nullptr;
  if (ne > 0 && (!src || !dst)) return set_error(ENT_EINVAL, "NULL argument");
  if (n < 1) return set_error(ENT_EINVAL, "n=%lld < 1", (long long)n);
  int rc = check_tuples(n, ne, src, dst);
  if (rc) return rc;
  HIP_TRY(hipSetDevice(device));
  const int64_t records = ne * ((flags & ENT_CSR_REVERSE) ? 2 : 1);
  HostBuild hb;
  ContextLease ctx;
  if ((rc = hb.alloc(device, n, ne, records, false)) || (rc = ctx.take(device))) return rc;
  hipStream_t stream = ctx.c->stream;
  long long m = 0;
  if ((rc = hb.upload(stream, ne, src, dst, nullptr)) ||
      (rc = build_csr(*ctx.c, n, ne, hb.s.as<int>(), hb.d.as<int>(), nullptr, flags, hb.beg.as<long long>(),
                      hb.adj.as<int>(), records, nullptr, &m, nullptr)))
    return rc;
  // The offsets come back for the host-side degree tables; the adjacency is
  // copied device to device into the handle's CSR.
  std::vector<int64_t> beg(size_t(n) + 1);
  HIP_TRY(hipMemcpyAsync(beg.data(), hb.beg.p, 8 * size_t(n + 1), hipMemcpyDeviceToHost, stream));
  HIP_TRY(hipStreamSynchronize(stream));
  ctx.give();
  return upload_graph(beg.data(), hb.adj.as<int32_t>(), true, n, m, device, upload_flags, out);
}

}  // extern "C"
