// Several levels per launch for graphs of low degree and high diameter
// (grids, road networks). The reference runs one level at a time with the
// host in between (bfs_gpu_opt.cuh:66-288).
//
// One level per launch costs a launch and a chain of about five dependent
// memory round trips (queue entry, row offsets, adjacency, claim, counts) for
// a frontier of a few thousand vertices: 9.7 us a level on a 4096 x 4096
// grid, whatever the frontier's size. Here a block takes its share of the
// frontier's queue through kDeepLevels levels on its own, in LDS, and only
// then hands the vertices of the last of them to the next launch:
//
//  - A neighbour u of a vertex at depth d is claimed with atomicMin(depth[u],
//    d + 1); the claim is won if the old depth was larger. Blocks do not wait
//    for each other, so a block may reach a vertex by a longer way first: the
//    block that finds the shorter one lowers the depth and expands the vertex
//    again. When the launch ends, a vertex at true distance at most L + K has
//    its depth: some vertex one closer got its own true depth by a claim, and
//    the block that made that claim expanded it.
//  - Each claim knows the depth it replaced, so the launch's counts of
//    vertices per level are exact.
//  - Queue entries lowered after they were queued are skipped: their depth is
//    below the queue's level.
//  - A claim loads the vertex's neighbours beside the atomic, from a copy of
//    the adjacency in rows of 4 or 8 padded entries, so a level is one memory
//    round trip and a block barrier. Degrees above 8 take the CSR: offsets
//    beside the claim, then the adjacency, two round trips.
//
// Bound: the round trip of a claim, about 1.4 us a level with its barrier, plus
// 7.4 us a launch. 4096 x 4096 grid, 6,229 levels: 62 -> 10.4 ms (18.2 with 8
// levels a launch and the CSR, 11.9 with 16 and padded rows); 200 x 200: 2.27
// -> 0.49 ms. Many sources fill the chip with claims: 24 to 30 G a second.
//
// A launch derives its state from the previous launch's state and counts, as
// the other forms do. A block whose level outgrows its LDS queue, or a launch
// that outgrows the striped queues, marks the search failed and the caller
// runs it the ordinary way. The block stops there: a sparse random graph's first
// batch, whose every source outgrows its block within ten levels (131,072
// vertices of mean degree 4, 256 sources), takes 390 us more than a later one's
// 490; with blocks that went on to the last level it was 3,750 more.
#include <hip/hip_runtime.h>

#include <cstring>
#include <new>
#include <thread>

#include "ent_bfs.h"
#include "ent_common.h"
#include "ent_deep.h"
#include "ent_device.h"

namespace ent {
namespace {

constexpr int kDeepBS = 128;
constexpr int kDeepChunk = 256;   // queue entries a block takes through its levels at a time
constexpr int kDeepShare = 4;    // fewest entries given to a block
constexpr int kDeepLatencySources = 4;  // up to here a batch waits for its chains (see SKIP)
constexpr unsigned kDeepTagMul = 0x9E3779B1u;

// An LDS queue entry: the vertex's neighbours (-1 behind the last), or, for
// W = 0, its row start << 5 | degree (in the last level's queue: the vertex).
template <int W>
struct DeepEntry {
  int4 n[W];
};
template <>
struct DeepEntry<0> {
  unsigned long long row;
};

// SKIP: the entries carry their vertex too, and a claimed vertex's row leaves
// out the one that claimed it, whose depth is smaller: a quarter of a grid's
// claims. That pays where the chip is full of claims (2048 x 2048 grid, 64
// sources: 44.9 -> 35.8 ms, 16: 12.9 -> 11.1) and not where one search waits
// for its own (4096 x 4096: 10.4 -> 11.0 ms). kCap: LDS queue entries per
// level and block; four blocks fit a CU (W = 1).
template <int W, bool SKIP>
struct DeepSmem {
  static constexpr int kCap = SKIP ? 768 : 1024;
  DeepEntry<W> q[2][kCap];
  int id[2][SKIP ? kCap : 1];
  unsigned lcnt[3];
  int nf[kDeepLevels + 1];
  unsigned long long mf;
  int ovf;
  unsigned base;
  unsigned qpre[kDeepStripes + 1];
  DeepState S;
};

// State of this launch in sm.S, the queue's stripe prefix in sm.qpre.
template <int W, bool SKIP>
__device__ __forceinline__ void deep_begin(const DeepArgs &a, DeepSmem<W, SKIP> &sm, DeepCtl *c, long long i) {
  if (threadIdx.x < kWave) {
    const int lane = threadIdx.x;
    constexpr int kWords = int(sizeof(DeepState) / 4);
    static_assert(kWords > kWave && kWords <= 2 * kWave, "two state words per lane");
    const unsigned *s32 = reinterpret_cast<const unsigned *>(&c->st[(i + 1) & 1]);
    const unsigned w0 = s32[lane], w1 = lane + kWave < kWords ? s32[lane + kWave] : 0u;
    const uint4 *src = reinterpret_cast<const uint4 *>(&c->cnt[(i + 2) % 3][lane * kDeepStripeU32]);
    const uint4 h = src[0];
    unsigned long long mf = (static_cast<unsigned long long>(h.y) << 32) | h.x;
    const unsigned qn = h.z;
    const unsigned flags = wave_or32(h.w);
    int nf[kDeepLevels];
#pragma unroll
    for (int j = 0; j < kDeepLevels; j += 4) {
      const uint4 y = src[1 + j / 4];
      nf[j] = int(y.x);
      nf[j + 1] = int(y.y);
      nf[j + 2] = int(y.z);
      nf[j + 3] = int(y.w);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mf += __shfl_xor(mf, o);
#pragma unroll
    for (int j = 0; j < kDeepLevels; ++j) nf[j] = wave_sum(nf[j]);
    unsigned *d32 = reinterpret_cast<unsigned *>(&sm.S);
    d32[lane] = w0;
    if (lane + kWave < kWords) d32[lane + kWave] = w1;
    wave_sync();
    DeepState &S = sm.S;
    const bool advance = !S.done && S.launches > 0;  // the first launch takes the given state
    if (advance) S.qn[lane] = min(qn, unsigned(a.qcap_s));
    wave_sync();
    if (lane == 0 && !S.done) {
      if (advance) {
        int last = 0;
        unsigned long long all = 0;
#pragma unroll
        for (int j = 0; j < kDeepLevels; ++j) {
          all += (unsigned long long)nf[j];
          if (nf[j] > 0) last = j + 1;
        }
        S.total_nf += all;
        S.total_mf += mf;
        S.par ^= 1;
        if (flags) {
          S.error = DEEP_OVERFLOW;
          S.done = 1;
        } else if (nf[kDeepLevels - 1] == 0) {
          S.levels = S.level + last + 1;
          S.td_levels += last + 1;
          S.done = 1;
        } else {
          S.level += kDeepLevels;
          S.td_levels += kDeepLevels;
        }
        if (S.done) S.t_end = rt_clock();
      }
      S.launches += 1;
    }
    wave_sync();
    const int incl = wave_incl_scan(int(S.qn[lane]));
    sm.qpre[lane + 1] = unsigned(incl);
    if (lane == 0) {
      sm.qpre[0] = 0;
      sm.mf = 0;
      sm.ovf = 0;
    }
    if (lane <= kDeepLevels) sm.nf[lane] = 0;
    wave_sync();
    if (blockIdx.x == 0) {
      const unsigned *o32 = reinterpret_cast<const unsigned *>(&S);
      unsigned *p32 = reinterpret_cast<unsigned *>(&c->st[i & 1]);
      for (int w = lane; w < kWords; w += kWave) p32[w] = o32[w];
      if (lane < kDeepHostWords) {
        const unsigned tag = unsigned(S.launches) + unsigned(S.search) * kDeepTagMul;
        a.hmir[((long long)blockIdx.y * 2 + (i & 1)) * kDeepHostWords + lane] =
            (static_cast<unsigned long long>(tag) << 32) | o32[lane];
      }
      uint4 *z = reinterpret_cast<uint4 *>(&c->cnt[(i + 1) % 3][lane * kDeepStripeU32]);
#pragma unroll
      for (int w = 0; w < (DK_NF + kDeepLevels) / 4; ++w) z[w] = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  __syncthreads();
}

// The neighbours of one entry, four at a time: claims them at depth nd and
// queues the ones won. Every lane of the wavefront calls it.
template <int W, bool SKIP>
struct DeepStep {
  const DeepArgs &a;
  DeepSmem<W, SKIP> &sm;
  unsigned *depth;
  int L;
  unsigned long long &mf;

  __device__ __forceinline__ void claim(const int (&u)[4], int self, int j, DeepEntry<W> *out, int *oid, unsigned *ocnt) {
    const unsigned nd = unsigned(L + j + 1);
    const int lane = lane_id();
    unsigned old[4];
    DeepEntry<W> row[4];
    int deg[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const bool in = u[x] >= 0;
      old[x] = in ? atomicMin(depth + u[x], nd) : 0u;
      if constexpr (W > 0) {
#pragma unroll
        for (int y = 0; y < W; ++y)
          row[x].n[y] = in ? reinterpret_cast<const int4 *>(a.rows)[(long long)u[x] * W + y] : make_int4(-1, -1, -1, -1);
      } else {
        const long long s = in ? a.off[u[x]] : 0, e = in ? a.off[u[x] + 1] : 0;
        deg[x] = int(e - s);
        row[x].row = ((unsigned long long)s << 5) | (unsigned long long)(e - s);
      }
    }
    int won = 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) won += old[x] > nd ? 1 : 0;
    const int incl = wave_incl_scan(won);
    const int all = wave_read(incl, kWave - 1);
    if (all == 0) return;
    unsigned pos = 0;
    if (lane == 0) {
      pos = atomicAdd(ocnt, unsigned(all));
      atomicAdd(&sm.nf[j + 1], all);
    }
    pos = unsigned(__builtin_amdgcn_readfirstlane(int(pos))) + unsigned(incl - won);
    const bool last = !SKIP && j + 1 == kDeepLevels;
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (old[x] > nd) {
        if constexpr (W > 0) {
          deg[x] = 0;
#pragma unroll
          for (int y = 0; y < W; ++y)
            deg[x] += (row[x].n[y].x >= 0) + (row[x].n[y].y >= 0) + (row[x].n[y].z >= 0) + (row[x].n[y].w >= 0);
#pragma unroll
          for (int y = 0; SKIP && y < W; ++y) {
            int4 &r = row[x].n[y];
            r.x = r.x == self ? -1 : r.x;
            r.y = r.y == self ? -1 : r.y;
            r.z = r.z == self ? -1 : r.z;
            r.w = r.w == self ? -1 : r.w;
          }
          if (last) row[x].n[0].x = u[x];
        } else {
          if (last) row[x].row = (unsigned long long)u[x];
        }
        if (old[x] == ~0u) mf += (unsigned long long)deg[x];
        else atomicSub(&sm.nf[old[x] - unsigned(L)], 1);
        if (pos < unsigned(sm.kCap)) {
          out[pos] = row[x];
          if constexpr (SKIP) oid[pos] = u[x];
        } else {
          sm.ovf = 1;
        }
        ++pos;
      }
  }
};

// Launch i: the next kDeepLevels levels of source blockIdx.y.
template <int W, bool SKIP>
__global__ __launch_bounds__(kDeepBS) void k_deep(DeepArgs a, long long i) {
  __shared__ DeepSmem<W, SKIP> sm;
  DeepCtl *c = a.ctl + blockIdx.y;
  deep_begin<W, SKIP>(a, sm, c, i);
  if (sm.S.done) return;
  const unsigned total = sm.qpre[kDeepStripes];
  const unsigned share = max((total + gridDim.x - 1) / gridDim.x, unsigned(kDeepShare));
  const unsigned begin = blockIdx.x * share, end = min(begin + share, total);
  if (begin >= total) return;
  const int t = threadIdx.x, wid = t / kWave, lane = lane_id();
  const int L = sm.S.level;
  const int *qin = a.q[sm.S.par & 1] + (long long)blockIdx.y * a.qstride;
  int *qout = a.q[(sm.S.par & 1) ^ 1] + (long long)blockIdx.y * a.qstride;
  unsigned *depth = reinterpret_cast<unsigned *>(a.depth + (long long)blockIdx.y * a.dstride);
  const int stripe = int(blockIdx.x) % a.nstripe;
  unsigned *cs = &c->cnt[i % 3][stripe * kDeepStripeU32];
  unsigned long long mf = 0;
  DeepStep<W, SKIP> step{a, sm, depth, L, mf};
  for (unsigned c0 = begin; c0 < end; c0 += kDeepChunk) {
    const unsigned nc = min(unsigned(kDeepChunk), end - c0);
    if (t < 3) sm.lcnt[t] = t == 0 ? nc : 0u;
    for (unsigned k = t; k < nc; k += kDeepBS) {
      const unsigned x = c0 + k;
      int lo = 0, hi = kDeepStripes - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sm.qpre[mid] <= x) lo = mid;
        else hi = mid - 1;
      }
      const int v = qin[(long long)lo * a.qcap_s + (x - sm.qpre[lo])];
      const bool live = depth[v] == unsigned(L);  // not lowered since it was queued
      DeepEntry<W> ent;
      if constexpr (W > 0) {
#pragma unroll
        for (int y = 0; y < W; ++y) {
          ent.n[y] = reinterpret_cast<const int4 *>(a.rows)[(long long)v * W + y];
          if (!live) ent.n[y] = make_int4(-1, -1, -1, -1);
        }
      } else {
        const long long s = a.off[v], e = a.off[v + 1];
        ent.row = live ? ((unsigned long long)s << 5) | (unsigned long long)(e - s) : 0ull;
      }
      sm.q[0][k] = ent;
      if constexpr (SKIP) sm.id[0][k] = v;
    }
    int j = 0;
    unsigned cnt = 0;
    for (; j < kDeepLevels; ++j) {
      __syncthreads();
      // Not written in this level, so the whole block sees the same.
      cnt = sm.lcnt[j % 3];
      if (cnt == 0 || cnt > unsigned(sm.kCap)) break;
      if (t == 0) sm.lcnt[(j + 2) % 3] = 0;
      const DeepEntry<W> *in = sm.q[j & 1];
      DeepEntry<W> *out = sm.q[(j + 1) & 1];
      int *oid = SKIP ? sm.id[(j + 1) & 1] : nullptr;
      unsigned *ocnt = &sm.lcnt[(j + 1) % 3];
      for (unsigned k0 = unsigned(wid) * kWave; k0 < cnt; k0 += kDeepBS) {
        const unsigned k = k0 + lane;
        if constexpr (W > 0) {
          const int self = SKIP && k < cnt ? sm.id[j & 1][k] : -2;
#pragma unroll
          for (int y = 0; y < W; ++y) {
            const int4 r = k < cnt ? in[k].n[y] : make_int4(-1, -1, -1, -1);
            if (y > 0 && __ballot((r.x & r.y & r.z & r.w) >= 0) == 0) break;
            const int u[4] = {r.x, r.y, r.z, r.w};
            step.claim(u, self, j, out, oid, ocnt);
          }
        } else {
          const unsigned long long ent = k < cnt ? in[k].row : 0ull;
          const int deg = int(ent & 31);
          const long long s = (long long)(ent >> 5);
          for (int i0 = 0; __ballot(i0 < deg) != 0; i0 += 4) {
            int u[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) u[x] = i0 + x < deg ? a.adj[s + i0 + x] : -1;
            step.claim(u, -2, j, out, oid, ocnt);
          }
        }
      }
    }
    __syncthreads();
    if (cnt > unsigned(sm.kCap)) break;  // failed: sm.ovf is set
    if (j == kDeepLevels) {
      cnt = min(sm.lcnt[kDeepLevels % 3], unsigned(sm.kCap));
      if (t == 0 && cnt) {
        const unsigned b = atomicAdd(&cs[DK_QN], cnt);
        if (b + cnt > unsigned(a.qcap_s)) sm.ovf = 1;
        sm.base = b;
      }
      __syncthreads();
      const unsigned b = sm.base;
      const DeepEntry<W> *out = sm.q[kDeepLevels & 1];
      for (unsigned k = t; k < cnt; k += kDeepBS)
        if (b + k < unsigned(a.qcap_s)) {
          int v;
          if constexpr (SKIP) v = sm.id[kDeepLevels & 1][k];
          else if constexpr (W > 0) v = out[k].n[0].x;
          else v = int(out[k].row);
          qout[(long long)stripe * a.qcap_s + b + k] = v;
        }
      __syncthreads();
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mf += __shfl_xor(mf, o);
  if (lane == 0 && mf) atomicAdd(&sm.mf, mf);
  __syncthreads();
  if (t == 0 && sm.mf) atomicAdd(reinterpret_cast<unsigned long long *>(&cs[DK_MF]), sm.mf);
  if (t == kWave && sm.ovf) atomicOr(&cs[DK_FLAGS], 1u);
  if (t >= 1 && t <= kDeepLevels && sm.nf[t]) atomicAdd(&cs[DK_NF + t - 1], unsigned(sm.nf[t]));
}

// Padded rows of 4 W entries.
template <int W>
__global__ __launch_bounds__(256) void k_deep_rows(const long long *off, const int *adj, long long n, int4 *rows) {
  for (long long v = (long long)blockIdx.x * 256 + threadIdx.x; v < n; v += (long long)gridDim.x * 256) {
    const long long s = off[v], e = off[v + 1];
    int u[4 * W];
#pragma unroll
    for (int x = 0; x < 4 * W; ++x) u[x] = s + x < e ? adj[s + x] : -1;
#pragma unroll
    for (int y = 0; y < W; ++y) rows[v * W + y] = make_int4(u[4 * y], u[4 * y + 1], u[4 * y + 2], u[4 * y + 3]);
  }
}

// Rows of a batch: every entry -1.
__global__ __launch_bounds__(256) void k_deep_fill(int *rows, long long n) {
  const long long gt = (long long)blockIdx.x * 256 + threadIdx.x, nt = (long long)gridDim.x * 256;
  // 16-byte stores from the first aligned entry (rows are 4-byte aligned).
  const long long head = min(n, (long long)((0ull - reinterpret_cast<unsigned long long>(rows)) & 15ull) >> 2);
  const long long nq = (n - head) >> 2;
  int4 *q = reinterpret_cast<int4 *>(rows + head);
  for (long long i = gt; i < nq; i += nt) q[i] = make_int4(-1, -1, -1, -1);
  const long long t0 = head + (nq << 2);
  if (gt < head) rows[gt] = -1;
  else if (gt < head + (n - t0)) rows[t0 + (gt - head)] = -1;
}

// Source blockIdx.x: its root at depth 0, queued, and a fresh state.
__global__ __launch_bounds__(256) void k_deep_seed(DeepArgs a, const int *roots, int search) {
  const int s = blockIdx.x, root = roots[s];
  DeepCtl *c = a.ctl + s;
  for (int k = threadIdx.x; k < 3 * kDeepStripes * kDeepStripeU32; k += 256) (&c->cnt[0][0])[k] = 0;
  if (threadIdx.x) return;
  a.depth[(long long)s * a.dstride + root] = 0;
  a.q[0][(long long)s * a.qstride] = root;
  DeepState S{};
  S.search = search;
  S.total_nf = 1;
  S.total_mf = (unsigned long long)(a.off[root + 1] - a.off[root]);
  S.qn[0] = 1;
  c->st[1] = S;
}

// Adds 8 + 12 deg(v) for every distinct depth of vertex v among the at most
// R <= 64 rows of group blockIdx.y.
template <int R>
__global__ __launch_bounds__(256) void k_deep_joint(const long long *off, const int *rows, const int *order, int n,
                                                    int k, unsigned long long *bytes) {
  const int r0 = blockIdx.y * 64, nr = min(64, k - r0);
  unsigned long long sum = 0;
  for (long long v = (long long)blockIdx.x * 256 + threadIdx.x; v < n; v += (long long)gridDim.x * 256) {
    int seen[R];
    int distinct = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) seen[r] = r < nr ? rows[(long long)order[r0 + r] * n + v] : -1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int dup = seen[r] >> 31;  // 0, or -1 where unreached
#pragma unroll
      for (int q = 0; q < r; ++q) dup |= seen[q] == seen[r] ? 1 : 0;
      distinct += dup ? 0 : 1;
    }
    sum += (unsigned long long)distinct * (8ull + 12ull * (unsigned long long)(off[v + 1] - off[v]));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane_id() == 0 && sum) atomicAdd(bytes, sum);
}

bool read_deep(const DeepWorkspace *w, int s, int slot, DeepState *out, unsigned *tag) {
  const volatile unsigned long long *m = w->h_mir + (size_t(s) * 2 + size_t(slot)) * kDeepHostWords;
  unsigned word[kDeepHostWords];
  const unsigned t0 = unsigned(m[0] >> 32);
  bool same = true;
  for (int k = 0; k < kDeepHostWords; ++k) {
    const unsigned long long x = m[k];
    same = same && unsigned(x >> 32) == t0;
    word[k] = unsigned(x);
  }
  std::memcpy(static_cast<void *>(out), word, sizeof word);
  *tag = t0;
  return same;
}

}  // namespace

size_t deep_bytes(int k, int qcap_s) {
  return size_t(k) * (sizeof(DeepCtl) + 2 * sizeof(int) * kDeepStripes * size_t(qcap_s));
}

void deep_free(ent_graph *g, DeepWorkspace *w) {
  if (!w) return;
  const size_t qb = sizeof(int) * size_t(w->kcap) * kDeepStripes * size_t(w->qcap_s);
  dev_free(g, w->ctl, sizeof(DeepCtl) * size_t(w->kcap));
  dev_free(g, w->q[0], qb);
  dev_free(g, w->q[1], qb);
  if (w->h_mir) ignore(hipHostFree(w->h_mir));
  delete w;
}

DeepWorkspace *deep_alloc(ent_graph *g, int k, int qcap_s) {
  DeepWorkspace *w = new (std::nothrow) DeepWorkspace();
  if (!w) return nullptr;
  w->kcap = k;
  w->qcap_s = qcap_s;
  const size_t qb = sizeof(int) * size_t(k) * kDeepStripes * size_t(qcap_s);
  const size_t mb = sizeof(unsigned long long) * 2 * kDeepHostWords * size_t(k);
  void *dev = nullptr;
  if (dev_alloc(g, reinterpret_cast<void **>(&w->ctl), sizeof(DeepCtl) * size_t(k)) ||
      (qcap_s && (dev_alloc(g, reinterpret_cast<void **>(&w->q[0]), qb) ||
                  dev_alloc(g, reinterpret_cast<void **>(&w->q[1]), qb))) ||
      hipHostMalloc(reinterpret_cast<void **>(&w->h_mir), mb, hipHostMallocCoherent) != hipSuccess ||
      hipHostGetDevicePointer(&dev, w->h_mir, 0) != hipSuccess) {
    ignore(hipGetLastError());
    clear_error();
    deep_free(g, w);
    return nullptr;
  }
  w->h_mir_dev = static_cast<unsigned long long *>(dev);
  std::memset(w->h_mir, 0, mb);
  return w;
}

int deep_build_rows(ent_graph *g) {
  GraphStore &st = *g->store;
  const int want = st.max_deg <= 4 ? 1 : st.max_deg <= 8 ? 2 : 0;
  if (!want || g->n < kDeepBatchVertices) return ENT_OK;
  if (dev_alloc(g, reinterpret_cast<void **>(&st.rows), 16 * size_t(want) * size_t(g->n))) {
    clear_error();  // no room: the CSR form
    return ENT_OK;
  }
  const dim3 grid(unsigned(g->cus) * 8);
  int4 *out = reinterpret_cast<int4 *>(st.rows);
  if (want == 1) hipLaunchKernelGGL(k_deep_rows<1>, grid, dim3(256), 0, g->stream, g->off, g->adj, (long long)g->n, out);
  else hipLaunchKernelGGL(k_deep_rows<2>, grid, dim3(256), 0, g->stream, g->off, g->adj, (long long)g->n, out);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(g->stream));  // other handles read them on their own streams
  st.rows_width = want;
  return ENT_OK;
}

int deep_run(ent_graph *g, const DeepWorkspace *w, const DeepArgs &a, int k, int blocks, unsigned search,
             DeepState *fin) {
  const int width = a.rows ? g->store->rows_width : 0;
  const bool skip = k > kDeepLatencySources;
  const void *kernel = width == 0 ? reinterpret_cast<const void *>(&k_deep<0, false>)
                       : width == 1
                           ? skip ? reinterpret_cast<const void *>(&k_deep<1, true>)
                                  : reinterpret_cast<const void *>(&k_deep<1, false>)
                           : skip ? reinterpret_cast<const void *>(&k_deep<2, true>)
                                  : reinterpret_cast<const void *>(&k_deep<2, false>);
  std::vector<char> done(size_t(k), 0);
  int open = k;
  // Four launches are queued at a time; the next four follow once the last of
  // them has started, so at most four exit at once behind the end.
  constexpr int kQueued = 4;
  const long long max_launches = (long long)g->n / kDeepLevels + 16;
  for (long long i = 0; open; i += kQueued) {
    if (i > max_launches) return set_error(ENT_EINTERNAL, "search did not finish in %lld launches", i);
    for (int j = 0; j < kQueued; ++j) {
      DeepArgs args = a;
      long long li = i + j;
      void *p[] = {&args, &li};
      HIP_TRY(hipLaunchKernel(kernel, dim3(unsigned(blocks), unsigned(k)),
                              dim3(kDeepBS), p, 0, g->stream));
    }
    HIP_TRY(hipEventRecord(g->ev1, g->stream));
    const unsigned want = unsigned(i + kQueued) + search * kDeepTagMul;
    bool drained = false;
    for (int s = 0; s < k; ++s) {
      if (done[size_t(s)]) continue;
      for (unsigned long spins = 0;; ++spins) {
        DeepState st{};
        unsigned tag;
        bool hit = false;
        for (int sl = 0; sl < 2 && !hit; ++sl) {
          if (!read_deep(w, s, sl, &st, &tag) || unsigned(st.search) != search) continue;
          hit = st.done || tag == want;
        }
        if (hit) {
          if (st.done) {
            fin[s] = st;
            if (st.error) return ENT_OK;
            done[size_t(s)] = 1;
            --open;
          }
          break;
        }
        if (drained) return set_error(ENT_EINTERNAL, "search state of source %d not published", s);
        if ((spins & 255) == 255) {
          const hipError_t e = hipStreamQuery(g->stream);
          if (e == hipSuccess) drained = true;  // the mirror is complete: one more look
          else if (e != hipErrorNotReady) return set_error(ENT_EDEVICE, "search failed: %s", hipGetErrorString(e));
        }
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
        if (spins >= (1ul << 14)) std::this_thread::yield();
      }
    }
  }
  return ENT_OK;
}

int deep_batch(ent_graph *g, const DeepWorkspace *w, const int32_t *roots, int k, int *rows, DeepState *fin) {
  DeepArgs a{};
  a.off = g->off;
  a.adj = g->adj;
  a.depth = rows;
  a.dstride = g->n;
  a.q[0] = w->q[0];
  a.q[1] = w->q[1];
  a.qstride = (long long)kDeepStripes * w->qcap_s;
  a.ctl = w->ctl;
  a.hmir = w->h_mir_dev;
  a.rows = g->store->rows;
  // About 1,024 blocks over all sources (four per CU fit their LDS).
  const int blocks = std::max(8, std::min(2 * g->cus, 4 * g->cus / k));
  a.nstripe = std::min(blocks, kDeepStripes);
  a.qcap_s = w->qcap_s * kDeepStripes / a.nstripe;
  // One numbering with the single-source searches, which use the same mirror.
  if (++g->search_seq == 0) g->search_seq = 1;
  const unsigned search = g->search_seq;
  hipLaunchKernelGGL(k_deep_fill, dim3(unsigned(g->cus) * 8), dim3(256), 0, g->stream, rows,
                     (long long)k * (long long)g->n);
  hipLaunchKernelGGL(k_deep_seed, dim3(unsigned(k)), dim3(256), 0, g->stream, a, roots, int(search));
  HIP_TRY(hipGetLastError());
  return deep_run(g, w, a, k, blocks, search, fin);
}

int deep_queue_joint_bytes(ent_graph *g, const int *rows, const int *order_dev, int k, unsigned long long *host) {
  unsigned long long *d = static_cast<unsigned long long *>(g->aux);
  HIP_TRY(hipMemsetAsync(d, 0, sizeof *d, g->stream));
  const unsigned blocks = unsigned(std::min<int64_t>(g->cus * 8, (g->n + 255) / 256));
  const dim3 grid(blocks, unsigned((k + 63) / 64));
  auto kernel = k <= 16 ? &k_deep_joint<16> : k <= 32 ? &k_deep_joint<32> : &k_deep_joint<64>;
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, g->stream, g->off, rows, order_dev, int(g->n), k, d);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(host, d, sizeof *host, hipMemcpyDeviceToHost, g->stream));
  return ENT_OK;
}

}  // namespace ent
