// One block per search for small graphs, shared by the single-source
// (bfs_plain.hip) and the batched (bfs_batch.hip) form.
#pragma once

#include <hip/hip_runtime.h>

#include "ent_device.h"
#include "ent_internal.h"

namespace ent {

// Whole search of a small graph in one block: visited bits and frontier
// queues in LDS, the frontier's edges spread over all threads.
//
// A launch per level costs about 8 us of launch, prologue and dependent round
// trips whatever the graph's size, and a hub's row goes to one wavefront. Here
// eight lanes take two frontier vertices' rows at a time, the whole block a row
// of kTinyHub edges or more, and a neighbour is claimed with an atomic OR
// in LDS and queued there: two round trips to L2 and a few block barriers a
// level. Bound: one CU's instruction issue, about 2 edges a nanosecond, so the
// rule stops at kTinyEdges. Against a launch per level: R-MAT 1,024 vertices 91
// -> 34.5 us, 2,000 with 60,000 edges 75 -> 40, 10,000 with 93,000 edges 79 ->
// 70 (and with 220,000 edges 59 -> 124, hence the rule), uniform 2,000 90 ->
// 28, a 30 x 40 grid 183 -> 55. More rows in flight per group, sixteen lanes
// a row, and a queue rebuilt from the new bits were all slower.
constexpr int kTinyThreads = 1024;
constexpr int kTinyVertices = 1 << 14;  // 16-bit queue entries, 64 KiB for both queues
constexpr int kTinyLanes = 8;
constexpr int kTinyRows = 2;            // rows a group of lanes has in flight
constexpr unsigned kTinyHub = 256;
constexpr int64_t kTinyEdges = 3 << 15;
constexpr int kTinyHubs = kTinyEdges / kTinyHub;  // there are no more rows of that length
struct TinySmem {
  unsigned vis[kTinyVertices / 32];
  unsigned short q[2][kTinyVertices];
  unsigned hub_s[kTinyHubs], hub_d[kTinyHubs];
  unsigned qn[2], nhub[2];
  unsigned long long mf;
};

// What a search found. The total degree is in sm.mf behind the last barrier.
struct TinyResult {
  int levels;
  unsigned reached;
};

__device__ __forceinline__ TinyResult tiny_search(TinySmem &sm, const long long *off, const int *adj, int *depth, int n,
                                                  int root) {
  const int t = threadIdx.x, lane = lane_id();
  for (int k = t; k < kTinyVertices / 32; k += kTinyThreads) sm.vis[k] = k == (root >> 5) ? 1u << (root & 31) : 0u;
  for (int v = t; v < n; v += kTinyThreads) depth[v] = v == root ? 0 : -1;
  if (t == 0) {
    sm.q[0][0] = (unsigned short)root;
    sm.qn[0] = 1;
    sm.nhub[0] = sm.nhub[1] = 0;
    sm.mf = 0;
  }
  __syncthreads();
  unsigned long long mf = 0;
  unsigned total_nf = 0;
  int L = 0;
  for (;; ++L) {
    const unsigned short *qin = sm.q[L & 1];
    unsigned short *qout = sm.q[(L + 1) & 1];
    unsigned *qcnt = &sm.qn[(L + 1) & 1], *nhub = &sm.nhub[L & 1];
    const unsigned cnt = sm.qn[L & 1];
    total_nf += cnt;
    if (cnt == 0) break;  // the whole block
    if (t == 0) {
      *qcnt = 0;
      sm.nhub[(L + 1) & 1] = 0;
    }
    __syncthreads();
    // Claims u and queues it if it was unvisited (-1: no neighbour).
    auto claim = [&](int u) {
      if (u < 0) return;
      const unsigned bit = 1u << (u & 31);
      // A plain look first: most edges lead back.
      if ((sm.vis[u >> 5] & bit) || (atomicOr(&sm.vis[u >> 5], bit) & bit)) return;
      qout[atomicAdd(qcnt, 1u)] = (unsigned short)u;
      depth[u] = L + 1;
    };
    // Neighbours i, i + stride, i + 2 stride, i + 3 stride of the row [s, s + d).
    auto visit = [&](unsigned s, unsigned d, unsigned i, unsigned stride) {
      int u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = i + j * stride < d ? adj[s + i + j * stride] : -1;
#pragma unroll
      for (int j = 0; j < 4; ++j) claim(u[j]);
    };
    constexpr unsigned kGroups = kTinyThreads / kTinyLanes;
    const unsigned gl = unsigned(t) % kTinyLanes;
    for (unsigned k0 = unsigned(t) / kTinyLanes; k0 < cnt; k0 += kTinyRows * kGroups) {
      unsigned s[kTinyRows], d[kTinyRows];
#pragma unroll
      for (int x = 0; x < kTinyRows; ++x) {
        const unsigned k = k0 + x * kGroups;
        s[x] = d[x] = 0;
        if (k < cnt) {
          const int v = qin[k];
          const long long b = off[v];
          s[x] = unsigned(b);
          d[x] = unsigned(off[v + 1] - b);
        }
      }
      int u[kTinyRows][2];
#pragma unroll
      for (int x = 0; x < kTinyRows; ++x) {
        if (gl == 0) mf += d[x];
        if (d[x] >= kTinyHub) {
          if (gl == 0) {
            const unsigned h = atomicAdd(nhub, 1u);
            sm.hub_s[h] = s[x];
            sm.hub_d[h] = d[x];
          }
          d[x] = 0;
        }
        u[x][0] = gl < d[x] ? adj[s[x] + gl] : -1;
        u[x][1] = gl + kTinyLanes < d[x] ? adj[s[x] + gl + kTinyLanes] : -1;
      }
#pragma unroll
      for (int x = 0; x < kTinyRows; ++x) {
        claim(u[x][0]);
        claim(u[x][1]);
      }
#pragma unroll
      for (int x = 0; x < kTinyRows; ++x)
        for (unsigned i = gl + 2 * kTinyLanes; i < d[x]; i += 4 * kTinyLanes) visit(s[x], d[x], i, kTinyLanes);
    }
    __syncthreads();
    const unsigned nh = *nhub;
    for (unsigned h = 0; h < nh; ++h) {
      const unsigned s = sm.hub_s[h], d = sm.hub_d[h];
      for (unsigned i = t; i < d; i += 4 * kTinyThreads) visit(s, d, i, kTinyThreads);
    }
    __syncthreads();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mf += __shfl_xor(mf, o);
  if (lane == 0) atomicAdd(&sm.mf, mf);
  __syncthreads();
  return TinyResult{L, total_nf};
}

inline bool tiny_graph(const ent_graph *g) { return g->n <= kTinyVertices && g->m <= kTinyEdges; }

// Whether searches on g run in one block each: at most kTinyVertices vertices
// and kTinyEdges edges, and a configuration that neither asks for bottom-up
// levels, for the reference's switch, for a launch form that keeps levels
// apart, for a tally nor for no queues.
inline bool tiny_fits(const ent_graph *g) {
  const ent_bfs_config &c = g->cfg;
  return tiny_graph(g) && !c.count_examined && g->hub_slots == 0 && c.queue_small >= 0 &&
         (c.direction == ENT_DIR_AUTO || c.direction == ENT_DIR_TOPDOWN) &&
         (c.launch == ENT_LAUNCH_STREAM || c.launch == ENT_LAUNCH_GRAPH);
}

}  // namespace ent
