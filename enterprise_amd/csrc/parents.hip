// Parent (BFS tree) output derived from a depth array, behind
// ent_bfs_parents[_device] (ent_bfs.h). The reference outputs depths only
// (bfs_gpu_opt.cuh:446); the tree it would have to pass is Graph500's:
// parent[root] = root, parent[v] a neighbour of v one level closer to the
// root, -1 for unreached vertices.
//
// One lane per vertex: it probes the first neighbours of its row four at a
// time (rows start with high-degree neighbours, which sit on the levels
// nearest the root most often) and stops at the first one with depth one
// less; rows not resolved within the probe go to the whole wavefront, one
// vertex at a time, with a ballot early exit. Every reached vertex other
// than the root has such a neighbour when the depths are a BFS from root;
// vertices that do not are counted in `bad` and get parent -2.
//
// Rows still open after kParentWave entries are listed, and a second kernel
// scans them in pieces of kParentPiece, every block at once: on R-MAT 20 the
// probes read 1 to 2 M of the 31 M entries, but a single hub's row, whose
// parent is one of the root's few neighbours, can take 47,000 of them, 64 at a
// time. Bound before by that one wavefront (259 us on R-MAT 20), now by the
// pass over the vertices (23.5 us, and 9 us for the two short kernels).
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstring>

#include "ent_bfs.h"
#include "ent_common.h"
#include "ent_device.h"
#include "ent_internal.h"

namespace ent {

constexpr int kParentProbe = 16;
constexpr int kParentWave = 1024;    // entries a wavefront scans before it lists the row
constexpr int kParentPiece = 1024;   // entries one block of the second kernel scans at a time
constexpr int kParentList = 1 << 16; // listed rows; past them the wavefront scans on

// In g->aux: what a call counts. Zero before every call (k_parents_fix leaves
// it so).
struct ParentCounts {
  unsigned bad, listed;
};

__global__ __launch_bounds__(256) void k_parents(const long long *off, const int *adj, const int *depth, int n,
                                                 int root, int *parent, ParentCounts *pc, int *list,
                                                 unsigned *first) {
  const int lane = lane_id();
  const long long nthreads = (long long)gridDim.x * blockDim.x;
  unsigned int nbad = 0;
  // Wave-uniform trip count: every lane of a wavefront runs the same number
  // of iterations (the ballot loop below needs all lanes).
  for (long long base = (long long)blockIdx.x * blockDim.x + threadIdx.x - lane; base < n; base += nthreads) {
    const long long v = base + lane;
    const bool valid = v < n;
    const int d = valid ? depth[v] : -1;
    int par = -1;
    long long s = 0, e = 0, p = 0;
    bool open = false;  // reached, not the root, parent not found yet
    if (valid && d > 0) {
      s = off[v];
      e = off[v + 1];
      open = true;
      const long long pe = min(e, s + kParentProbe);
      for (p = s; p < pe && open; p += 4) {
        int u[4], du[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = p + j < pe ? adj[p + j] : -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) du[j] = u[j] >= 0 ? depth[u[j]] : -2;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (open && du[j] == d - 1) {
            par = u[j];
            open = false;
          }
      }
      if (p > pe) p = pe;
    } else if (valid && d == 0) {
      par = int(v);
      open = v != root;  // depth 0 belongs to the root alone
    }
    unsigned long long lmask = __ballot(open && d > 0 && p < e);
    while (lmask) {
      const int src = __ffsll((long long)lmask) - 1;
      lmask &= lmask - 1;
      const long long pp = __shfl(p, src), ee = __shfl(e, src);
      const int dd = __shfl(d, src);
      int found = -1;
      long long limit = min(ee, pp + kParentWave);
      for (long long q0 = pp; q0 < limit && found < 0;) {
        int u[4];
        unsigned long long hm[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = q0 + j * kWave + lane < limit ? adj[q0 + j * kWave + lane] : -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) hm[j] = __ballot(u[j] >= 0 && depth[u[j]] == dd - 1);
#pragma unroll
        for (int j = 3; j >= 0; --j)
          if (hm[j]) found = __shfl(u[j], __ffsll((long long)hm[j]) - 1);
        q0 += 4 * kWave;
        if (q0 >= limit && found < 0 && limit < ee) {
          unsigned at = 0;
          if (lane == 0) at = atomicAdd(&pc->listed, 1u);
          at = unsigned(__builtin_amdgcn_readfirstlane(int(at)));
          if (at < unsigned(kParentList)) {
            const int vv = int(base) + src;
            if (lane == 0) {
              list[at] = vv;
              first[at] = ~0u;
            }
            found = vv;  // k_parents_fix writes the parent
          } else {
            limit = ee;
          }
        }
      }
      if (lane == src) {
        par = found;
        open = found < 0;
      }
    }
    if (valid) {
      if (open) {  // no neighbour one level up: the depths are not a BFS from root
        par = -2;
        ++nbad;
      }
      parent[v] = par;
    }
  }
  if (nbad) atomicAdd(&pc->bad, nbad);
}

// Listed rows from kParentProbe + kParentWave on: rows to blockIdx.y, pieces
// to blockIdx.x. first[i] becomes the smallest position in the row of a
// neighbour one level closer; pieces behind a known position are skipped.
__global__ __launch_bounds__(256) void k_parents_long(const long long *off, const int *adj, const int *depth,
                                                      const ParentCounts *pc, const int *list, unsigned *first) {
  const unsigned nl = min(pc->listed, unsigned(kParentList));
  for (unsigned i = blockIdx.y; i < nl; i += gridDim.y) {
    const int v = list[i];
    const long long s = off[v], len = off[v + 1] - s;
    const int want = depth[v] - 1;
    for (long long q0 = kParentProbe + kParentWave + (long long)blockIdx.x * kParentPiece; q0 < len;
         q0 += (long long)gridDim.x * kParentPiece) {
      if (ld_agent(&first[i]) < unsigned(q0)) break;
      int u[kParentPiece / 256];
#pragma unroll
      for (int j = 0; j < kParentPiece / 256; ++j) {
        const long long q = q0 + j * 256 + threadIdx.x;
        u[j] = q < len ? adj[s + q] : -1;
      }
#pragma unroll
      for (int j = 0; j < kParentPiece / 256; ++j) {
        const unsigned long long hm = __ballot(u[j] >= 0 && depth[u[j]] == want);
        if (hm && lane_id() == 0)
          atomicMin(&first[i], unsigned(q0) + unsigned(j * 256 + int(threadIdx.x)) + unsigned(__ffsll((long long)hm) - 1));
      }
    }
  }
}

// Parents of the listed rows, the count of vertices without one to the host
// (*host_bad, pinned) and the counters back to zero. One block.
__global__ __launch_bounds__(1024) void k_parents_fix(const long long *off, const int *adj, int *parent,
                                                      ParentCounts *pc, const int *list, const unsigned *first,
                                                      unsigned *host_bad) {
  __shared__ unsigned bad;
  if (threadIdx.x == 0) bad = pc->bad;
  const unsigned nl = min(pc->listed, unsigned(kParentList));
  __syncthreads();
  for (unsigned i = threadIdx.x; i < nl; i += 1024) {
    const int v = list[i];
    const unsigned f = first[i];
    parent[v] = f == ~0u ? -2 : adj[off[v] + f];
    if (f == ~0u) atomicAdd(&bad, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    *host_bad = bad;
    *pc = ParentCounts{0u, 0u};
  }
}

}  // namespace ent

using namespace ent;

extern "C" int ent_bfs_parents_device(ent_graph *g, int32_t root, const int32_t *depth_dev, int32_t *parent_dev) {
  clear_error();
  if (!g || !depth_dev || !parent_dev) return set_error(ENT_EINVAL, "NULL argument");
  if (root < 0 || root >= g->n) return set_error(ENT_EINVAL, "root %d outside [0, %lld)", root, (long long)g->n);
  std::lock_guard<std::mutex> lk(g->mu);
  HIP_TRY(hipSetDevice(g->device));
  static_assert(sizeof(ParentCounts) <= kParentCountBytes, "counters");
  ParentCounts *pc = reinterpret_cast<ParentCounts *>(static_cast<char *>(g->aux) + kAuxBytes);
  // The queues of the single-source search are idle between searches.
  int *list = g->qbuf[0];
  unsigned *first = reinterpret_cast<unsigned *>(g->qbuf[1]);
  unsigned *host_bad = g->h_bad;
  const int grid = int(std::min<int64_t>(int64_t(g->cus) * 8, (g->n + 255) / 256));
  hipLaunchKernelGGL(k_parents, dim3(std::max(grid, 1)), dim3(256), 0, g->stream, g->off, g->adj, depth_dev,
                     int(g->n), int(root), parent_dev, pc, list, first);
  // A graph without rows that long lists none.
  if (g->store->max_deg > kParentProbe + kParentWave)
    hipLaunchKernelGGL(k_parents_long, dim3(32, 32), dim3(256), 0, g->stream, g->off, g->adj, depth_dev, pc, list,
                       first);
  hipLaunchKernelGGL(k_parents_fix, dim3(1), dim3(1024), 0, g->stream, g->off, g->adj, parent_dev, pc, list, first,
                     g->h_bad_dev);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(g->stream));
  const unsigned h_bad = *host_bad;
  if (h_bad)
    return set_error(ENT_EINVAL, "%u reached vertices have no neighbour one level closer to root %d", h_bad, root);
  return ENT_OK;
}

extern "C" int ent_bfs_parents(ent_graph *g, int32_t root, int32_t *depth_host, int32_t *parent_host,
                               ent_stats *st) {
  int rc = ent_bfs_device(g, root, nullptr, st);
  if (rc) return rc;
  if (!g->parent) {
    std::lock_guard<std::mutex> lk(g->mu);
    if (!g->parent && (rc = dev_alloc(g, reinterpret_cast<void **>(&g->parent), sizeof(int) * size_t(g->n))))
      return rc;
  }
  if ((rc = ent_bfs_parents_device(g, root, g->depth, g->parent))) return rc;
  if (depth_host && (rc = ent_copy_to_host(g, g->depth, depth_host, g->n))) return rc;
  if (parent_host && (rc = ent_copy_to_host(g, g->parent, parent_host, g->n))) return rc;
  return ENT_OK;
}
