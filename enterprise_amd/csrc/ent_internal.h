// Host-side definition of the opaque graph handle, shared by the
// single-source (bfs_plain.hip) and batched (bfs_batch.hip) translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <algorithm>
#include <cstdint>
#include <memory>
#include <mutex>
#include <vector>

#include "ent_bfs.h"
#include "ent_common.h"

struct ent_graph;
namespace ent {
struct Args;
struct Control;
struct BatchWorkspace;
struct DeepWorkspace;
template <class T>
inline void ignore(T) {}

// Resident CSR shared by every handle made with ent_graph_share; freed with
// the last handle.
struct GraphStore {
  int device = 0;
  long long *off = nullptr;              // int64[n + 1]
  int *adj = nullptr;                    // int32[m]
  unsigned long long *nzmask = nullptr;  // bit v: degree(v) > 0
  std::vector<int32_t> h_deg;            // host copy of degrees (for the static lists)
  int32_t max_deg = 0;
  bool skewed = false;                   // largest degree far above the mean (kSkew)
  int *head = nullptr;                   // first neighbour of each row, or null (bfs_plain.hip)
  int *rows = nullptr;                   // padded rows, or null (ent_deep.h)
  int rows_width = 0;                    // their width in int4
  // A search (batch) of several levels per launch outgrew its queues: the graph
  // spreads too fast for that form, and later ones, on any handle, start in the
  // ordinary one.
  std::atomic<bool> deep_off{false}, deep_batch_off{false};
  ~GraphStore() {
    if (hipSetDevice(device) != hipSuccess) return;
    ignore(hipFree(off));
    ignore(hipFree(adj));
    ignore(hipFree(nzmask));
    ignore(hipFree(rows));
    ignore(hipFree(head));
  }
};
// Reorders every adjacency row by descending floor(log2(neighbour degree)),
// stably (adj_order.hip).
int order_rows_by_degree(ent_graph *g);
// ent_graph_upload_ex with the adjacency either in host memory or already in
// device memory of `device` (adj_on_device; copied device to device).
int upload_graph(const int64_t *beg_pos, const int32_t *adj, bool adj_on_device, int64_t n, int64_t m, int device,
                 int32_t flags, ent_graph **out);
}  // namespace ent

struct ent_graph {
  int device = 0;
  int64_t n = 0, m = 0, n_active = 0, nwords = 0;
  hipStream_t stream = nullptr;
  std::shared_ptr<ent::GraphStore> store;  // resident CSR (shared)
  long long *off = nullptr;                 // = store->off
  int *adj = nullptr;                       // = store->adj
  unsigned long long *nzmask = nullptr;     // = store->nzmask
  int *hub_block = nullptr;
  int *piece_v = nullptr;
  int *piece_k = nullptr;
  int n_hub_block = 0, n_pieces = 0;
  int lists_t_block = -1, lists_t_grid = -1, lists_piece = -1;
  int *hub_slot = nullptr;  // LDS hub table source (hub_slots entries)
  int *hub_tag = nullptr;   // level at which hub_slot[s] joined the frontier
  int hub_slots = 0;        // entries built (0: none)
  int hub_min = 0;          // smallest degree in the table
  int lists_hub = -1, lists_hub_tw = -1;
  int *depth = nullptr;
  void *aux = nullptr;     // kAuxBytes of device scratch for host-side calls (counters), then the parent counters
  unsigned *h_bad = nullptr, *h_bad_dev = nullptr;  // pinned: vertices ent_bfs_parents_device found no parent for
  unsigned long long *hashbuf = nullptr;  // kHashRows row checksums (ent_device_row_hash)
  int *parent = nullptr;   // parent array of ent_bfs_parents (allocated on first use)
  int trace_launches = 0;  // launches recorded by the last counting search
  void *stage[2] = {nullptr, nullptr};  // pinned staging for copies to pageable host memory
  hipEvent_t stage_ev[2] = {nullptr, nullptr};
  unsigned *narrow_flags = nullptr, *narrow_flags_dev = nullptr;  // pinned: copy_depths' flags, then its bytes
  unsigned char *narrow = nullptr, *narrow_dev = nullptr;
  unsigned narrow_seq = 0;  // tag of the latest k_narrow launch
  unsigned long long *visited = nullptr;
  unsigned long long *front[2] = {nullptr, nullptr};
  unsigned char *mark = nullptr;
  // Every mark is zero: the last search on the handle completed (a top-down
  // level marks only unvisited vertices, and the inspection that always
  // follows it clears every mark it finds). False until the first search.
  bool marks_clean = false;
  int *qbuf[2] = {nullptr, nullptr};  // striped frontier queues (kQStripes x qcap_s)
  int qcap_s = 0;
  ent::Control *ctl = nullptr;
  ent::Control *h_ctl = nullptr;           // pinned; the persistent form's state copy
  unsigned long long *h_mir = nullptr;     // host-coherent tagged state mirror, written by the kernels
  unsigned long long *h_mir_dev = nullptr; // the same memory as a device pointer
  unsigned search_seq = 0;                 // number of the latest search on this handle (never 0)
  ent_bfs_config cfg{};
  int cus = 0;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  unsigned char graph_args[512] = {};  // launch arguments baked into the captured graph
  const void *graph_fn = nullptr;           // and its kernel
  int graph_bs = 0, graph_grid = 0, graph_k = 0;
  size_t dev_bytes = 0;
  size_t dev_limit = 0;  // dev_alloc fails beyond it (tests; 0: none)
  int last_grid = 0;
  int expect_launches = 12;
  ent::DeepWorkspace *deep = nullptr;    // several levels per launch (ent_deep.h), or null
  ent::BatchWorkspace *batch = nullptr;  // lazily allocated multi-source workspace
  std::mutex mu;
};


#define HIP_TRY(expr)                                                                     \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return ent::set_error(ENT_EDEVICE, "%s failed: %s", #expr, hipGetErrorString(e_));  \
  } while (0)

namespace ent {

// Rows one ent_device_row_hash launch sums (its per-handle buffer's length).
constexpr int kHashRows = 512;
// Bytes of ent_graph::aux, and of the parent counters behind them.
constexpr size_t kAuxBytes = 256, kParentCountBytes = 16;

// Frees the idle construction context of `device` (csr_build.hip).
void build_give_back(int device);

// hipMalloc that gives the idle construction context back before it fails.
inline hipError_t device_malloc(int device, void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  ignore(hipGetLastError());
  build_give_back(device);
  return hipMalloc(p, bytes);
}

inline int dev_alloc(ent_graph *g, void **p, size_t bytes) {
  if (bytes == 0) bytes = 8;
  const bool over = g->dev_limit && g->dev_bytes + bytes > g->dev_limit;
  hipError_t e = over ? hipErrorOutOfMemory : device_malloc(g->device, p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    ignore(hipGetLastError());
    return set_error(ENT_ENOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
  }
  g->dev_bytes += bytes;
  return ENT_OK;
}

inline void dev_free(ent_graph *g, void *p, size_t bytes) {
  if (!p) return;
  ignore(hipFree(p));
  g->dev_bytes -= std::min(g->dev_bytes, bytes);
}

// Frees the batched workspace (defined in bfs_batch.hip).
void batch_release(ent_graph *g);

// Device-to-host copy on g's stream, returning when it is complete (pinned
// or small destinations in one DMA, pageable ones through pinned staging).
// The caller holds g->mu.
int copy_to_host(ent_graph *g, void *dst, const void *src, size_t bytes);


}  // namespace ent
