// Queue-driven searches that run several levels per launch (bfs_deep.hip):
// the tail of a single-source search (bfs_plain.hip) and batches of few
// sources (bfs_batch.hip) on graphs of low degree and high diameter.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "ent_internal.h"

namespace ent {

constexpr int kDeepMaxDegree = 16;  // largest degree of a graph searched this way
constexpr int64_t kDeepBatchVertices = 1 << 12;  // smallest graph whose batches are
constexpr int kDeepLevels = 24;     // levels per launch
constexpr int kDeepQueue = 512;     // queue entries per stripe and source of a batch
constexpr int kDeepStripes = 64;    // counter and queue stripes
constexpr int kDeepStripeU32 = 32;  // 128 B between stripes

enum : int { DEEP_OVERFLOW = 1, DEEP_NOT_TAKEN = 2 };

// Search state before a launch; launch i reads st[(i + 1) & 1] and the counts
// of launch i - 1 and publishes its own in st[i & 1].
struct DeepState {
  int level;     // depth of the vertices in the queue
  int par;       // queue that holds them
  int done;
  int error;
  int launches;  // launches run so far
  int search;
  int levels;
  int td_levels;
  unsigned long long total_nf, total_mf;
  unsigned long long t_end;
  unsigned qn[kDeepStripes];
};
constexpr int kDeepHostWords = int(offsetof(DeepState, qn) / 4);

// Counter words of a stripe: degree sum (64 bits), queue entries, overflow
// flags, then the vertices of level L + 1 + j at DK_NF + j.
enum : int { DK_MF = 0, DK_QN = 2, DK_FLAGS = 3, DK_NF = 4 };
static_assert(DK_NF + kDeepLevels <= kDeepStripeU32 && kDeepLevels % 4 == 0, "one stripe line, read as int4");

struct DeepCtl {
  DeepState st[2];
  unsigned cnt[3][kDeepStripes * kDeepStripeU32];
};

struct DeepArgs {
  const long long *off;
  const int *adj;
  const int *rows;    // padded rows (deep_build_rows), or null
  int *depth;         // source s: depth + s * dstride
  long long dstride;
  int *q[2];          // source s: q[p] + s * qstride, stripe t at + t * qcap_s
  long long qstride;
  DeepCtl *ctl;       // one per source
  unsigned long long *hmir;  // two tagged slots of kDeepHostWords per source
  int qcap_s;
  int nstripe;        // stripes in use: min(blocks per source, kDeepStripes)
};

// Tables for up to kcap sources. A handle has one for its single-source
// searches (no queues: those of the search), its batch workspace one for its
// batches; both are made with the workspace they belong to, so that a search
// allocates nothing. Where there is no room for one, that handle's searches
// (batches) stay in the ordinary form.
struct DeepWorkspace {
  int kcap = 0, qcap_s = 0;
  DeepCtl *ctl = nullptr;
  int *q[2] = {nullptr, nullptr};
  unsigned long long *h_mir = nullptr, *h_mir_dev = nullptr;
};

// Builds the store's padded rows, for every handle on the graph: vertex v's
// neighbours at rows[4 * rows_width * v], -1 behind the last. None for degrees
// above 8, for small graphs, and where there is no room.
int deep_build_rows(ent_graph *g);

// Tables for k sources with queues of qcap_s entries per stripe (0: none), or
// null where there is no room.
DeepWorkspace *deep_alloc(ent_graph *g, int k, int qcap_s);
void deep_free(ent_graph *g, DeepWorkspace *w);
size_t deep_bytes(int k, int qcap_s);

// Runs launches of `blocks` blocks per source until every one of the k
// searches whose states are in w->ctl[s].st[1] is done, or one of them has
// failed (the caller then runs all of them the ordinary way, behind what is
// queued); their final states go to fin[0 .. k). The host spins on the mirror, as
// for the other forms.
int deep_run(ent_graph *g, const DeepWorkspace *w, const DeepArgs &a, int k, int blocks, unsigned search,
             DeepState *fin);

// Batch of k sources from their roots (device memory) into rows of n
// entries.
int deep_batch(ent_graph *g, const DeepWorkspace *w, const int32_t *roots, int k, int *rows, DeepState *fin);

// Queues the algorithmic bytes of the joint frontiers, 8 + 12 deg(v) for each
// distinct (vertex, depth) pair of each 64-source group (rows order[64 g] on),
// and their copy to *host (pinned).
int deep_queue_joint_bytes(ent_graph *g, const int *rows, const int *order_dev, int k, unsigned long long *host);

}  // namespace ent
