// Levels of narrow frontiers inside one launch: a cluster of workgroups runs
// a traversal level after level, with a barrier between levels where the wide
// pipeline has kernel launches and a host round trip.
//
// What bounds a narrow level is latency.  A lattice of 10^6 vertices has about
// 1750 levels of 570 vertices; the wide pipeline spends 15 us on each (BFS,
// two launches) or 28 us (bucketed SSSP, four), for two to four thousand
// edges.  Here a level is the chain LDS queue -> destination -> atomic min on
// its value, with the row bounds of the next entry loaded beside it -> LDS
// queue, and a barrier: 3.4 us (BFS 1000^2) and 5.3 us (SSSP 1500^2, 1000
// vertices and 3600 edges per level), 26.4 -> 6.0 ms and 109 -> 19.9 ms per
// query.  What was tried on the way, same cases: one queue in global memory
// with a shared tail, 9.3 / 25.8 ms; a global segment per wavefront with its
// own report, 8.1 / 28 ms; the same with DPP scans instead of shuffles, 7.4 /
// 23.0 ms; all workgroups on one XCD, 0-20 % slower than spread over the
// eight in each of these; LDS queues with 8 / 16 / 32 workgroups of 256
// threads, 8.4 / 6.8 / 6.5 and 36 / 28 / 22 ms; 16 of 512, 6.2 / 21.4 ms; 8 /
// 16 / 32 of 1024, 6.0 / 6.0 / 6.4 and 20.3 / 19.9 / 21.8 ms (kept: 16).
//
// Queues.  A workgroup queues what it discovers in its own LDS (the entries
// past kClusterLds in global memory) and expands it in the next level, so
// entries cross workgroups only when a queue is long and twice the average:
// then all are dealt out evenly (2-30 times in the runs above).  An entry is
// a piece of a row of at most kClusterChunk edges, so a hub spreads over
// wavefronts; a wavefront spreads the edges of a few consecutive entries over
// its lanes.  A vertex improved several times in a level (SSSP, CC) has
// several entries, each with its value, and only the one whose value still
// stands when the level starts is expanded.
//
// Barrier.  Each workgroup adds one 64-bit word to the level's report --
// arrived, vertices, edges, wants to leave, has a long queue -- and polls the
// report until all have: one line, one atomic per workgroup, and the level's
// totals come with it.  Data that crosses workgroups goes through agent-scope
// atomics only (values, bitmaps, segments, counters), and every wavefront
// waits for its own (s_waitcnt) before its workgroup reports: a release at
// agent scope would write the L2 back at every level.
//
// Handing over.  The bitmaps hold the frontier at every level, so the cluster
// can take a frontier over from the wide pipeline and hand one back: when it
// has more than max_edges out-edges, a queue or a list runs out of room, or
// (hub deferral) a vertex should wait.  Vertices without edges are counted,
// not queued; their bits may stay set, which no later step minds.
//
// Bucketed runs (delta != 0): a vertex whose value is at or above the
// threshold goes to a far list with that value; when nothing is queued the
// threshold moves to the lists' smallest value + delta and each workgroup
// splits its own list: entries whose vertex has improved since are dropped
// (the improvement was queued), those below the new threshold are queued.  In
// a batch, where no frontier is handed back, a waiting vertex that a full list
// has no room for goes to a third bitmap, which a split walks too: taken into
// the frontier instead, it is expanded long before its bucket and so are all
// that follow (four queries in buckets of 3000 on a 3-D lattice of 160^3 vertices
// 292-353 ms, 620 of 1100 levels walking the bitmap, 39 ms now; 32 queries
// 448-509 and 73 ms).
//
// The workgroups need not all be resident: they register, the first one
// closes the registration once all have come or after 20 us, and barriers
// wait for registered (hence running) workgroups only; one that comes later
// leaves at once.
#pragma once

#include "kernels.hpp"

namespace cg {

constexpr int kClusterBlock = 1024;
constexpr int kClusterWaves = kClusterBlock / kWave;
constexpr uint32_t kClusterMaxGroups = 16;
constexpr uint32_t kClusterChunk = 64;          // edges per queue entry
constexpr uint32_t kClusterLds = 1024;          // queue entries a workgroup holds in LDS
constexpr uint32_t kClusterSegment = 1u << 13;  // and altogether
constexpr uint32_t kClusterFar = 1u << 13;      // far entries per workgroup
constexpr uint32_t kClusterNone = 0xFFFFFFFFu;
// A frontier of more out-edges than this is the wide pipeline's: 2^16 edges
// are four rounds of the cluster's lanes, about what an iteration of the wide
// pipeline costs in launches alone.
constexpr uint64_t kClusterEdges = 1u << 16;
// From this many edges on an update reads the value before it tries the
// atomic: smaller levels are bound by the chain, where the read would be one
// more access, larger ones by contended atomics.
constexpr uint32_t kClusterCheck = 8192;

// A queue entry: a vertex, the value it was queued with, and a piece of its
// row -- start (40 bits) | whether it is the row's first piece (bit 40) |
// length (from bit 48).
struct alignas(16) ClusterEntry {
  unsigned long long vertex;  // vertex | value << 32
  unsigned long long row;
};
struct alignas(128) ClusterFarState {
  uint32_t count, min_val;
  uint32_t over;  // batches: some of them are in the bitmap ClusterJob::wait
};
struct ClusterCtl {
  alignas(128) uint32_t join;
  alignas(128) uint32_t members;
  alignas(128) unsigned long long query;     // batches: turn << 32 | query
  alignas(128) uint32_t bar;                 // barriers of a redistribution
  alignas(128) unsigned long long level[3][16];  // level L's report: word [L % 3][0], one per line
  ClusterFarState far[3];                     // far lists, rotating at each split
  alignas(128) unsigned long long edges_done;
  unsigned long long verts_done;
  alignas(128) uint32_t seg[2][kClusterMaxGroups];  // queue lengths for a redistribution, by level parity
};

// What a cluster run did, published to mapped host memory (tag last).
struct ClusterRecord {
  uint32_t levels;           // iterations
  uint32_t n;                // vertices of the frontier handed back (0: the traversal is complete)
  uint32_t threshold;        // bucketed runs
  uint32_t tag;
  unsigned long long edges, verts;  // out-edges and vertices of the expanded frontiers
};

struct ClusterJob {
  const uint64_t* off;
  const uint32_t* dst;
  const void* w;        // weights of the width the kernel was instantiated for (SSSP)
  uint32_t* val;
  uint64_t* bm[2];      // frontier of iteration k in bm[(k - 1) & 1]
  uint64_t words;
  ClusterEntry* q[2];
  uint32_t cap;         // entries per workgroup
  unsigned long long* far[2];  // bucketed runs: kClusterFar entries per workgroup
  uint32_t k0;          // iteration of the frontier taken over
  uint64_t max_edges;
  uint32_t hub_degree;  // a frontier vertex of at least this degree also asks for the wide pipeline (0: off)
  uint32_t delta, threshold;
  uint32_t root;            // batches: the query's root, and the largest level count so far
  uint32_t* batch_levels;
  uint64_t* wait;           // batches, bucketed: waiting vertices beyond the far lists' room
  // wide pipeline's state, written when a frontier is handed back
  RunState* rs;
  DevStats* st;
  unsigned long long* bfs_cnt;  // BFS: first-visit counters, two parities
  ClusterCtl* ctl;              // this launch's, zeroed
  ClusterCtl* ctl_next;         // the next launch's, zeroed by this one
  ClusterRecord* host_out;
  uint32_t tag;
};

// Entries any frontier of the graph needs at most.
inline uint64_t cluster_entry_bound(uint64_t V, uint64_t E) { return V + E / kClusterChunk + 1; }

// Workgroups of an engine's cluster: a graph with fewer edges than that many
// lanes needs fewer (R-MAT s12, 28 677 edges: 4 / 8 / 16 of them 111 / 104 / 99 us).
inline uint32_t cluster_groups(uint64_t E) {
  const uint64_t g = E / 1024;
  return (uint32_t)(g < 1 ? 1 : (g > kClusterMaxGroups ? kClusterMaxGroups : g));
}

// A batched query for a cluster: every value unreached, bitmaps zero (2 * words,
// with delta 3 * words).
struct ClusterQuery {
  const uint64_t* off;
  const uint32_t* dst;
  const uint32_t* w;
  uint32_t* val;
  uint64_t* bm;
  uint64_t words;
  int alg;
  uint32_t root, delta;
};
struct ClusterBatch {
  const ClusterQuery* q;
  uint32_t nq;
  uint32_t* next;     // 0: the first query not yet taken
  uint32_t* levels;   // 0: the largest level count of a query
  ClusterCtl* ctl;    // one per cluster, zeroed
  ClusterEntry* entries;     // 2 * groups * cap per cluster
  unsigned long long* far;   // 2 * groups * kClusterFar per cluster
  uint32_t groups, cap;
};
int launch_cluster_batch(const ClusterBatch& b, uint32_t clusters, hipStream_t s);

// Largest out-degree of a graph whose frontiers are taken to be narrow from
// any root (lattices, roads).
constexpr uint64_t kClusterRootDegree = 64;

// One cluster of `groups` workgroups runs job (cluster.hip).  w_bytes: the
// width of job.w for SSSP.
int launch_cluster(int alg, int w_bytes, const ClusterJob& job, uint32_t groups, hipStream_t s);

}  // namespace cg
