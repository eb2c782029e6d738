// WCC (weakly connected components) by min-label hooking on a symmetric graph.
//
// The reference computes CC by pushing labels: value[i] = i, then every
// active vertex lowers its neighbours' labels with write_min / atomicMin
// (my_project/CGgraph/host_algorithm.hpp:412-433, device_algorithm.cuh:430-465).
// On a symmetric graph the fixed point is the minimum vertex id of each
// connected component.  This file reaches the same labels by hooking:
//   parent[v] = v; for every edge (u, v) link the two trees by pointing the
//   larger root at the smaller one (CAS); finally compress every path.
// parent[x] <= x holds throughout, so each tree's root is its minimum id and
// the final labels equal the label-propagation fixed point bit for bit.
// The edge order follows Afforest (Sutton, Ben-Nun, Bar, IPDPS'18): link the
// first neighbours of every vertex, compress, find the most frequent root by
// sampling, then let only vertices outside that component link their
// remaining edges -- an edge between the large component and another vertex
// is seen from the other side, because the graph is symmetric.
//
// The first neighbour needs no linking: rows are ascending, so parent[v] =
// min(v, first neighbour) is already a forest of edges of the graph (round 0,
// fused with the initialisation: no atomics, no reads of other parents).  On
// skewed graphs that alone leaves almost every vertex in one tree, and the
// second sampled neighbour -- another line of nearly every row -- is skipped;
// a lattice, where it leaves many, takes it.  The line: at most 1/8 of the
// sampled vertices outside the most frequent tree with an edge left to look
// at, found on the device, so the kernels of the second round are always
// queued and return at once.  R-MAT s24, 16.8 M vertices, 521 M edges:
// 0.66 ms of kernels with two linked rounds, 0.39 ms now (0.68 -> 0.42 ms per
// query with the waits): the first round 275 -> 136 us, the second 183 -> 4 us,
// compression and the remaining edges 160 -> 223 us, for more of them.
#include <algorithm>

#include "kernels.hpp"

namespace cg {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ uint32_t ld_relaxed(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Link the trees of u and v (Afforest's Link): climb towards the roots; when
// the larger candidate is a root, CAS it onto the smaller one.
__device__ void link(uint32_t u, uint32_t v, uint32_t* __restrict__ parent) {
  uint32_t p1 = ld_relaxed(parent + u);
  uint32_t p2 = ld_relaxed(parent + v);
  while (p1 != p2) {
    const uint32_t high = p1 > p2 ? p1 : p2;
    const uint32_t low = p1 + p2 - high;
    const uint32_t p_high = ld_relaxed(parent + high);
    if (p_high == low) break;
    if (p_high == high) {
      uint32_t expected = high;
      if (__hip_atomic_compare_exchange_strong(parent + high, &expected, low, __ATOMIC_RELAXED,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        break;
    }
    p1 = ld_relaxed(parent + ld_relaxed(parent + high));
    p2 = ld_relaxed(parent + low);
  }
}

// Climbs from the lane's N vertices base + k * stride (those below V), given
// their parents p and grandparents gp, to their roots p; every step is stored,
// so the climbs of a long chain's vertices shorten each other.  The N climb
// together: one after the other, those that wait leave their part of the chain
// one step long for every climb above it (paths of 0.1 / 1 / 4 M vertices 331 /
// 420 / 910 us per query, together 68 / 100 / 240; lattices of 300^2 / 1000^2 /
// 2048^2 101 / 203 / 550, together 90 / 168 / 465).
template <int N>
__device__ __forceinline__ void climb(uint64_t base, uint32_t stride, uint32_t V, uint32_t (&p)[N], uint32_t (&gp)[N],
                                      uint32_t* __restrict__ parent) {
  bool more = true;
  while (more) {
    more = false;
    bool moved[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      moved[k] = p[k] != gp[k] && base + k * stride < V;
      if (moved[k]) {
        __hip_atomic_store(parent + base + k * stride, gp[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        p[k] = gp[k];
        more = true;
      }
    }
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (moved[k]) gp[k] = ld_relaxed(parent + p[k]);
  }
}

// Round 0: parent[v] = min(v, first neighbour).  Bound by one line per row
// (off is streamed); kIlp rows per lane keep that many in flight.
constexpr int kIlp = 4;
// and where chains are climbed (lattices of 100^2 / 300^2 / 1000^2 / 2048^2, us per
// query with 4: 69 / 94 / 168 / 453, 2: 64 / 90 / 168 / 465, 1: 62 / 90 / 175 / 518)
constexpr int kChainIlp = 2;

__global__ __launch_bounds__(kBlock) void k_first(DevGraph g, uint32_t* __restrict__ parent) {
  const uint64_t base = blockIdx.x * (uint64_t)(kBlock * kIlp) + threadIdx.x;
  uint64_t s[kIlp], e[kIlp];
  uint32_t d[kIlp];
#pragma unroll
  for (int k = 0; k < kIlp; ++k) {
    const uint64_t v = base + k * kBlock;
    s[k] = v < g.V ? g.off[v] : 0;
    e[k] = v < g.V ? g.off[v + 1] : 0;
  }
#pragma unroll
  for (int k = 0; k < kIlp; ++k) d[k] = s[k] < e[k] ? g.dst[s[k]] : 0xFFFFFFFFu;
#pragma unroll
  for (int k = 0; k < kIlp; ++k) {
    const uint64_t v = base + k * kBlock;
    if (v < g.V) parent[v] = d[k] < (uint32_t)v ? d[k] : (uint32_t)v;
  }
}

// What the sampling found: the most frequent root, and how many neighbours of
// every vertex are linked before the rest (1 or 2).
struct WccPlan {
  uint32_t mode, rounds;
};

__global__ __launch_bounds__(kBlock) void k_link_round(DevGraph g, uint32_t r, const WccPlan* __restrict__ plan,
                                                       uint32_t* __restrict__ parent) {
  if (r >= plan->rounds) return;
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < g.V;
       v += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t s = g.off[v], e = g.off[v + 1];
    if (s + r < e) link((uint32_t)v, g.dst[s + r], parent);
  }
}

// plan: only if that many rounds were linked (NULL: always).
template <int ILP>
__global__ __launch_bounds__(kBlock) void k_compress(uint32_t V, uint32_t* __restrict__ parent,
                                                     const WccPlan* __restrict__ plan, uint32_t rounds) {
  if (plan && plan->rounds != rounds) return;
  for (uint64_t base = blockIdx.x * (uint64_t)(kBlock * ILP) + threadIdx.x; base < V;
       base += (uint64_t)gridDim.x * (kBlock * ILP)) {
    uint32_t p[ILP], gp[ILP];
#pragma unroll
    for (int k = 0; k < ILP; ++k) p[k] = base + k * kBlock < V ? ld_relaxed(parent + base + k * kBlock) : 0u;
#pragma unroll
    for (int k = 0; k < ILP; ++k) gp[k] = ld_relaxed(parent + p[k]);
    climb<ILP>(base, kBlock, V, p, gp, parent);
  }
}

// The most frequent root among kSamples random vertices (ties to the smaller
// id) and the number of rounds to link, on the device so the host never
// waits: one workgroup, each thread counting its sample's occurrences in LDS.
// Any choice gives the same labels; a good one lets most vertices skip their
// remaining edges.  rounds: what is linked when it is called; a second call
// (rounds 2) only looks again if the first asked for that round.  Round 0's
// trees are climbed here, at most kClimb steps (longer chains, as in a
// lattice, count as outside and so ask for the second round).
constexpr int kClimb = 24;
constexpr uint32_t kSamples = 512;

__global__ __launch_bounds__(kSamples) void k_sample(DevGraph g, const uint32_t* __restrict__ parent, uint64_t seed,
                                                     uint32_t rounds, WccPlan* __restrict__ plan) {
  if (rounds == 2 && plan->rounds != 2) return;
  __shared__ uint4 x4[kSamples / 4];
  __shared__ unsigned long long best[kSamples / 64];
  __shared__ uint32_t outside;
  uint32_t* const x = reinterpret_cast<uint32_t*>(x4);
  const uint32_t t = threadIdx.x;
  uint64_t z = seed + (uint64_t)(t + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  const uint32_t v = (uint32_t)(z % g.V);
  const uint64_t deg = g.off[v + 1] - g.off[v];
  uint32_t mine = parent[v];
  bool root = false;
  for (int i = 0; i < kClimb && !root; ++i) {
    const uint32_t p = parent[mine];
    root = p == mine;
    mine = p;
  }
  x[t] = mine;
  if (t == 0) outside = 0;
  __syncthreads();
  uint32_t c = 0;
  for (uint32_t j = 0; j < kSamples / 4; ++j) {
    const uint4 y = x4[j];
    c += (y.x == mine) + (y.y == mine) + (y.z == mine) + (y.w == mine);
  }
  // key: larger count first, then smaller id
  unsigned long long key = ((unsigned long long)c << 32) | (0xFFFFFFFFu - mine);
  for (int d = 32; d >= 1; d >>= 1) {
    const unsigned long long o = __shfl_xor(key, d, 64);
    key = o > key ? o : key;
  }
  if (__lane_id() == 0) best[t / 64] = key;
  __syncthreads();
  key = best[0];
  for (uint32_t w = 1; w < kSamples / 64; ++w) key = best[w] > key ? best[w] : key;
  const uint32_t mode = 0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFu);
  const uint64_t out = __ballot((mine != mode || !root) && deg > rounds);
  if (__lane_id() == 0) atomicAdd(&outside, (uint32_t)__popcll(out));
  __syncthreads();
  if (t == 0) {
    plan->mode = mode;
    plan->rounds = rounds == 2 || outside > kSamples / 8 ? 2 : 1;
  }
}

// Remaining edges of vertices outside the large component.  A wavefront
// climbs from 256 consecutive vertices, four per lane (compressing as it
// goes), tests them 64 at a time (root outside the large component, edges
// left), and each lane links the first kOwnEdges of its
// own row; what is left of longer rows is linked one row at a time with the
// row spread over the 64 lanes.  Most vertices are in the large component or
// have no edges, so the test is the bulk of the work and runs 64 wide; most of
// the others are leaves below their only neighbour, which a row per wavefront
// step would take one by one (R-MAT s24 after round 0 alone: 300 us with that,
// 140 us with the lanes' own edges first, both behind a compression of 91 us;
// 194 us with the compression in it).
constexpr int kOwnEdges = 4;

__global__ __launch_bounds__(kBlock) void k_link_rest(DevGraph g, const WccPlan* __restrict__ plan,
                                                      uint32_t* __restrict__ parent) {
  const uint32_t skip = plan->mode, r = plan->rounds;
  const uint32_t lane = __lane_id();
  const uint64_t base = (blockIdx.x * (uint64_t)(kBlock / 64) + threadIdx.x / 64) * (64 * kIlp) + lane;
  uint32_t p[kIlp], gp[kIlp];
#pragma unroll
  for (int k = 0; k < kIlp; ++k) p[k] = base + k * 64 < g.V ? ld_relaxed(parent + base + k * 64) : skip;
#pragma unroll
  for (int k = 0; k < kIlp; ++k) gp[k] = ld_relaxed(parent + p[k]);
  climb<kIlp>(base, 64, g.V, p, gp, parent);
#pragma unroll 1
  for (int k = 0; k < kIlp; ++k) {
    const uint64_t v = base + k * 64;
    uint64_t s = 0, e = 0;
    // the degree array spares the offsets of isolated vertices; a vertex below
    // its first neighbour was not linked to it by round 0
    if (v < g.V && p[k] != skip && g.deg[v] != 0) {
      s = g.off[v];
      e = g.off[v + 1];
      if (g.dst[s] < (uint32_t)v) s += r;
    }
#pragma unroll 1
    for (int i = 0; i < kOwnEdges; ++i)
      if (s < e) link((uint32_t)v, g.dst[s++], parent);
    for (uint64_t need = __ballot(s < e); need; need &= need - 1) {
      const int l = __builtin_ctzll(need);
      const uint64_t rs = __shfl(s, l, 64), re = __shfl(e, l, 64);
      for (uint64_t x = rs + lane; x < re; x += 64) link((uint32_t)(v - lane + l), g.dst[x], parent);
    }
  }
}

}  // namespace

int wcc_hooking(const DevGraph& g, uint32_t* parent, void* workspace, hipStream_t s) {
  const uint32_t V = g.V;
  if (V == 0) return CG_OK;
  if (!g.deg) return set_error(CG_ERR_INTERNAL, "component hooking without the degree array");
  WccPlan* const plan = static_cast<WccPlan*>(workspace);
  constexpr uint64_t kSeed = 0x5EEDull;
  const dim3 block(kBlock), rows((unsigned)(((uint64_t)V + kBlock * kIlp - 1) / (kBlock * kIlp)));
  // strides; most often these return at once
  const dim3 capped(std::min(rows.x, 2048u)), chains(std::min(rows.x * (kIlp / kChainIlp), 2048u));
  hipLaunchKernelGGL(k_first, rows, block, 0, s, g, parent);
  hipLaunchKernelGGL(k_sample, dim3(1), dim3(kSamples), 0, s, g, parent, kSeed, 1u, plan);
  hipLaunchKernelGGL(k_compress<kChainIlp>, chains, block, 0, s, V, parent, plan, 2u);
  hipLaunchKernelGGL(k_link_round, capped, block, 0, s, g, 1u, plan, parent);
  hipLaunchKernelGGL(k_compress<kChainIlp>, chains, block, 0, s, V, parent, plan, 2u);
  hipLaunchKernelGGL(k_sample, dim3(1), dim3(kSamples), 0, s, g, parent, kSeed, 2u, plan);
  hipLaunchKernelGGL(k_link_rest, rows, block, 0, s, g, plan, parent);
  hipLaunchKernelGGL(k_compress<kIlp>, rows, block, 0, s, V, parent, (const WccPlan*)nullptr, 0u);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CG_ERR_HIP, "WCC kernels: %s", hipGetErrorString(e));
  return CG_OK;
}

}  // namespace cg
