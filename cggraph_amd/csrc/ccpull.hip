// Label propagation (directed CC): bottom-up rounds in front of the push
// rounds.
//
// Every label that travels is the id of a vertex with out-edges, so none is
// below z, the smallest such vertex: a vertex that has found a neighbour
// labelled z is done.  Where z's out-neighbours send many edges (the rule
// below), a bottom-up round in which every vertex stops at the first in-neighbour
// labelled z settles almost all of them after a few edges each, as
// direction-optimising BFS does (Beamer, Asanovic, Patterson, SC'12), where a
// push round relaxes every edge with a gather and often an atomic.  Directed
// R-MAT s22, 4.2 M vertices, 65 M edges: the first push round took 676 us; two
// rounds here take 68 + 34 us and leave 0.1 M edges to push (0.94 -> 0.29 ms
// per query).  A third round never had enough to do on R-MAT s13-s22.
//
// The rule: z's out-neighbours send at least 1/16 of the edges -- Beamer's
// line, where a vertex finds a neighbour labelled z after about 16 edges -- and
// the graph has more edges than the level cluster takes at once.  It is a
// property of the graph, found with the engine (cc_source).
//
// A vertex not at z takes the minimum over all its in-neighbours, so after a
// round only the out-edges of vertices that changed in it are open: the
// round leaves exactly those in the frontier bitmap and pushes go on from
// there.  Values may be read while they fall; whoever falls is in the bitmap.
//
// Rows: a lane scans up to kLaneEdges in-edges of its own, the wavefront the
// rest of the rows that are not settled then, and rows of more than
// kLongRow edges go to a list that a second kernel takes a workgroup each, so
// that no hub outside z's reach holds one wavefront up.
#include "kernels.hpp"
#include "wave.hpp"

namespace cg {

namespace {

constexpr int kBlock = 256;
constexpr int kLongBlock = 1024;
constexpr uint32_t kLaneEdges = 32;
constexpr uint64_t kLongRow = 16384;

__device__ __forceinline__ uint32_t min_u32(uint32_t a, uint32_t b) { return a < b ? a : b; }

// Whether round r has anything to do: the first always, the second if the
// vertices changed in the one before send many edges.  Every workgroup takes
// the same decision.
__device__ __forceinline__ bool runs(const CcPullCounters* cnt, int r, uint64_t E) {
  if (r == 0) return true;
  unsigned long long m = 0;
#pragma unroll
  for (int k = 0; k < kStripes; ++k) m += cnt[r - 1].edges[k * kCcStride];
  return m * kCcShare > E;
}

__global__ __launch_bounds__(kBlock) void k_cc_pull(DevGraph g, uint64_t E, uint32_t z, uint32_t* __restrict__ val,
                                                    uint64_t* __restrict__ changed_bm, CcPullCounters* cnt, int r,
                                                    uint32_t* __restrict__ list) {
  if (!runs(cnt, r, E)) return;
  const uint32_t lane = __lane_id();
  const uint64_t words = ((uint64_t)g.V + 63) / 64;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
  unsigned long long m = 0;
  for (uint64_t wd = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; wd < words; wd += nwaves) {
    const uint64_t v = wd * 64 + lane;
    uint32_t cur = v < g.V ? val[v] : 0u;
    uint64_t k = 0, e = 0;
    if (v < g.V && cur > z) {
      k = g.in_off[v];
      e = g.in_off[v + 1];
    }
    uint32_t best = cur;
    const uint64_t own = e - k < kLaneEdges ? e : k + kLaneEdges;
    for (; k < own && best != z;) {
      // four gathers in flight per lane
      uint32_t u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = g.in_src[k + j < own ? k + j : k];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = val[u[j]];
      best = min_u32(best, min_u32(min_u32(u[0], u[1]), min_u32(u[2], u[3])));
      k += 4;
    }
    bool more = best != z && k < e;
    if (more && e - k > kLongRow) {
      list[atomicAdd(&cnt[r].rows, 1u)] = (uint32_t)v;
      more = false;
    }
    for (uint64_t need = __ballot(more); need; need &= need - 1) {
      const int l = __builtin_ctzll(need);
      const uint64_t re = __shfl(e, l, kWave);
      uint32_t x = 0xFFFFFFFFu;
      for (uint64_t b = __shfl(k, l, kWave); b < re; b += 4 * kWave) {  // wave-uniform
        uint32_t u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = g.in_src[b + j * kWave + lane < re ? b + j * kWave + lane : b];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = val[u[j]];
        x = min_u32(x, min_u32(min_u32(u[0], u[1]), min_u32(u[2], u[3])));
        if (__ballot(x == z)) break;
      }
      x = wave_min_u32(x);
      if ((int)lane == l) best = min_u32(best, x);
    }
    const bool fell = best < cur;
    if (fell) {
      val[v] = best;
      m += g.deg[v];
    }
    const uint64_t mask = __ballot(fell);
    if (lane == 0) changed_bm[wd] = mask;
  }
  m = wave_sum_u64(m);
  if (lane == 0 && m) atomicAdd(&cnt[r].edges[(blockIdx.x % kStripes) * kCcStride], m);
}

__global__ __launch_bounds__(kLongBlock) void k_cc_pull_long(DevGraph g, uint64_t E, uint32_t z,
                                                             uint32_t* __restrict__ val,
                                                             uint64_t* __restrict__ changed_bm, CcPullCounters* cnt,
                                                             int r, const uint32_t* __restrict__ list) {
  if (!runs(cnt, r, E)) return;
  __shared__ uint32_t best;
  const uint32_t n = cnt[r].rows;
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t v = list[i];
    const uint64_t s = g.in_off[v], e = g.in_off[v + 1];
    if (threadIdx.x == 0) best = 0xFFFFFFFFu;
    __syncthreads();
    uint32_t x = 0xFFFFFFFFu;
    for (uint64_t k = s + threadIdx.x; k < e; k += 4 * kLongBlock) {
      uint32_t u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = g.in_src[k + j * kLongBlock < e ? k + j * kLongBlock : k];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = val[u[j]];
      x = min_u32(x, min_u32(min_u32(u[0], u[1]), min_u32(u[2], u[3])));
      if (x == z) break;
    }
    x = wave_min_u32(x);
    if (__lane_id() == 0) atomicMin(&best, x);
    __syncthreads();
    if (threadIdx.x == 0 && best < val[v]) {
      val[v] = best;
      atomicOr(reinterpret_cast<unsigned long long*>(changed_bm) + (v >> 6), 1ull << (v & 63));
      atomicAdd(&cnt[r].edges[(blockIdx.x % kStripes) * kCcStride], (unsigned long long)g.deg[v]);
    }
    __syncthreads();
  }
}

// out[0]: the smallest vertex with out-edges
__global__ __launch_bounds__(kBlock) void k_first_source(const uint32_t* __restrict__ deg, uint32_t V,
                                                         uint32_t* __restrict__ out) {
  uint32_t x = 0xFFFFFFFFu;
  for (uint64_t v = blockIdx.x * (uint64_t)kBlock + threadIdx.x; v < V && x == 0xFFFFFFFFu;
       v += (uint64_t)gridDim.x * kBlock)
    if (deg[v]) x = (uint32_t)v;
  x = wave_min_u32(x);
  if (__lane_id() == 0 && x != 0xFFFFFFFFu) atomicMin(out, x);
}

// the out-edges of z's out-neighbours
__global__ __launch_bounds__(kBlock) void k_source_reach(DevGraph g, const uint32_t* __restrict__ z,
                                                         unsigned long long* __restrict__ m) {
  if (*z >= g.V) return;
  const uint64_t s = g.off[*z], e = g.off[*z + 1];
  unsigned long long x = 0;
  for (uint64_t k = s + blockIdx.x * (uint64_t)kBlock + threadIdx.x; k < e; k += (uint64_t)gridDim.x * kBlock)
    x += g.deg[g.dst[k]];
  x = wave_sum_u64(x);
  if (__lane_id() == 0 && x) atomicAdd(m, x);
}

}  // namespace

int cc_source(const DevGraph& g, uint64_t E, uint32_t* z, bool* pull, hipStream_t s) {
  *z = 0;
  *pull = false;
  if (!g.V || !E) return CG_OK;
  DevBuf<unsigned long long> out;
  CG_TRY(out.ensure(2));
  CG_TRY(launch_fill_u64(reinterpret_cast<uint64_t*>(out.p), 0, 1, s));
  CG_TRY(launch_fill_u64(reinterpret_cast<uint64_t*>(out.p) + 1, ~0ull, 1, s));
  uint32_t* const dz = reinterpret_cast<uint32_t*>(out.p + 1);
  hipLaunchKernelGGL(k_first_source, dim3(256), dim3(kBlock), 0, s, g.deg, g.V, dz);
  hipLaunchKernelGGL(k_source_reach, dim3(256), dim3(kBlock), 0, s, g, dz, out.p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CG_ERR_HIP, "label source: %s", hipGetErrorString(e));
  unsigned long long h[2] = {0, 0};
  CG_HIP(hipMemcpyAsync(h, out.p, sizeof(h), hipMemcpyDeviceToHost, s));
  CG_HIP(hipStreamSynchronize(s));
  *z = (uint32_t)h[1];
  *pull = h[0] * kCcShare > E;
  return CG_OK;
}

uint64_t cc_pull_list_size(uint64_t E) { return E / kLongRow + 1; }

int launch_cc_pull(const DevGraph& g, uint64_t E, uint32_t z, uint32_t* val, uint64_t* changed_bm, CcPullCounters* cnt,
                   uint32_t* list, hipStream_t s) {
  if (!g.in_off || !g.in_src || !g.deg) return set_error(CG_ERR_INTERNAL, "bottom-up labels without in-edges");
  const uint64_t words = ((uint64_t)g.V + 63) / 64;
  const uint64_t blocks = (words + kBlock / kWave - 1) / (kBlock / kWave);
  const dim3 grid((unsigned)(blocks < 8192 ? blocks : 8192));
  for (int r = 0; r < kCcRounds; ++r) {
    hipLaunchKernelGGL(k_cc_pull, grid, dim3(kBlock), 0, s, g, E, z, val, changed_bm, cnt, r, list);
    hipLaunchKernelGGL(k_cc_pull_long, dim3(256), dim3(kLongBlock), 0, s, g, E, z, val, changed_bm, cnt, r, list);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CG_ERR_HIP, "bottom-up labels: %s", hipGetErrorString(e));
  return CG_OK;
}

}  // namespace cg
