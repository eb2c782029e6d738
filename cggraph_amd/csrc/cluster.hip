// The level cluster of cluster.hpp: device code and launcher.
#include "cluster.hpp"

#include "wave.hpp"

namespace cg {

namespace {

constexpr uint32_t kClosed = 0x80000000u;
constexpr uint64_t kJoinTicks = 2000;  // 20 us of the 100 MHz wall clock

template <class T>
__device__ __forceinline__ T ld_agent(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void st_agent(T* p, T x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T add_agent(T* p, T x) {
  return __hip_atomic_fetch_add(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr unsigned long long kMask40 = (1ull << 40) - 1;
// A level's report, the sum of its workgroups': arrivals (6 bits) | those that
// ask for the wide pipeline (6) | those with a long queue (6) | vertices (23) |
// out-edges (23).  A workgroup's share of the last two saturates, so that the
// fields hold kClusterMaxGroups of them: a level's sums are exact unless one
// of them reaches kShareMax (a row that long counts as kShareMax) or a queue
// had no room (stop), which is beyond the edge limit of a level.
constexpr int kFieldN = 23, kFieldM = 23, kFieldCount = 6;
constexpr uint32_t kShareMax = 1u << 17;
static_assert(kClusterMaxGroups < (1u << kFieldCount), "arrivals field");
static_assert(kClusterEdges < kShareMax && kClusterMaxGroups * (unsigned long long)kShareMax < (1ull << kFieldM), "counts field");

// A level as every workgroup sees it behind the barrier.
struct LevelView {
  uint32_t n, m, stop, uneven;
};

struct ClusterShared {
  ClusterEntry q[2][kClusterLds];
  uint32_t cnt[2];        // queue lengths by level parity
  uint32_t n, m, stop;    // the next frontier's, while it is made
  uint32_t far_cnt[2];    // far list lengths by parity
  uint32_t end[kClusterMaxGroups];
  LevelView view;
  uint32_t id, members;
  uint32_t query;
  uint32_t level, list, moves;  // between two traversals of a launch
};

// Registers the workgroup with a cluster of `want`; false: it came after the
// registration closed and leaves.
__device__ __forceinline__ bool cluster_join(ClusterShared& S, ClusterCtl* ctl, uint32_t want) {
  if (threadIdx.x == 0) {
    uint32_t id = add_agent(&ctl->join, 1u), members = 0;
    if (id == 0) {
      for (int i = 0; i < 3; ++i) st_agent(&ctl->far[i].min_val, kClusterNone);
      const uint64_t t0 = wall_clock64();
      while (ld_agent(&ctl->join) < want && wall_clock64() - t0 < kJoinTicks) __builtin_amdgcn_s_sleep(1);
      members = __hip_atomic_fetch_or(&ctl->join, kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      st_agent(&ctl->members, members);
    } else if (!(id & kClosed)) {
      // the first workgroup is running, so this ends
      while ((members = ld_agent(&ctl->members)) == 0) __builtin_amdgcn_s_sleep(1);
    }
    S.id = id;
    S.members = members;
    S.cnt[0] = S.cnt[1] = S.n = S.m = S.stop = S.far_cnt[0] = S.far_cnt[1] = 0;
    S.view = LevelView{};
    S.level = S.list = S.moves = 0;
  }
  __syncthreads();
  return !(S.id & kClosed);
}

// One traversal by a cluster.  BATCH: from J.root to its end, whatever the
// frontiers hold (a queue or list without room leaves its level's frontier to
// the bitmap, which is then expanded from there); otherwise from the frontier
// in the bitmap to its end or to a frontier that is handed back, with a record
// to the host.
template <int ALG, class WT, bool BATCH>
__device__ __forceinline__ void cluster_run(ClusterShared& S, const ClusterJob& J) {
  ClusterCtl* const ctl = J.ctl;
  const uint32_t t = threadIdx.x, lane = __lane_id(), wv = t / kWave;
  const uint32_t id = S.id, members = S.members;
  const uint32_t nthreads = members * kClusterBlock, gt = id * kClusterBlock + t;
  const uint32_t nwaves = members * kClusterWaves, gw = id * kClusterWaves + wv;
  const WT* const w = static_cast<const WT*>(J.w);

  uint32_t nv = 0, stop = 0, m = 0;  // the wavefront's part of the next frontier: vertices
                                     // (wave-uniform), wide pipeline wanted, out-edges (per lane)
  uint32_t e_done = 0, v_done = 0;   // edges and vertices expanded (per lane; SSSP, CC)
  // level, far list and redistributions, counted from the launch's start
  uint32_t L = S.level, F = S.list, moves = S.moves;

  // Ends level lvl, which filled the queue of parity qp: the workgroup adds its
  // counts to the level's report and waits until all have.  The queue read in
  // this level becomes the next one to fill.
  auto barrier = [&](uint32_t lvl, uint32_t qp) {
    const uint32_t ms = wave_sum_u32(m);
    const bool any_stop = __ballot(stop != 0) != 0;
    if (lane == 0) {
      if (nv) {
        atomicAdd(&S.n, nv);
        atomicAdd(&S.m, ms);
      }
      if (any_stop) S.stop = 1;
    }
    nv = stop = m = 0;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // the wavefront's stores and atomics are done
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (t == 0) {
      unsigned long long* const word = ctl->level[lvl % 3];
      // a queue that takes more than one round of the workgroup's lanes and
      // is twice as long as the average one of the last level
      const bool uneven = S.cnt[qp] > kClusterBlock / 4 && S.cnt[qp] > 2 * (S.view.n / members);
      unsigned long long mine = 1ull << (kFieldN + kFieldM + 2 * kFieldCount);
      mine |= (unsigned long long)S.stop << (kFieldN + kFieldM + kFieldCount);
      mine |= (unsigned long long)uneven << (kFieldN + kFieldM);
      mine |= (unsigned long long)(S.n < kShareMax ? S.n : kShareMax) << kFieldM;
      mine |= S.m < kShareMax ? S.m : kShareMax;
      unsigned long long all = add_agent(word, mine) + mine;
      while ((uint32_t)(all >> (kFieldN + kFieldM + 2 * kFieldCount)) < members) all = ld_agent(word);
      LevelView v;
      v.stop = (uint32_t)(all >> (kFieldN + kFieldM + kFieldCount)) & ((1u << kFieldCount) - 1);
      v.uneven = (uint32_t)(all >> (kFieldN + kFieldM)) & ((1u << kFieldCount) - 1);
      v.n = (uint32_t)(all >> kFieldM) & ((1u << kFieldN) - 1);
      v.m = (uint32_t)all & ((1u << kFieldM) - 1);
      S.view = v;
      S.n = S.m = S.stop = 0;
      S.cnt[qp ^ 1] = 0;
      // the word of the level after the next: every workgroup has left level
      // lvl - 1, whose word it was, and none reports there before the next barrier
      if (id == 0) st_agent(ctl->level[(lvl + 2) % 3], 0ull);
    }
    __syncthreads();
  };
  auto segment = [&](uint32_t group, uint32_t qp) { return J.q[qp] + (size_t)group * J.cap; };
  auto put = [&](uint32_t qp, uint32_t pos, unsigned long long vertex, unsigned long long row) {
    if (pos < kClusterLds) {
      S.q[qp][pos] = ClusterEntry{vertex, row};
    } else {
      ClusterEntry* const e = segment(id, qp) + pos;
      st_agent(&e->vertex, vertex);
      st_agent(&e->row, row);
    }
  };
  auto get = [&](uint32_t qp, uint32_t pos) -> ClusterEntry {
    if (pos < kClusterLds) return S.q[qp][pos];
    const ClusterEntry* const e = segment(id, qp) + pos;
    return ClusterEntry{ld_agent(&e->vertex), ld_agent(&e->row)};
  };
  // Deals the queues of parity qp out evenly (a frontier too long for that
  // stays where it is).
  auto redistribute = [&](uint32_t qp) {
    const uint32_t c = S.cnt[qp];
    ClusterEntry* const own = segment(id, qp);
    for (uint32_t i = t; i < c && i < kClusterLds; i += kClusterBlock) {
      const ClusterEntry e = S.q[qp][i];
      st_agent(&own[i].vertex, e.vertex);
      st_agent(&own[i].row, e.row);
    }
    if (t == 0) st_agent(&ctl->seg[moves & 1][id], c);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (t == 0) {
      const uint32_t target = (moves + 1) * members;
      uint32_t a = add_agent(&ctl->bar, 1u) + 1;
      while (a < target) a = ld_agent(&ctl->bar);
    }
    __syncthreads();
    if (wv == 0) {
      const uint32_t x = wave_scan(lane < members ? ld_agent(&ctl->seg[moves & 1][lane]) : 0u);
      if (lane < members) S.end[lane] = x;
    }
    __syncthreads();
    ++moves;
    const uint32_t total = S.end[members - 1];
    if ((total + members - 1) / members > kClusterLds) return;  // uniform over the cluster
    const uint32_t lo = (uint32_t)((uint64_t)total * id / members), hi = (uint32_t)((uint64_t)total * (id + 1) / members);
    for (uint32_t i = lo + t; i < hi; i += kClusterBlock) {
      uint32_t g = 0, top = members - 1;
      while (g < top) {  // the first segment that ends behind entry i
        const uint32_t mid = (g + top) / 2;
        if (S.end[mid] <= i) g = mid + 1;
        else top = mid;
      }
      const ClusterEntry* const e = segment(g, qp) + (i - (g ? S.end[g - 1] : 0u));
      S.q[qp][i - lo] = ClusterEntry{ld_agent(&e->vertex), ld_agent(&e->row)};
    }
    if (t == 0) S.cnt[qp] = hi - lo;
    __syncthreads();
  };
  // The flagged lanes' vertices join the next frontier, in the workgroup's
  // queue of parity qp.  All lanes of the wavefront call it.
  auto push = [&](bool p, uint32_t v, uint32_t value, uint64_t s, uint64_t deg, uint32_t qp) {
    const uint64_t pm = __ballot(p);
    if (!pm) return;
    nv += (uint32_t)__popcll(pm);
    if (p) {
      m += deg < kShareMax ? (uint32_t)deg : kShareMax;
      if (J.hub_degree && deg >= J.hub_degree) stop = 1;
    }
    const uint32_t pieces = p ? (uint32_t)((deg + kClusterChunk - 1) / kClusterChunk) : 0u;
    const uint64_t many = __ballot(pieces > 1);
    uint32_t pos, total;
    if (!many) {
      const uint64_t om = __ballot(pieces != 0);
      pos = (uint32_t)__popcll(om & ((1ull << lane) - 1));
      total = (uint32_t)__popcll(om);
    } else {
      const uint32_t some = pieces < J.cap ? pieces : J.cap;
      const uint32_t incl = wave_scan(some);
      pos = incl - some;
      total = lane_value(incl, kWave - 1);
    }
    uint32_t base = 0;
    if (lane == 0 && total) base = atomicAdd(&S.cnt[qp], total);
    base = lane_value(base, 0);
    if (base + total > J.cap) {
      stop = 1;  // the bitmap has the vertices: the frontier is handed back
      return;
    }
    pos += base;
    const unsigned long long vw = (unsigned long long)value << 32 | v;
    if (pieces) {
      const uint64_t len = deg < kClusterChunk ? deg : kClusterChunk;
      put(qp, pos, vw, (unsigned long long)(s | 1ull << 40 | len << 48));
    }
    for (uint64_t b = many; b; b &= b - 1) {  // long rows: the wavefront writes the other pieces
      const int l = __builtin_ctzll(b);
      const uint32_t np = __shfl(pieces, l, kWave), at = __shfl(pos, l, kWave);
      const uint64_t rs = __shfl(s, l, kWave), rd = __shfl(deg, l, kWave);
      const unsigned long long rv = __shfl(vw, l, kWave);
      for (uint32_t c = 1 + lane; c < np; c += kWave) {
        const uint64_t o = (uint64_t)c * kClusterChunk;
        const uint64_t len = rd - o < kClusterChunk ? rd - o : kClusterChunk;
        put(qp, at + c, rv, (unsigned long long)((rs + o) | len << 48));
      }
    }
  };
  auto set_bit = [&](uint64_t* bm, uint32_t v) {
    (void)__hip_atomic_fetch_or(reinterpret_cast<unsigned long long*>(bm) + (v >> 6), 1ull << (v & 63),
                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // The flagged lanes' (vertex, value) join the workgroup's part of far list
  // fl.  An entry whose vertex has a smaller value by the time the list is
  // split is dropped there: the improvement queued the vertex again.
  auto far_at = [&](uint32_t fl, uint32_t i) { return J.far[fl & 1] + (size_t)id * kClusterFar + i; };
  // Without room for it the vertex waits in the bitmap (BATCH), or the result
  // is true: it then goes into the frontier that is handed back.
  auto push_far = [&](bool p, uint32_t v, uint32_t value, uint32_t fl) -> bool {
    const uint64_t pm = __ballot(p);
    if (!pm) return false;
    uint32_t mn = p ? value : kClusterNone;
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) {
      const uint32_t o = __shfl_xor(mn, d, kWave);
      mn = o < mn ? o : mn;
    }
    uint32_t base = 0;
    if (lane == 0) {
      base = atomicAdd(&S.far_cnt[fl & 1], (uint32_t)__popcll(pm));
      (void)add_agent(&ctl->far[fl % 3].count, (uint32_t)__popcll(pm));
      (void)__hip_atomic_fetch_min(&ctl->far[fl % 3].min_val, mn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t pos = lane_value(base, 0) + (uint32_t)__popcll(pm & ((1ull << lane) - 1));
    if (p && pos < kClusterFar) st_agent(far_at(fl, pos), (unsigned long long)value << 32 | v);
    const bool full = p && pos >= kClusterFar;
    if constexpr (BATCH) {
      if (full) set_bit(J.wait, v);
      if (__ballot(full) && lane == 0) st_agent(&ctl->far[fl % 3].over, 1u);
      return false;
    }
    if (full) stop = 1;
    return full;
  };
  // The launch's record, and the next launch's control block cleared (late
  // workgroups of this one still register in its own); one wavefront.
  auto publish = [&](ClusterRecord r) {
    for (uint32_t i = lane; i < sizeof(ClusterCtl) / 8; i += kWave) reinterpret_cast<uint64_t*>(J.ctl_next)[i] = 0;
    if (lane != 0) return;
    r.tag = ~J.tag;
    *J.host_out = r;
    // the release store orders the record before its tag at system scope
    __hip_atomic_store(&J.host_out->tag, J.tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  };

  uint32_t k = J.k0;
  uint32_t thr = J.delta ? J.threshold : kClusterNone;
  uint32_t prev_n = 0;
  unsigned long long edges = 0, verts = 0;

  if constexpr (BATCH) {
    // ---- the root ----
    if (gw == 0) {
      if (lane == 0) {
        st_agent(J.val + J.root, 0u);
        set_bit(J.bm[(k - 1) & 1], J.root);
      }
      push(lane == 0, J.root, 0, J.off[J.root], J.off[J.root + 1] - J.off[J.root], L & 1);
    }
    barrier(L, L & 1);
  } else {
    // ---- the frontier taken over: counted first (one too large is left as
    // it is), then queued; the other bitmap is cleared ----
    uint64_t* in = J.bm[(k - 1) & 1];
    uint64_t* out = J.bm[k & 1];
    uint32_t c = 0;
    if constexpr (ALG == CG_BFS) {
      // the step that made the frontier counted it
      if (t < (uint32_t)kStripes) c = (uint32_t)J.bfs_cnt[(size_t)((k - 1) & 1) * kBfsCntWords + t * kBfsCntStride];
      c = wave_sum_u32(c < kShareMax ? c : kShareMax);
      if (wv == 0 && id == 0) nv = c;
    } else {
      for (uint64_t i = gt; i < J.words; i += nthreads) {
        c += (uint32_t)__popcll(in[i]);
      }
      nv = wave_sum_u32(c);
    }
    barrier(L++, 0);
    const uint32_t total = S.view.n;
    if (total == 0 || total > J.max_edges) {  // uniform over the cluster
      if (gw == 0) {
        ClusterRecord r{};
        r.n = total;
        r.threshold = thr;
        publish(r);
      }
      return;
    }
    // a wavefront takes eight words from each of eight places at a time, and
    // neighbouring places belong to different workgroups, so a frontier packed
    // into few words spreads over the queues
    const uint64_t groups = (J.words + 7) / 8;
    for (uint64_t r = 0; r * 8 * nwaves < groups; ++r) {  // uniform
      const uint64_t i = ((r * 8 + lane / 8) * nwaves + wv * members + id) * 8 + lane % 8;
      uint64_t bits = 0, waits = 0;
      if (i < J.words) {
        bits = in[i];
        st_agent(out + i, (uint64_t)0);
      }
      while (__ballot(bits != 0)) {
        bool p = bits != 0, far = false;
        uint32_t v = 0, x = 0;
        uint64_t s = 0, e = 0;
        if (p) {
          const int j = __builtin_ctzll(bits);
          v = (uint32_t)(i * 64 + (uint64_t)j);
          s = J.off[v];
          e = J.off[v + 1];
          x = ld_agent(J.val + v);
          bits &= bits - 1;
          if (ALG == CG_SSSP && x >= thr) {
            far = true;
            p = false;
          }
        }
        push(p, v, x, s, e - s, L & 1);
        if (ALG == CG_SSSP && J.delta && !push_far(far, v, x, 0) && far) waits |= 1ull << (v & 63);
      }
      if (waits) st_agent(in + i, in[i] & ~waits);
    }
    barrier(L, L & 1);
  }

  // ---- levels ----
  bool wide = false;
  for (;;) {
    const LevelView V = S.view;
    if (!BATCH && (V.stop || V.m > J.max_edges)) {
      wide = true;
      break;
    }
    uint64_t* const bin = J.bm[(k - 1) & 1];
    uint64_t* const bout = J.bm[k & 1];
    const uint32_t qc = L & 1, qp = qc ^ 1;
    const bool by_bitmap = BATCH && V.stop;
    if (V.uneven && !by_bitmap) redistribute(qc);
    if (V.n == 0 && !by_bitmap) {
      // bucketed run with nothing near: split the far list
      if (!J.delta) break;
      // (nothing is added to it in this level, so every wavefront reads the same)
      const uint32_t far_count = ld_agent(&ctl->far[F % 3].count), far_min = ld_agent(&ctl->far[F % 3].min_val);
      if (!far_count) break;
      const uint32_t last_thr = thr;
      const bool over = BATCH && ld_agent(&ctl->far[F % 3].over) != 0;
      const uint64_t nt = (uint64_t)far_min + J.delta;
      thr = nt > 0xFFFFFFFEull ? 0xFFFFFFFEu : (uint32_t)nt;
      if (gt == 0) {
        st_agent(&ctl->far[(F + 2) % 3].count, 0u);
        st_agent(&ctl->far[(F + 2) % 3].min_val, kClusterNone);
        st_agent(&ctl->far[(F + 2) % 3].over, 0u);
      }
      const uint32_t own = S.far_cnt[F & 1] < kClusterFar ? S.far_cnt[F & 1] : kClusterFar;
      for (uint32_t b = wv * kWave; b < own; b += kClusterBlock) {  // wave-uniform
        const bool in = b + lane < own;
        uint32_t v = 0, x = 0;
        uint64_t s = 0, e = 0;
        bool valid = false;
        if (in) {
          const unsigned long long far = ld_agent(far_at(F, b + lane));
          v = (uint32_t)far;
          x = (uint32_t)(far >> 32);
          valid = ld_agent(J.val + v) == x;
          s = J.off[v];
          e = J.off[v + 1];
        }
        const bool near = valid && x < thr;
        if (near) set_bit(bout, v);
        push(near, v, x, s, e - s, qp);
        if (push_far(valid && x >= thr, v, x, F + 1)) set_bit(bout, v);
      }
      if (over) {
        // the bitmap of those without room: a value below the last threshold
        // has improved since (and was queued), one that still waits keeps its
        // bit and counts for the next split
        const uint64_t places = (J.words + 7) / 8;
        uint32_t stay_n = 0, stay_min = kClusterNone;  // per lane
        for (uint64_t r = 0; r * 8 * nwaves < places; ++r) {  // uniform
          const uint64_t i = ((r * 8 + lane / 8) * nwaves + wv * members + id) * 8 + lane % 8;
          uint64_t bits = i < J.words ? ld_agent(J.wait + i) : 0ull, gone = 0;
          while (__ballot(bits != 0)) {
            bool near = false;
            uint32_t v = 0, x = 0;
            uint64_t s = 0, e = 0;
            if (bits) {
              const int j = __builtin_ctzll(bits);
              bits &= bits - 1;
              v = (uint32_t)(i * 64 + (uint64_t)j);
              x = ld_agent(J.val + v);
              if (x >= thr) {
                ++stay_n;
                stay_min = x < stay_min ? x : stay_min;
              } else {
                gone |= 1ull << j;
                near = x >= last_thr;
              }
              if (near) {
                s = J.off[v];
                e = J.off[v + 1];
                set_bit(bout, v);
              }
            }
            push(near, v, x, s, e - s, qp);
          }
          // (bits that the lists' vertices set meanwhile stay)
          if (gone)
            (void)__hip_atomic_fetch_and(reinterpret_cast<unsigned long long*>(J.wait) + i, ~(unsigned long long)gone,
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        stay_n = wave_sum_u32(stay_n);
        stay_min = wave_min_u32(stay_min);
        if (lane == 0 && stay_n) {
          ClusterFarState* const next = &ctl->far[(F + 1) % 3];
          (void)add_agent(&next->count, stay_n);
          (void)__hip_atomic_fetch_min(&next->min_val, stay_min, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          st_agent(&next->over, 1u);
        }
      }
      __syncthreads();
      if (t == 0) S.far_cnt[F & 1] = 0;
      ++F;
    } else {
      edges += V.m;
      verts += V.n;
      prev_n = V.n;
      // Expands up to 64 entries, one per lane (the first `num`): their edges
      // spread over the lanes.  now: the vertex's value at present.
      auto expand = [&](uint32_t num, uint32_t deg, uint32_t sv, uint32_t now, uint64_t s, uint32_t first_piece,
                        bool check) {
        uint64_t fresh = 0;  // entries whose vertex was not improved again since (it has another entry then)
        const uint32_t incl = wave_scan(deg);
        const uint32_t total = lane_value(incl, kWave - 1);
        const uint32_t excl = incl - deg;
        for (uint32_t j0 = 0; j0 < total; j0 += 2 * kWave) {
          // two rounds of 64 edges in flight
          bool ok[2], act[2], near[2], far[2];
          uint32_t d[2], cand[2], was[2], own[2];
          uint64_t ds[2], de[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const uint32_t j = j0 + u * kWave + lane;
            ok[u] = j < total;
            d[u] = cand[u] = was[u] = own[u] = 0;
            ds[u] = de[u] = 0;
            if (u && j0 + kWave >= total) continue;  // wave-uniform
            // the entry that holds edge j: the entries that end at or before it
            uint32_t lo = 0;
            if (num <= 16) {
              for (uint32_t i = 0; i + 1 < num; ++i) lo += lane_value(incl, i) <= j ? 1u : 0u;
            } else {
#pragma unroll
              for (uint32_t step = kWave / 2; step >= 1; step >>= 1) {
                const uint32_t pm = __shfl(excl, (int)(lo + step), kWave);
                if (pm <= j) lo += step;
              }
            }
            const uint64_t os = __shfl(s, (int)lo, kWave);
            const uint32_t osv = __shfl(sv, (int)lo, kWave);
            const uint32_t oex = __shfl(excl, (int)lo, kWave);
            own[u] = lo;
            if (ok[u]) {
              const uint64_t e = os + (j - oex);
              d[u] = J.dst[e];
              if constexpr (ALG == CG_BFS) cand[u] = osv + 1;
              else if constexpr (ALG == CG_SSSP) cand[u] = osv + (uint32_t)w[e];
              else cand[u] = osv;
            }
          }
          if constexpr (ALG != CG_BFS) {
            // the entry's value was loaded beside the destinations
            if (j0 == 0) {
              const bool f = lane < num && now == sv;
              fresh = __ballot(f);
              if (f) {
                e_done += deg;
                v_done += first_piece;
              }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) ok[u] = ok[u] && (fresh >> own[u] & 1);
          }
          if (check) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
              if (ok[u]) was[u] = ld_agent(J.val + d[u]);
#pragma unroll
            for (int u = 0; u < 2; ++u) ok[u] = ok[u] && cand[u] < was[u];
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            if (ok[u]) {
              // the row bounds are needed only if the value falls; loading
              // them beside the atomic takes them out of the level's chain
              ds[u] = J.off[d[u]];
              de[u] = J.off[d[u] + 1];
              was[u] = __hip_atomic_fetch_min(J.val + d[u], cand[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            act[u] = ok[u] && cand[u] < was[u];
            near[u] = far[u] = false;
            if (act[u]) {
              far[u] = ALG == CG_SSSP && cand[u] >= thr;
              near[u] = !far[u];
              if (near[u]) set_bit(bout, d[u]);
            }
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            push(near[u], d[u], cand[u], ds[u], de[u] - ds[u], qp);
            if (ALG == CG_SSSP && J.delta && push_far(far[u], d[u], cand[u], F)) set_bit(bout, d[u]);
          }
        }
      };
      if (by_bitmap) {
        const uint64_t places = (J.words + 7) / 8;
        for (uint64_t r = 0; r * 8 * nwaves < places; ++r) {  // uniform
          const uint64_t i = ((r * 8 + lane / 8) * nwaves + wv * members + id) * 8 + lane % 8;
          uint64_t bits = i < J.words ? ld_agent(bin + i) : 0ull;
          if (bits) st_agent(bin + i, (uint64_t)0);
          while (__ballot(bits != 0)) {
            uint32_t sv = 0, deg = 0;
            uint64_t s = 0;
            if (bits) {
              const uint32_t v = (uint32_t)(i * 64 + (uint64_t)__builtin_ctzll(bits));
              bits &= bits - 1;
              s = J.off[v];
              deg = (uint32_t)(J.off[v + 1] - s);
              sv = ld_agent(J.val + v);
            }
            expand(kWave, deg, sv, sv, s, 0, true);
          }
        }
      }
      const uint32_t tail = by_bitmap ? 0u : S.cnt[qc];
      const bool check = V.m > kClusterCheck;
      uint32_t gs = (tail + kClusterWaves - 1) / kClusterWaves;
      if (gs > (uint32_t)kWave) gs = kWave;
      for (uint32_t first = wv * gs; first < tail; first += kClusterWaves * gs) {  // wave-uniform
        const uint32_t num = tail - first < gs ? tail - first : gs;
        uint32_t deg = 0, sv = 0, now = 0, first_piece = 0;
        uint64_t s = 0;
        if (lane < num) {
          const ClusterEntry e = get(qc, first + lane);
          const uint32_t v = (uint32_t)e.vertex;
          sv = (uint32_t)(e.vertex >> 32);
          s = e.row & kMask40;
          deg = (uint32_t)(e.row >> 48);
          st_agent(bin + (v >> 6), (uint64_t)0);  // every vertex of the word is in this frontier
          if constexpr (ALG != CG_BFS) now = ld_agent(J.val + v);
          first_piece = e.row >> 40 & 1;
        }
        expand(num, deg, sv, now, s, first_piece, check);
      }
    }
    ++L;
    ++k;
    barrier(L, qp);
  }

  if constexpr (BATCH) {
    __syncthreads();  // every wavefront has read the view and the counters kept for the next traversal
    if (t == 0) {
      S.level = L + 1;
      S.list = F;
      S.moves = moves;
      if (id == 0) atomicMax(J.batch_levels, k - J.k0);
    }
    __syncthreads();
    return;
  }

  // ---- the end ----
  const LevelView V = S.view;
  if constexpr (ALG != CG_BFS) {
    const unsigned long long es = ((unsigned long long)wave_sum_u32(e_done >> 16) << 16) + wave_sum_u32(e_done & 0xFFFFu);
    v_done = wave_sum_u32(v_done);
    if (lane == 0 && v_done) {
      (void)add_agent(&ctl->edges_done, es);
      (void)add_agent(&ctl->verts_done, (unsigned long long)v_done);
    }
    if (wide && J.delta) {
      // a frontier handed back keeps the waiting vertices in it
      const uint32_t own = S.far_cnt[F & 1] < kClusterFar ? S.far_cnt[F & 1] : kClusterFar;
      for (uint32_t i = t; i < own; i += kClusterBlock)
        set_bit(J.bm[(k - 1) & 1], (uint32_t)ld_agent(far_at(F, i)));
    }
    barrier(L + 1, 0);
    edges = ld_agent(&ctl->edges_done);
    verts = ld_agent(&ctl->verts_done);
  }
  // The front kernel sizes its chunks by the out-edges of the frontier handed
  // back, so it needs their number even where the report's saturates; the
  // vertices are exact (one level's edges discovered them).  One pass over the
  // bitmap; bits of vertices without edges add nothing.
  unsigned long long front_m = V.m;
  if constexpr (ALG == CG_BFS) {
    if (wide && k != J.k0 && (V.stop || V.m >= kShareMax)) {  // uniform over the cluster
      const uint64_t* const front = J.bm[(k - 1) & 1];
      unsigned long long ms = 0;
      for (uint64_t i = gt; i < J.words; i += nthreads)
        for (uint64_t bits = ld_agent(front + i); bits; bits &= bits - 1) {
          const uint64_t v = i * 64 + (uint64_t)__builtin_ctzll(bits);
          ms += J.off[v + 1] - J.off[v];
        }
      ms = wave_sum_u64(ms);
      if (lane == 0 && ms) (void)add_agent(&ctl->edges_done, ms);
      barrier(L + 1, 0);
      front_m = ld_agent(&ctl->edges_done);
    }
  }
  if (gw != 0) return;
  if (wide && lane == 0) {
    if constexpr (ALG == CG_BFS) {
      const uint32_t c = (k - 1) & 1;
      RunState r = J.rs[(J.k0 - 1) & 1];
      r.visited += verts;
      r.iter = k - 1;
      r.pull = 0;
      r.m_explored += edges;
      if (prev_n) r.prev_active = prev_n;
      J.rs[c] = r;
      if (k != J.k0) {  // a frontier handed back as it was taken over has its counts
        unsigned long long* const bc = J.bfs_cnt + (size_t)c * kBfsCntWords;
        for (int i = 0; i < kStripes; ++i)
          for (int j = 0; j < 3; ++j) bc[i * kBfsCntStride + j] = 0;
        bc[0] = V.n;
        bc[1] = front_m;
      }
    } else {
      J.rs->iter = k - 1;
      J.rs->pad = 0;
    }
    for (int i = 0; i < 2; ++i) {
      J.st[i].n_small = 0;
      J.st[i].n_med = 0;
      J.st[i].n_chunk = 0;
      J.st[i].min_val = kClusterNone;  // no hub waits in the next iteration
      J.st[i].choice = -1;
    }
  }
  ClusterRecord r{};
  r.levels = k - J.k0;
  r.n = wide ? (V.n ? V.n : 1u) : 0;  // (a full far list hands back waiting vertices only)
  r.threshold = thr;
  r.edges = edges;
  r.verts = verts;
  publish(r);
}

template <int ALG, class WT>
__global__ __launch_bounds__(kClusterBlock) void k_cluster(ClusterJob J) {
  __shared__ ClusterShared S;
  if (cluster_join(S, J.ctl, gridDim.x)) cluster_run<ALG, WT, false>(S, J);
}

// Batched queries: clusters of b.groups workgroups take queries from the list
// in order until none is left.
__global__ __launch_bounds__(kClusterBlock) void k_cluster_batch(ClusterBatch b) {
  __shared__ ClusterShared S;
  const uint32_t c = blockIdx.x / b.groups;
  ClusterCtl* const ctl = b.ctl + c;
  if (!cluster_join(S, ctl, b.groups)) return;
  for (uint32_t turn = 1;; ++turn) {
    // the first workgroup takes the next query; the others wait for its turn
    if (threadIdx.x == 0) {
      uint32_t q;
      if (S.id == 0) {
        q = add_agent(b.next, 1u);
        st_agent(&ctl->query, (unsigned long long)turn << 32 | q);
      } else {
        unsigned long long x;
        do {
          __builtin_amdgcn_s_sleep(2);
          x = ld_agent(&ctl->query);
        } while ((x >> 32) != turn);
        q = (uint32_t)x;
      }
      S.query = q;
    }
    __syncthreads();
    const uint32_t qi = S.query;
    if (qi >= b.nq) return;  // uniform over the cluster
    const ClusterQuery Q = b.q[qi];
    ClusterJob J{};
    J.off = Q.off;
    J.dst = Q.dst;
    J.w = Q.w;
    J.val = Q.val;
    J.bm[0] = Q.bm;
    J.bm[1] = Q.bm + Q.words;
    J.words = Q.words;
    J.cap = b.cap;
    J.q[0] = b.entries + (size_t)c * 2 * b.groups * b.cap;
    J.q[1] = J.q[0] + (size_t)b.groups * b.cap;
    J.far[0] = b.far + (size_t)c * 2 * b.groups * kClusterFar;
    J.far[1] = J.far[0] + (size_t)b.groups * kClusterFar;
    J.k0 = 1;
    J.root = Q.root;
    J.delta = Q.delta;
    J.threshold = Q.delta;
    J.ctl = ctl;
    J.batch_levels = b.levels;
    J.wait = Q.bm + 2 * Q.words;
    if (Q.alg == CG_BFS) cluster_run<CG_BFS, uint32_t, true>(S, J);
    else cluster_run<CG_SSSP, uint32_t, true>(S, J);
  }
}

}  // namespace

int launch_cluster_batch(const ClusterBatch& b, uint32_t clusters, hipStream_t s) {
  if (b.groups < 1 || b.groups > kClusterMaxGroups || !clusters)
    return set_error(CG_ERR_INTERNAL, "%u clusters of %u workgroups", clusters, b.groups);
  hipLaunchKernelGGL(k_cluster_batch, dim3(clusters * b.groups), dim3(kClusterBlock), 0, s, b);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CG_ERR_HIP, "batched level clusters: %s", hipGetErrorString(e));
  return CG_OK;
}

int launch_cluster(int alg, int w_bytes, const ClusterJob& job, uint32_t groups, hipStream_t s) {
  if (groups < 1 || groups > kClusterMaxGroups) return set_error(CG_ERR_INTERNAL, "level cluster of %u workgroups", groups);
  const dim3 grid(groups), block(kClusterBlock);
  if (alg == CG_BFS) hipLaunchKernelGGL((k_cluster<CG_BFS, uint32_t>), grid, block, 0, s, job);
  else if (alg == CG_CC) hipLaunchKernelGGL((k_cluster<CG_CC, uint32_t>), grid, block, 0, s, job);
  else if (alg == CG_SSSP && w_bytes == 1) hipLaunchKernelGGL((k_cluster<CG_SSSP, uint8_t>), grid, block, 0, s, job);
  else if (alg == CG_SSSP && w_bytes == 2) hipLaunchKernelGGL((k_cluster<CG_SSSP, uint16_t>), grid, block, 0, s, job);
  else if (alg == CG_SSSP) hipLaunchKernelGGL((k_cluster<CG_SSSP, uint32_t>), grid, block, 0, s, job);
  else return set_error(CG_ERR_INTERNAL, "level cluster: algorithm %d", alg);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(CG_ERR_HIP, "level cluster launch: %s", hipGetErrorString(e));
  return CG_OK;
}

}  // namespace cg
