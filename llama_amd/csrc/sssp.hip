// Weighted single-source shortest paths (task sssp_weighted,
// benchmark/benchmarks/sssp.h:59-172) over the snapshot out-CSR and its
// per-edge FP32 weights (the levels' `weight` property, compacted with the
// snapshot).
//
// The reference runs synchronous Bellman-Ford rounds over the vertices
// updated in the previous round.  Here the rounds follow the near/far
// schedule (Davidson, Baxter, Garland, Owens, IPDPS 2014): a round relaxes
// the out-edges of a queue of vertices edge-parallel, in one launch, with
// atomicMin on the distances' bit patterns -- non-negative FP32 values order like their
// unsigned bit patterns.  A vertex whose distance dropped below the threshold
// T is queued for the next round once (round stamp); one whose new distance is
// >= T is flagged far.  Rounds are launched several at a time: their queue
// lengths and the decision whether a round runs stay on the device, and the
// host reads them back per batch.  When the queue runs dry, T grows by delta and the far
// vertices now below T whose distance changed since their edges were last
// relaxed form the next queue.  Every order of relaxations ends at the same
// fixed point, dist[v] = min over paths of the FP32 sums dist[u] + w taken in
// path order (each sum is monotone in dist[u] and never below it), so
// distances match the reference bit for bit; the schedule only cuts repeated
// relaxations.  Unreached vertices keep INT_MAX-1 converted to float, as the
// reference stores them.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>

#include "ll_gpu_internal.h"

namespace llgpu {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr float kUnreachedDist = float(INT_MAX - 1);
constexpr uint64_t kAutoMinQueueDiv = 8;  // smallest tail phase queue: V / 8 vertices
constexpr uint32_t kBigRow = 256;         // out-edges past which a queued vertex is shared by the grid
constexpr uint32_t kChunk = 1024;         // edges of such a vertex one workgroup takes
constexpr uint32_t kStage = 2048;         // appends a workgroup stages
constexpr uint32_t kNotRelaxed = ~0u;     // a NaN pattern: equal to no distance; -1 as an int

// A round's queue: n vertices of up to kBigRow out-edges, n_big chunks of
// vertices with more; the edges relaxed by the round itself and by all rounds before it.  Rounds use
// a ring of slots: round r reads slot r, fills slot r + 1 and zeroes slot r + 2.
struct alignas(64) Slot {
  unsigned long long n, n_big, edges, before;
};
constexpr int kSlots = 8;
// rounds launched per host read-back; those past the end of a phase find an
// empty queue
constexpr int kBatch = 3;
static_assert(kBatch + 3 <= kSlots, "the slots of a batch and its neighbours are distinct");

struct Queues {
  uint32_t* q[2];  // by round parity
  uint2* big[2];   // {vertex, chunk}
};

struct RelaxArgs {
  Queues qs;
  Slot* slots;
  const uint64_t* ofs;
  const uint32_t* adj;
  const float* w;
  const uint32_t* outdeg;
  uint32_t* dist;
  int32_t* stamp;
  uint8_t* far;
  uint32_t* relaxed;
  uint64_t E, min_queue;
  uint32_t t_bits;
  bool near_far;
};

// A vertex of more than kBigRow out-edges (d) joins its round's list, chunk by
// chunk.  Several waves read its distance, which may drop meanwhile, so
// `relaxed` keeps the largest one any of them used since the vertex last left
// the far pile (as ints; the scatter resets it to -1, below every distance).
// It is not reset when a round lists the vertex: chunks of it may still be
// waiting in that same round, and a later small value would hide that the
// earlier ones used a larger distance.
__device__ inline void list_chunks(uint2* big, uint64_t at, uint32_t v, uint32_t d) {
  for (uint32_t c = 0; c < (d + kChunk - 1) / kChunk; c++) big[at + c] = make_uint2(v, c);
}

__global__ void k_sssp_init(uint32_t* dist, int32_t* stamp, uint8_t* far, uint32_t* relaxed,
                            uint64_t V, uint32_t root, const uint32_t* outdeg, Queues qs,
                            Slot* slots, uint32_t* hist, uint32_t nhist) {
  const uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (v < V) {
    dist[v] = v == root ? __float_as_uint(0.0f) : __float_as_uint(kUnreachedDist);
    stamp[v] = -1;
    relaxed[v] = kNotRelaxed;
  }
  if (v < (V + 3) / 4 * 4) far[v] = 0;
  if (blockIdx.x == 0) {
    if (threadIdx.x < kSlots) {
      Slot t{0, 0, 0, 0};
      if (threadIdx.x == 0) {  // a root without out-edges gives an empty first round
        const uint32_t d = outdeg[root];
        t.n = d > 0 && d <= kBigRow ? 1 : 0;
        t.n_big = d > kBigRow ? (d + kChunk - 1) / kChunk : 0;
      }
      slots[threadIdx.x] = t;
    }
    for (uint32_t i = threadIdx.x; i < nhist; i += blockDim.x) hist[i] = i + 1 < nhist ? 0u : ~0u;
  }
  if (v == root) {
    qs.q[0][0] = root;
    if (outdeg[root] > kBigRow) list_chunks(qs.big[0], 0, root, outdeg[root]);
  }
}

// Whether a round of n queued vertices runs: small queues rejoin the far pile
// in the tail, once edges worth half the snapshot have been relaxed (early
// phases keep the step).
__host__ __device__ inline bool round_runs(uint64_t n, uint64_t done, uint64_t E,
                                           uint64_t min_queue, bool near_far, bool force) {
  return n > 0 && (!near_far || force || done * 2 < E || n >= min_queue);
}

// One edge: lowers the distance of its head; a head with out-edges whose
// distance dropped below the threshold is queued for the next round once
// (stamp), else flagged far.  Returns 1 (queue), 2 (queue, big row) or 0.
__device__ inline int relax_edge(const RelaxArgs& a, uint32_t v, float cand, int32_t next) {
  const uint32_t cb = __float_as_uint(cand);
  if (cb >= a.dist[v] || cb >= atomicMin(&a.dist[v], cb)) return 0;
  const uint32_t od = a.outdeg[v];
  if (od == 0) return 0;
  if (cb >= a.t_bits) {
    a.far[v] = 1;
    return 0;
  }
  if (atomicExch(&a.stamp[v], next) == next) return 0;
  return od > kBigRow ? 2 : 1;
}

// Big vertices of a workgroup, staged in LDS so that their chunks take one
// reservation on the list's counter (one each: 1.1 ms for the 30000 of a
// split at 2^24 vertices).
struct BigStage {
  static constexpr uint32_t kRoom = 512;
  uint32_t v[kRoom], at[kRoom];
  uint32_t n, chunks;
  unsigned long long base;

  __device__ void clear() {  // one thread
    n = 0;
    chunks = 0;
  }
  __device__ void add(uint32_t x, uint32_t d, uint2* big, unsigned long long* n_big) {
    const uint32_t k = (d + kChunk - 1) / kChunk;
    const uint32_t i = atomicAdd(&n, 1u);
    if (i < kRoom) {
      v[i] = x;
      at[i] = atomicAdd(&chunks, k);
    } else {
      list_chunks(big, atomicAdd(n_big, (unsigned long long)k), x, d);
    }
  }
  // every thread of the workgroup, the stage complete; clears it
  __device__ void flush(const uint32_t* outdeg, uint2* big, unsigned long long* n_big) {
    __syncthreads();
    const uint32_t m = min(n, kRoom);
    if (m) {  // uniform
      if (threadIdx.x == 0) base = atomicAdd(n_big, (unsigned long long)chunks);
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < m; i += kBlock) list_chunks(big, base + at[i], v[i], outdeg[v[i]]);
      __syncthreads();
      if (threadIdx.x == 0) clear();
    }
  }
};

// The calling wave's appends (take) to the workgroup's stage, or straight to
// the queue once the stage is full: *l_end is the first position that did not
// fit (every later one does not either), so the stage holds the positions
// below min(*l_n, *l_end).
__device__ inline void wave_append(bool take, uint32_t v, uint32_t* l_q, uint32_t* l_n,
                                   uint32_t* l_end, uint32_t* q, unsigned long long* n) {
  const uint64_t m = __ballot(take);
  if (!m) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((long long)m) - 1;
  const uint32_t k = uint32_t(__popcll(m));
  const uint32_t rank = uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1)));
  uint32_t at = 0;
  if (lane == leader) at = atomicAdd(l_n, k);
  at = uint32_t(__shfl(int(at), leader, 64));
  if (at + k <= kStage) {
    if (take) l_q[at + rank] = v;
  } else {
    unsigned long long g = 0;
    if (lane == leader) {
      atomicMin(l_end, at);
      g = atomicAdd(n, (unsigned long long)k);
    }
    g = __shfl(g, leader, 64);
    if (take) q[g + rank] = v;
  }
}

// One round in one launch over a fixed grid: no prefix sum of the queue's
// degrees is needed.  A wave takes 64 queued vertices, scans their degrees in
// registers and relaxes their edges flattened over its lanes; the workgroups
// share the edges of the big ones.  Appends are staged in LDS and reserved
// with one atomic per workgroup (the queue counter is a single address).
// Bound by the gathers of the heads' distances and, in most rounds, by the
// launch and the latency of the wave's dependent loads.  2^20 vertices, 16.8 M
// edges: 4.19 -> 1.86 ms a search against one launch each for the queue's
// degrees, their prefix sum, the blocks' bounds and the relaxation with a
// round trip per round (2.34 with the same steps); 2^24 vertices 9.6 -> 8.3.
// kBigRow 512: 2.01, 1024: 2.08; 64 queued vertices a wave whatever their
// number: 6.6.
__global__ __launch_bounds__(kBlock) void k_relax(RelaxArgs a, uint32_t round, bool force) {
  __shared__ uint32_t l_pre[kWaves][64];
  __shared__ uint64_t l_base[kWaves][64];
  __shared__ float l_dist[kWaves][64];
  __shared__ uint32_t l_q[kStage];
  __shared__ uint32_t l_n, l_end;
  __shared__ BigStage l_big;
  __shared__ unsigned long long l_at;
  Slot& cur = a.slots[round % kSlots];
  Slot& nxt = a.slots[(round + 1) % kSlots];
  const Slot& prev = a.slots[(round + kSlots - 1) % kSlots];
  const unsigned long long done = prev.before + prev.edges;
  const uint64_t n = cur.n, n_big = cur.n_big;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    cur.before = done;
    a.slots[(round + 2) % kSlots] = Slot{0, 0, 0, 0};
  }
  if (!round_runs(n + n_big, done, a.E, a.min_queue, a.near_far, force)) return;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t* q = a.qs.q[round & 1];
  uint32_t* q_next = a.qs.q[(round + 1) & 1];
  uint2* big_next = a.qs.big[(round + 1) & 1];
  const int32_t next = int32_t(round + 1);
  if (threadIdx.x == 0) {
    l_n = 0;
    l_end = kStage;
    l_big.clear();
  }
  __syncthreads();
  unsigned long long edges = 0;
  // entries a wave takes at a time: as few as spread the queue over the grid
  const uint64_t waves = uint64_t(gridDim.x) * kWaves;
  const uint32_t per = uint32_t(min(uint64_t(64), (n + waves - 1) / waves));
  for (uint64_t i0 = (uint64_t(blockIdx.x) * kWaves + wave) * per; i0 < n; i0 += waves * per) {
    uint32_t d = 0;
    if (lane < per && i0 + lane < n) {
      const uint32_t v = q[i0 + lane];
      d = a.outdeg[v];
      const uint32_t x = a.dist[v];
      a.relaxed[v] = x;
      l_dist[wave][lane] = __uint_as_float(x);
      l_base[wave][lane] = a.ofs[v];
    }
    uint32_t inc = d;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o, 64);
      if (lane >= uint32_t(o)) inc += y;
    }
    const uint32_t total = __shfl(inc, 63, 64);
    l_pre[wave][lane] = inc;  // edges of the entries up to this one
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) edges += total;
    for (uint32_t x0 = 0; x0 < total; x0 += 64 * 4) {
      uint32_t head[4];
      float cand[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t x = x0 + 64u * uint32_t(k) + lane;
        uint32_t lo = 0;  // the first entry with l_pre > x
#pragma unroll
        for (uint32_t h = 32; h > 0; h >>= 1)
          if (l_pre[wave][lo + h - 1] <= x) lo += h;
        lo = min(lo, 63u);
        const uint64_t e = l_base[wave][lo] + (x - (lo ? l_pre[wave][lo - 1] : 0u));
        const bool in = x < total;
        head[k] = in ? a.adj[e] : 0u;
        cand[k] = in ? l_dist[wave][lo] + a.w[e] : kUnreachedDist;
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int r = x0 + 64u * uint32_t(k) + lane < total ? relax_edge(a, head[k], cand[k], next) : 0;
        if (r == 2) l_big.add(head[k], a.outdeg[head[k]], big_next, &nxt.n_big);
        wave_append(r == 1, head[k], l_q, &l_n, &l_end, q_next, &nxt.n);
      }
    }
    __builtin_amdgcn_wave_barrier();  // the wave's LDS is rewritten
  }
  // big vertices: a workgroup per chunk
  const uint2* big = a.qs.big[round & 1];
  for (uint64_t k = blockIdx.x; k < n_big; k += gridDim.x) {
    const uint2 t = big[k];
    const uint32_t v = t.x;
    const uint64_t e0 = a.ofs[v];
    const uint64_t lo = e0 + uint64_t(t.y) * kChunk, hi = min(e0 + a.outdeg[v], lo + kChunk);
    // one read for the wave
    const uint32_t xb = uint32_t(__shfl(int(lane == 0 ? a.dist[v] : 0u), 0, 64));
    if (lane == 0) atomicMax(reinterpret_cast<int*>(&a.relaxed[v]), int(xb));
    const float xd = __uint_as_float(xb);
    if (threadIdx.x == 0) edges += hi - lo;
    uint32_t head[kChunk / kBlock];
    float cand[kChunk / kBlock];
#pragma unroll
    for (uint32_t u = 0; u < kChunk / kBlock; u++) {
      const uint64_t e = lo + u * kBlock + threadIdx.x;
      head[u] = e < hi ? a.adj[e] : 0u;
      cand[u] = e < hi ? xd + a.w[e] : kUnreachedDist;
    }
#pragma unroll
    for (uint32_t u = 0; u < kChunk / kBlock; u++) {
      const int r = lo + u * kBlock + threadIdx.x < hi ? relax_edge(a, head[u], cand[u], next) : 0;
      if (r == 2) l_big.add(head[u], a.outdeg[head[u]], big_next, &nxt.n_big);
      wave_append(r == 1, head[u], l_q, &l_n, &l_end, q_next, &nxt.n);
    }
  }
  l_big.flush(a.outdeg, big_next, &nxt.n_big);
  const uint32_t staged = min(l_n, l_end);
  if (threadIdx.x == 0 && staged) l_at = atomicAdd(&nxt.n, (unsigned long long)staged);
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < staged; k += kBlock) q_next[l_at + k] = l_q[k];
  block_atomic_add(&cur.edges, edges);
}

// The far pile.  far[v] = 1 marks a far vertex; a split bins every far
// vertex by distance into steps of delta above the current threshold `base`
// (bin 0 also holds anything below base + delta, the last bin everything past
// the others) and stores the bin in far[v] as 2 + bin, so the scatter takes
// exactly the vertices the histogram counted.  Far vertices whose edges were
// relaxed with their current distance are dropped.  hist[kBins] = the smallest
// far distance's bits.
constexpr unsigned kBins = 128;

__global__ __launch_bounds__(kBlock) void k_far_hist(uint8_t* far, const uint32_t* dist,
                                                     const uint32_t* relaxed, uint64_t V,
                                                     float base, float delta, uint32_t* hist) {
  __shared__ uint32_t h[kBins];
  __shared__ uint32_t rm[kWaves];
  for (uint32_t i = threadIdx.x; i < kBins; i += kBlock) h[i] = 0;
  __syncthreads();
  uint32_t mn = ~0u;
  // four flags at a time (the array is padded to a multiple of four)
  const uint64_t words = (V + 3) / 4;
  for (uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x; i < words;
       i += uint64_t(gridDim.x) * kBlock) {
    uint32_t f = reinterpret_cast<const uint32_t*>(far)[i];
    if (!f) continue;
    for (uint32_t k = 0; k < 4; k++) {
      if (!((f >> (8 * k)) & 0xffu)) continue;
      const uint64_t v = i * 4 + k;
      const uint32_t d = dist[v];
      uint32_t mark = 0;
      if (d != relaxed[v]) {
        const float x = (__uint_as_float(d) - base) / delta;
        const uint32_t bin = x >= 1.0f ? uint32_t(min(x, float(kBins - 1))) : 0u;
        mark = 2 + bin;
        atomicAdd(&h[bin], 1u);
        mn = min(mn, d);
      }
      f = (f & ~(0xffu << (8 * k))) | mark << (8 * k);
    }
    reinterpret_cast<uint32_t*>(far)[i] = f;
  }
  for (int o = 32; o > 0; o >>= 1) mn = min(mn, uint32_t(__shfl_xor(int(mn), o, 64)));
  if ((threadIdx.x & 63) == 0) rm[threadIdx.x >> 6] = mn;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kBins; i += kBlock)
    if (h[i]) atomicAdd(&hist[i], h[i]);
  if (threadIdx.x == 0) {
    for (int i = 1; i < kWaves; i++) mn = min(mn, rm[i]);
    if (mn != ~0u) atomicMin(&hist[kBins], mn);
  }
}

__global__ void k_hist_zero(uint32_t* hist) {  // <<<1, kBins + 1>>>
  hist[threadIdx.x] = threadIdx.x < kBins ? 0u : ~0u;
}

// Take the far vertices of bins 0..k into the queue of `slot`.  A workgroup
// walks a contiguous range, stages what it takes and reserves queue entries
// when the stage may overflow and at its end.  Workgroup 0 also clears the
// histogram (read by the host) for the next split.
__global__ __launch_bounds__(kBlock) void k_far_scatter(uint8_t* far, uint64_t V, uint32_t k,
                                                        const uint32_t* outdeg, uint32_t* relaxed,
                                                        uint32_t* q, uint2* big, Slot* slot,
                                                        uint32_t* hist) {
  __shared__ uint32_t l_q[kStage];
  __shared__ uint32_t l_n;
  __shared__ BigStage l_big;
  __shared__ unsigned long long l_at;
  if (blockIdx.x == 0)
    for (uint32_t i = threadIdx.x; i <= kBins; i += kBlock) hist[i] = i < kBins ? 0u : ~0u;
  const uint64_t words = (V + 3) / 4;
  const uint64_t per = (words + gridDim.x - 1) / gridDim.x;
  const uint64_t w0 = uint64_t(blockIdx.x) * per, w1 = min(words, w0 + per);
  if (threadIdx.x == 0) {
    l_n = 0;
    l_big.clear();
  }
  __syncthreads();
  for (uint64_t b = w0; b < w1; b += kBlock) {
    const uint64_t i = b + threadIdx.x;
    uint32_t f = i < w1 ? reinterpret_cast<const uint32_t*>(far)[i] : 0u;
    if (f) {
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t m = (f >> (8 * j)) & 0xffu;
        if (m < 2 || m - 2 > k) continue;
        f &= ~(0xffu << (8 * j));
        const uint32_t v = uint32_t(i * 4 + j);
        const uint32_t d = outdeg[v];
        if (d > kBigRow) {
          relaxed[v] = kNotRelaxed;
          l_big.add(v, d, big, &slot->n_big);
        } else {
          l_q[atomicAdd(&l_n, 1u)] = v;  // at most 4 * kBlock per round
        }
      }
      reinterpret_cast<uint32_t*>(far)[i] = f;
    }
    __syncthreads();
    const uint32_t n = l_n;
    if (n > kStage - 4 * kBlock || b + kBlock >= w1) {  // uniform
      if (threadIdx.x == 0 && n) l_at = atomicAdd(&slot->n, (unsigned long long)n);
      __syncthreads();
      for (uint32_t t = threadIdx.x; t < n; t += kBlock) q[l_at + t] = l_q[t];
      __syncthreads();
      if (threadIdx.x == 0) l_n = 0;
    }
    __syncthreads();
  }
  l_big.flush(outdeg, big, &slot->n_big);
}
static_assert(kStage >= 8 * kBlock, "a round of the scatter fits beside what is staged");

// A queue too small for a round of its own rejoins the far pile.
__global__ void k_queue_to_far(const uint32_t* q, const uint2* big, const Slot* slot,
                               uint8_t* far) {
  const uint64_t n = slot->n, n_big = slot->n_big;
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n + n_big;
       i += uint64_t(gridDim.x) * blockDim.x)
    far[i < n ? q[i] : big[i - n].x] = 1;
}

// Sum of the edge weights (for the threshold step), FP64, fixed grid.
__global__ void k_weight_sum(const float* w, uint64_t n, double* out) {
  double t = 0;
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += uint64_t(gridDim.x) * blockDim.x)
    t += w[i];
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
  if ((threadIdx.x & 63) == 0) unsafeAtomicAdd(out, t);
}

__global__ void k_zero_f64(double* p) { *p = 0; }

// Reached vertices and the largest finite distance (fixed grid).
__global__ void k_sssp_summary(const uint32_t* dist, uint64_t V, unsigned long long* reached,
                               uint32_t* max_bits) {
  unsigned long long n = 0;
  uint32_t mx = 0;
  const uint32_t unreached = __float_as_uint(kUnreachedDist);
  for (uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < V;
       v += uint64_t(gridDim.x) * blockDim.x) {
    const uint32_t d = dist[v];
    if (d < unreached) {
      n++;
      mx = max(mx, d);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    n += __shfl_down(n, o, 64);
    mx = max(mx, __shfl_down(mx, o, 64));
  }
  __shared__ unsigned long long pn[4];
  __shared__ uint32_t pm[4];
  if ((threadIdx.x & 63) == 0) {
    pn[threadIdx.x >> 6] = n;
    pm[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < int(blockDim.x / 64); i++) {
      n += pn[i];
      mx = max(mx, pm[i]);
    }
    if (n) atomicAdd(reached, n);
    atomicMax(max_bits, mx);
  }
}

// Threshold step in thousandths of the mean edge weight: 5 from 2^24 vertices
// up, growing with the root of 2^24 / V below (to 160), since a phase of a
// small graph costs its launches and the round trip more than repeated
// relaxations.  ms by step (16 edges per vertex unless noted), the smallest
// tail queue V / 8: 2000 vertices, 8 edges 10: 1.51, 20: 1.06, 160: 0.57;
// 20000 10: 1.49, 20: 1.07, 145 (the rule) 0.73; 150000, 12 edges 10: 1.56,
// 20: 1.28, 53 (rule) 1.02; 2^20 5: 2.4, 20 (rule) 1.86, 40: 2.1; 2^24 2:
// 10.3, 5 (rule) 9.8, 10: 10.4 (before the staged big vertices).  V / 32 as
// the smallest tail queue: 0.71, 0.87, 1.25, 2.43 at those sizes.
double auto_delta_milli(uint64_t V) {
  return std::min(160.0, std::max(5.0, 5.0 * std::sqrt(double(1 << 24) / double(V))));
}

__global__ void k_sssp_summary_init(unsigned long long* reached, uint32_t* max_bits) {
  *reached = 0;
  *max_bits = 0;
}

}  // namespace

}  // namespace llgpu

extern "C" {

int ll_gpu_sssp(ll_gpu_graph* g, int level, int64_t root, float* dist_out, uint64_t* reached,
                double* max_dist, uint64_t* rounds) {
  if (!g) return LL_GPU_EINVAL;
  using namespace llgpu;
  try {
    LLG_HIP(hipSetDevice(g->ctx->device));
    ll_gpu_ctx* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint64_t V = g->V;
    LLG_CHECK(root >= 0 && uint64_t(root) < V, LL_GPU_EINVAL, "root outside [0, max_nodes)");
    const Csr& out = ensure_csr(g, LL_GPU_DIR_OUT, level);
    LLG_CHECK(out.w.p != nullptr, LL_GPU_ESTATE,
              "no edge weights for this snapshot (ll_gpu_graph_push_weights for every level)");
    // near/far threshold step in thousandths of the mean edge weight (0 = no
    // far pile: every improved vertex is queued)
    const long dm = ctx->options.count("sssp_delta_milli") ? ctx->options["sssp_delta_milli"] : -1;
    const double delta_milli = dm < 0 ? auto_delta_milli(V) : double(dm);
    const auto* rb = static_cast<const unsigned long long*>(ctx->readback);
    if (delta_milli > 0 && out.w_mean < 0) {
      DevBuf sum;
      sum.alloc(8, s);
      k_zero_f64<<<1, 1, 0, s>>>(sum.as<double>());
      k_weight_sum<<<std::min(grid_for(out.E, 256), 4u * unsigned(ctx->num_cus)), 256, 0, s>>>(
          out.w.as<float>(), out.E, sum.as<double>());
      LLG_HIP(hipMemcpyAsync(ctx->readback, sum.p, 8, hipMemcpyDeviceToHost, s));
      LLG_HIP(hipStreamSynchronize(s));
      double tot;
      std::memcpy(&tot, ctx->readback, 8);
      out.w_mean = out.E ? tot / double(out.E) : 0.0;
    }
    const double delta = delta_milli > 0 ? out.w_mean * delta_milli / 1000.0 : 0.0;
    const bool near_far = delta > 0;
    auto bits_of = [](double x) {
      const float f = float(std::min(x, double(kUnreachedDist)));
      uint32_t b;
      std::memcpy(&b, &f, 4);
      return b;
    };
    // a phase starts with at least min_queue vertices when the far pile has
    // them (smaller queues rejoin it); 0 = no merging
    const long mq_opt = ctx->options.count("sssp_min_queue") ? ctx->options["sssp_min_queue"] : -1;
    const uint64_t min_queue = mq_opt < 0 ? std::max<uint64_t>(V / kAutoMinQueueDiv, 1)
                                          : uint64_t(mq_opt);
    const uint32_t* outdeg = ensure_degrees(g, LL_GPU_DIR_OUT, level);
    DevBuf dist, stamp, far, relaxed, q[2], big[2], cnt, slots, hist;
    dist.alloc(V * 4, s);
    stamp.alloc(V * 4, s);
    far.alloc((V + 3) / 4 * 4, s);
    relaxed.alloc(V * 4, s);
    // chunks of the vertices past kBigRow: at most their edges / kChunk, one more each
    const uint64_t max_big = out.E / kChunk + out.E / kBigRow + 2;
    for (int i = 0; i < 2; i++) {
      q[i].alloc(V * 4, s);
      big[i].alloc(max_big * sizeof(uint2), s);
    }
    cnt.alloc(16, s);
    slots.alloc(kSlots * sizeof(Slot), s);
    hist.alloc((kBins + 1) * 4, s);
    RelaxArgs a{};
    a.qs = Queues{{q[0].as<uint32_t>(), q[1].as<uint32_t>()},
                  {big[0].as<uint2>(), big[1].as<uint2>()}};
    a.slots = slots.as<Slot>();
    a.ofs = out.ofs.as<uint64_t>();
    a.adj = out.adj.as<uint32_t>();
    a.w = out.w.as<float>();
    a.outdeg = outdeg;
    a.dist = dist.as<uint32_t>();
    a.stamp = stamp.as<int32_t>();
    a.far = far.as<uint8_t>();
    a.relaxed = relaxed.as<uint32_t>();
    a.E = out.E;
    a.min_queue = min_queue;
    a.near_far = near_far;
    k_sssp_init<<<grid_for((V + 3) / 4 * 4, 256), 256, 0, s>>>(
        a.dist, a.stamp, a.far, a.relaxed, V, uint32_t(root), outdeg, a.qs, a.slots,
        hist.as<uint32_t>(), kBins + 1);
    LLG_HIP(hipGetLastError());
    // a workgroup per 64 vertices, or per chunk of edges where the rows are long:
    // 64 vertices with 400000 edges took 2650 us a search on the one workgroup
    // of their vertices alone (343 now), 5000 with 5 M edges 2125 on 79 (994 now)
    const unsigned relax_grid = std::min(std::max(grid_for(V, 64), grid_for(out.E, kChunk)),
                                         4u * unsigned(ctx->num_cus));
    const unsigned far_grid = std::min(grid_for((V + 3) / 4, kBlock), 4u * unsigned(ctx->num_cus));
    uint64_t nrounds = 0;
    uint32_t r = 0;      // slot number of the next round
    double T = near_far ? delta : double(kUnreachedDist);
    a.t_bits = near_far ? bits_of(T) : ~0u;
    bool force = true;   // the root's queue, and a queue just taken from the far pile
    uint64_t work_done = 0;  // edges relaxed so far
    for (;;) {
      for (int k = 0; k < kBatch; k++) {
        TimedLaunch t(ctx, "k_relax");
        k_relax<<<relax_grid, kBlock, 0, s>>>(a, r + uint32_t(k), force && k == 0);
      }
      LLG_HIP(hipGetLastError());
      Slot h[kSlots];
      LLG_HIP(hipMemcpyAsync(ctx->readback, slots.p, sizeof(h), hipMemcpyDeviceToHost, s));
      LLG_HIP(hipStreamSynchronize(s));
      std::memcpy(h, ctx->readback, sizeof(h));
      int k = 0;
      for (; k < kBatch; k++) {
        const Slot& c = h[r % kSlots];
        if (!round_runs(c.n + c.n_big, c.before, out.E, min_queue, near_far, force)) break;
        work_done = c.before + c.edges;
        force = false;
        nrounds++;
        r++;
      }
      if (k == kBatch) continue;
      // the queue of slot r is empty, or too small for the tail
      if (!near_far) break;
      if (h[r % kSlots].n + h[r % kSlots].n_big > 0)
        k_queue_to_far<<<far_grid, kBlock, 0, s>>>(a.qs.q[r & 1], a.qs.big[r & 1],
                                                   a.slots + r % kSlots, a.far);
      // split: histogram of the far pile in steps of delta above T
      uint32_t c[kBins + 1];
      for (;;) {
        k_far_hist<<<far_grid, kBlock, 0, s>>>(a.far, a.dist, a.relaxed, V, float(T),
                                               float(delta), hist.as<uint32_t>());
        LLG_HIP(hipGetLastError());
        LLG_HIP(hipMemcpyAsync(ctx->readback, hist.p, sizeof(c), hipMemcpyDeviceToHost, s));
        LLG_HIP(hipStreamSynchronize(s));
        std::memcpy(c, ctx->readback, sizeof(c));
        uint64_t below_last = 0;
        for (unsigned i = 0; i + 1 < kBins; i++) below_last += c[i];
        if (below_last > 0 || c[kBins - 1] == 0) break;
        // everything lies past the histogram: restart it at the smallest distance
        float mf;
        std::memcpy(&mf, &c[kBins], 4);
        T = std::max(T, double(mf));
        k_hist_zero<<<1, kBins + 1, 0, s>>>(hist.as<uint32_t>());
      }
      // from the first non-empty bin on, enough bins to hold min_queue
      // vertices (in the tail only), never past the last non-empty one
      int first = -1, last = -1;
      for (unsigned i = 0; i < kBins; i++)
        if (c[i]) {
          if (first < 0) first = int(i);
          last = int(i);
        }
      if (first < 0) break;  // the far pile is empty: done
      const uint64_t want = work_done * 2 >= out.E ? min_queue : 0;
      uint32_t kb = uint32_t(first);
      uint64_t take = c[kb];
      while (int(kb) < last && take < want) take += c[++kb];
      r++;  // slot r may still hold the small queue; the next one is empty
      k_far_scatter<<<far_grid, kBlock, 0, s>>>(a.far, V, kb, outdeg, a.relaxed, a.qs.q[r & 1],
                                                a.qs.big[r & 1], a.slots + r % kSlots,
                                                hist.as<uint32_t>());
      LLG_HIP(hipGetLastError());
      T = kb + 1 < kBins ? T + double(kb + 1) * delta : double(kUnreachedDist);
      a.t_bits = bits_of(T);
      force = true;
    }
    k_sssp_summary_init<<<1, 1, 0, s>>>(cnt.as<unsigned long long>(),
                                        reinterpret_cast<uint32_t*>(cnt.as<unsigned long long>() + 1));
    k_sssp_summary<<<std::min(grid_for(V, 256), 4u * unsigned(ctx->num_cus)), 256, 0, s>>>(
        dist.as<uint32_t>(), V, cnt.as<unsigned long long>(),
        reinterpret_cast<uint32_t*>(cnt.as<unsigned long long>() + 1));
    LLG_HIP(hipGetLastError());
    if (dist_out) copy_to_host(ctx, dist_out, dist.p, V * 4);
    LLG_HIP(hipMemcpyAsync(ctx->readback, cnt.p, 16, hipMemcpyDeviceToHost, s));
    LLG_HIP(hipStreamSynchronize(s));
    if (reached) *reached = rb[0];
    if (max_dist) {
      const uint32_t bits = uint32_t(rb[1]);
      float f;
      std::memcpy(&f, &bits, 4);
      *max_dist = double(f);
    }
    if (rounds) *rounds = std::max<uint64_t>(nrounds, 1);  // a root without out-edges: one, empty
    return LL_GPU_OK;
  } catch (const Error& e) {
    g->ctx->err = e.msg;
    return e.code;
  } catch (...) {
    return llgpu::api_exception(g->ctx);
  }
}

}  // extern "C"
