// Betweenness centrality (tasks bc_adj / bc_random,
// benchmark/benchmarks/bc_adj.h, bc_random.h): Brandes from each source.
//
// Per source the direction-optimising BFS (bfs_core) gives the levels; then
//   forward, levels 1..D:  sigma[r] = sum of sigma[u] over in-neighbours u one
//                          level up (the reference adds sigma[v] to each
//                          down-neighbour atomically; the terms are the same),
//   reverse, levels D-1..1: delta[r] = sum over out-edges (r, w) to the next
//                          level, in iterator order, of
//                          sigma[r] / sigma[w] * (1 + delta[w]); BC[r] += delta[r]
//                          for r != source,
// in FP32 as the generated task code computes them.  Per source, each row
// block item gets a mask of the levels its rows are on, and per level a list
// of the items with a row there (long rows' pieces apart); a pass launches one
// workgroup per item of its level's list.  Within an item only the edges of
// rows on the level are loaded (an entry finds its row in a bitmap of row
// starts), their terms staged in LDS, and each row sums its own terms
// sequentially in edge order, so the reference's sums are reproduced bit for bit.  Long rows:
// the forward pass reduces pieces in parallel (path counts are whole numbers,
// exact in any order below 2^24) and a wave joins them; for the
// reverse pass their terms are computed piece-parallel into a buffer by edge
// position first, then one lane adds them in edge order while the other waves
// stage the next chunk.
#include <algorithm>
#include <cstring>

#include "ll_gpu_internal.h"
#include "rowblocks.h"

namespace llgpu {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kCap = 1024;  // row-block capacity of the path-count and dependency passes
constexpr uint32_t kMaxEdges = kCap + kCap / 2;
// Entries of one piece of a long row: one load per thread and entry slot, so a
// piece has no loop of dependent chunks (pieces of 8192 entries took 15.6 us a
// level for the reverse terms on 131101 vertices, a workgroup walking six
// chunks while most of the chip was idle; these take 5.2).
constexpr uint32_t kBcPiece = kMaxEdges;

// Per-vertex Brandes state in one 16-byte record, so visiting a neighbour is
// one load (level, path count and dependency together) instead of a level
// load followed by dependent path-count and dependency loads.
struct alignas(16) VState {
  int32_t lv;    // BFS level from the source, kUnreachedLevel when unreached
  float sigma;   // shortest-path count
  float delta;   // dependency
  float pad;
};

struct BcArgs {
  const RowItem* items;
  const uint64_t* ofs;
  const uint32_t* adj;
  VState* st;
  float* bc;
  float* part;      // partials of split rows, per item
  float* hub;       // reverse pass: terms of long rows, by out-edge position
  uint32_t source;
  int32_t d;        // the pass's level
};

constexpr uint32_t kPer = kMaxEdges / kBlock;  // entries per thread of a chunk
constexpr int32_t kUnreachedLevel = 2147483646;  // INT_MAX - 1, as the BFS marks it

// Term of edge (r, nb) whose far end is on level l: forward, sigma of an
// in-neighbour one level up; reverse, the reference's
// sigma[r] / sigma[w] * (1 + delta[w]) for an out-neighbour one level down.
template <bool kFwd>
__device__ inline float term(const BcArgs& a, const VState& w, float srow) {
  if (kFwd) return w.lv == a.d - 1 ? w.sigma : 0.0f;
  return w.lv == a.d + 1 ? srow / w.sigma * (1 + w.delta) : 0.0f;
}

// The state of neighbour nb, or an off-level placeholder for a skipped entry.
__device__ inline VState load_state(const BcArgs& a, bool need, uint32_t nb) {
  if (need) return a.st[nb];
  VState v;
  v.lv = -1;
  v.sigma = 0.0f;
  v.delta = 0.0f;
  v.pad = 0.0f;
  return v;
}

// The states of the neighbours of a long row's piece, entry k * kBlock +
// threadIdx.x in w[k]; past the piece the off-level placeholder.
__device__ inline void load_piece(const BcArgs& a, uint32_t r, uint32_t piece, VState (&w)[kPer]) {
  const uint64_t lo = a.ofs[r] + uint64_t(piece) * kBcPiece;
  const uint64_t hi = min(a.ofs[r + 1], lo + kBcPiece);
  uint32_t nb[kPer];
#pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    const uint64_t e = lo + k * kBlock + threadIdx.x;
    nb[k] = e < hi ? a.adj[e] : 0u;
  }
#pragma unroll
  for (uint32_t k = 0; k < kPer; k++)
    w[k] = load_state(a, lo + k * kBlock + threadIdx.x < hi, nb[k]);
}

template <bool kFwd>
__device__ inline void finish(const BcArgs& a, uint32_t r, float S) {
  if (kFwd) {
    a.st[r].sigma = S;
  } else {
    a.st[r].delta = S;
    if (r != a.source) a.bc[r] = a.bc[r] + S;
  }
}

// v[lo] + v[lo + 1] + ... in that order, one lane.  Each addition waits for
// the one before it; the LDS reads are kept kAhead terms ahead, so a row waits
// for its additions alone and not for an LDS read at each.
__device__ inline float ordered_sum(const float* v, uint32_t lo, uint32_t hi) {
  constexpr uint32_t kAhead = 8;
  float S = 0.0f;
  uint32_t j = lo;
  if (hi - lo >= 2 * kAhead) {
    float cur[kAhead];
#pragma unroll
    for (uint32_t k = 0; k < kAhead; k++) cur[k] = v[j + k];
    for (j += kAhead; j + kAhead <= hi; j += kAhead) {
      float nxt[kAhead];
#pragma unroll
      for (uint32_t k = 0; k < kAhead; k++) nxt[k] = v[j + k];
#pragma unroll
      for (uint32_t k = 0; k < kAhead; k++) S = S + cur[k];
#pragma unroll
      for (uint32_t k = 0; k < kAhead; k++) cur[k] = nxt[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < kAhead; k++) S = S + cur[k];
  }
  for (; j < hi; j++) S = S + v[j];
  return S;
}

__device__ inline uint64_t lane_u64(uint64_t x, uint32_t lane) {
  const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(x)), int(lane)));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(x >> 32)), int(lane)));
  return uint64_t(hi) << 32 | lo;
}

constexpr uint32_t kStartWords = kMaxEdges / 64;
static_assert(kStartWords <= 64 && kMaxEdges % 64 == 0, "a lane per word of row starts");

// One work item of a pass (all threads of the workgroup call it).
template <bool kFwd>
__device__ inline void bc_item(const BcArgs& a, uint64_t item) {
  __shared__ uint64_t rofs[kRowsPerItem + 1];
  __shared__ __align__(16) float vals[2][kMaxEdges];
  __shared__ float srow[kRowsPerItem];
  __shared__ uint8_t onf[kRowsPerItem];
  __shared__ unsigned long long starts[kStartWords];  // bit i: a row starts at entry i
  __shared__ uint8_t row_at[kMaxEdges];               // its row
  __shared__ float red[kBlock / 64];
  const RowItem it = a.items[item];
  if (it.npieces == 0) {
    const uint32_t nrows = it.row_end - it.row_begin;
    const uint32_t r = it.row_begin + threadIdx.x;
    const bool on = threadIdx.x < nrows && a.st[r].lv == a.d;
    if (!__syncthreads_or(on)) return;
    for (uint32_t i = threadIdx.x; i <= nrows; i += kBlock) rofs[i] = a.ofs[it.row_begin + i];
    if (threadIdx.x < kStartWords) starts[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t e0 = rofs[0];
    const uint32_t ne = uint32_t(rofs[nrows] - e0);
    const uint32_t lo = threadIdx.x < nrows ? uint32_t(rofs[threadIdx.x] - e0) : 0u;
    const uint32_t hi = threadIdx.x < nrows ? uint32_t(rofs[threadIdx.x + 1] - e0) : 0u;
    if (threadIdx.x < nrows) {
      onf[threadIdx.x] = on ? 1 : 0;
      srow[threadIdx.x] = on && !kFwd ? a.st[r].sigma : 0.0f;
      if (lo < hi) {
        atomicOr(&starts[lo >> 6], 1ull << (lo & 63));
        row_at[lo] = uint8_t(threadIdx.x);
      }
    }
    __syncthreads();
    // entries of rows off the level are neither loaded nor staged; all
    // neighbour IDs first, then their states, so the loads overlap
    uint32_t nb[kPer], rr[kPer];
    VState w[kPer];
    bool need[kPer];
    // an entry's row starts at the last set bit up to it: in its own word of
    // 64, which is the wave's, or in the nearest non-zero one before.  Passes of
    // four sources, ms at 2^17 / 2^24 vertices: 0.71 / 36.2; a search of the
    // offsets per entry (eight dependent LDS reads) 0.77 / 37.8, labels written
    // entry by entry by the rows 0.80 / 35.4
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint64_t mine = lane < kStartWords ? starts[lane] : 0ull;
    const uint64_t used = __ballot(mine != 0);
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t w = k * (kBlock / 64) + wave;
      const uint64_t before = used & ((uint64_t(1) << w) - 1);
      uint32_t p = 0;
      if (before) {
        const uint32_t q = 63 - uint32_t(__clzll((long long)before));
        p = q * 64 + 63 - uint32_t(__clzll((long long)lane_u64(mine, q)));
      }
      const uint64_t m = lane_u64(mine, w) & (~uint64_t(0) >> (63 - lane));
      if (m) p = w * 64 + 63 - uint32_t(__clzll((long long)m));
      rr[k] = row_at[p];
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t i = k * kBlock + threadIdx.x;
      need[k] = i < ne && onf[rr[k]];
      nb[k] = need[k] ? a.adj[e0 + i] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) w[k] = load_state(a, need[k], nb[k]);
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++)
      if (need[k]) vals[0][k * kBlock + threadIdx.x] = term<kFwd>(a, w[k], srow[rr[k]]);
    __syncthreads();
    if (on) {
      // the row's terms in edge order, as the reference's loop adds them
      finish<kFwd>(a, r, ordered_sum(vals[0], lo, hi));
    }
  } else if (!kFwd) {
    // Reverse pass, long row: k_bc_hub_terms has written the row's terms
    // (all pieces in parallel); the first piece's workgroup adds them in edge
    // order.  Waves 1-3 copy chunk c into LDS while lane 0 of wave 0 adds
    // chunk c-1, so the dependency is the reference's sequential sum.
    const uint32_t r = it.row_begin;
    if (it.piece != 0 || a.st[r].lv != a.d) return;  // uniform over the workgroup
    const uint64_t rb = a.ofs[r], re = a.ofs[r + 1];
    const uint32_t nch = uint32_t((re - rb + kMaxEdges - 1) / kMaxEdges);
    constexpr uint32_t kGather = kBlock - 64;
    constexpr uint32_t kPerG = kMaxEdges / kGather;
    static_assert(kMaxEdges % kGather == 0 && kMaxEdges % 32 == 0, "chunk layout");
    float S = 0.0f;
    for (uint32_t c = 0; c <= nch; c++) {
      if (threadIdx.x >= 64) {
        if (c < nch) {
          // entries past the row add +0: the sum is >= +0, so they change nothing
          const uint64_t c0 = rb + uint64_t(c) * kMaxEdges;
          const uint32_t t = threadIdx.x - 64;
          float* v = vals[c & 1];
          float x[kPerG];
#pragma unroll
          for (uint32_t k = 0; k < kPerG; k++) {
            const uint64_t e = c0 + k * kGather + t;
            x[k] = e < re ? a.hub[e] : 0.0f;
          }
#pragma unroll
          for (uint32_t k = 0; k < kPerG; k++) v[k * kGather + t] = x[k];
        }
      } else if (c > 0 && threadIdx.x == 0) {
        // the chunk in edge order; LDS reads of the next 32 terms are issued
        // before the additions of the current 32
        const float4* v4 = reinterpret_cast<const float4*>(vals[(c - 1) & 1]);
        constexpr uint32_t kG = 8, kGroups = kMaxEdges / 4 / kG;
        float4 cur[kG];
#pragma unroll
        for (uint32_t k = 0; k < kG; k++) cur[k] = v4[k];
        for (uint32_t g = 0; g < kGroups; g++) {
          float4 nxt[kG];
          if (g + 1 < kGroups) {
#pragma unroll
            for (uint32_t k = 0; k < kG; k++) nxt[k] = v4[(g + 1) * kG + k];
          }
#pragma unroll
          for (uint32_t k = 0; k < kG; k++) {
            S = S + cur[k].x;
            S = S + cur[k].y;
            S = S + cur[k].z;
            S = S + cur[k].w;
          }
#pragma unroll
          for (uint32_t k = 0; k < kG; k++) cur[k] = nxt[k];
        }
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) finish<false>(a, r, S);
  } else {
    // Forward pass, long row: path counts are whole numbers, exact in any
    // order below 2^24; pieces reduce in parallel, k_bc_fixup joins them.
    const uint32_t r = it.row_begin;
    if (a.st[r].lv != a.d) return;  // uniform over the workgroup
    VState w[kPer];
    load_piece(a, r, it.piece, w);
    float S = 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) S = S + term<true>(a, w[k], 0.0f);
    for (int o = 32; o > 0; o >>= 1) S = S + __shfl_down(S, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = S;
    __syncthreads();
    if (threadIdx.x == 0) {
      float t = red[0];
      for (int i = 1; i < kBlock / 64; i++) t = t + red[i];
      if (it.npieces == 1) finish<true>(a, r, t);
      else a.part[item] = t;
    }
  }
}

// A level's items: long rows' pieces from the front of its list, the other
// items from the back, so one launch fills both and each part's count bounds
// the launch that reads it.
struct LevelList {
  const uint32_t* list;
  uint32_t n;        // capacity (items of the direction)
  uint32_t nlong;    // entries at the front
  __device__ uint32_t at(uint32_t i) const {
    return i < nlong ? list[i] : list[n - 1 - (i - nlong)];
  }
};

// A pass: one workgroup per item of the level's list.
template <bool kFwd>
__global__ __launch_bounds__(kBlock) void k_bc_pass(BcArgs a, LevelList l) {
  bc_item<kFwd>(a, l.at(blockIdx.x));
}

// Reverse pass, long rows on the level: each piece writes its edges' terms
// to a.hub at their out-edge positions.
__global__ __launch_bounds__(kBlock) void k_bc_hub_terms(BcArgs a, LevelList l) {
  const RowItem it = a.items[l.list[blockIdx.x]];
  const uint32_t r = it.row_begin;
  if (a.st[r].lv != a.d) return;
  const uint64_t lo = a.ofs[r] + uint64_t(it.piece) * kBcPiece;
  const uint64_t hi = min(a.ofs[r + 1], lo + kBcPiece);
  const float sr = a.st[r].sigma;
  VState w[kPer];
  load_piece(a, r, it.piece, w);
#pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    const uint64_t e = lo + k * kBlock + threadIdx.x;
    if (e < hi) a.hub[e] = term<false>(a, w[k], sr);
  }
}

// Forward pass, rows split over several pieces: combine the partials, one
// wave per listed piece (the first piece of a row joins them); launched for
// the levels with long rows only, over their pieces.
__global__ __launch_bounds__(kBlock) void k_bc_fixup(BcArgs a, LevelList l) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (i >= l.nlong) return;
  const uint32_t item = l.list[i];
  const RowItem it = a.items[item];
  if (it.npieces <= 1 || it.piece != 0 || a.st[it.row_begin].lv != a.d) return;
  float t = 0.0f;
  for (uint32_t p = lane; p < it.npieces; p += 64) t = t + a.part[item + p];
  for (int o = 32; o > 0; o >>= 1) t = t + __shfl_down(t, o, 64);
  if (lane == 0) finish<true>(a, it.row_begin, t);
}

// One direction's items and what a source's lists need of them.
struct LevelItems {
  const RowItem* items;
  uint64_t n;
  uint32_t* mask;   // per item, the levels its rows are on (bit min(level, 31))
  uint32_t* list;   // 32 x n
  uint32_t* nlong;  // 32 counts: long rows' pieces
  uint32_t* nshort; // 32 counts: the other items
};

// Start of a source, one launch (a source's state, masks and lists in ten
// launches cost about 80 us of a 500 us source, most of it between them; two
// launches take about 12): the state from the BFS levels (one path to
// the source, no dependency), the level masks of both directions' items (one
// wave per item), the list counts cleared.
__global__ __launch_bounds__(kBlock) void k_bc_source(const int32_t* lv, VState* st, uint64_t V,
                                                      uint32_t src, LevelItems in, LevelItems out,
                                                      uint32_t* cnt) {
  const uint64_t t0 = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t nt = uint64_t(gridDim.x) * blockDim.x;
  if (blockIdx.x == 0 && threadIdx.x < 128) cnt[threadIdx.x] = 0;
  for (uint64_t v = t0; v < V; v += nt) {
    VState x;
    x.lv = lv[v];
    x.sigma = v == src ? 1.0f : 0.0f;
    x.delta = 0.0f;
    x.pad = 0.0f;
    st[v] = x;
  }
  const uint32_t lane = threadIdx.x & 63;
  for (uint64_t i = t0 >> 6; i < in.n + out.n; i += nt >> 6) {
    const bool first = i < in.n;
    const uint64_t j = first ? i : i - in.n;
    const RowItem it = first ? in.items[j] : out.items[j];
    const uint32_t re = it.npieces == 0 ? it.row_end : it.row_begin + 1;
    uint32_t m = 0;
    for (uint32_t r = it.row_begin + lane; r < re; r += 64) {
      const int32_t l = lv[r];
      if (l != kUnreachedLevel) m |= 1u << min(l, 31);
    }
    for (int o = 32; o > 0; o >>= 1) m |= __shfl_xor(m, o, 64);
    if (lane == 0) (first ? in.mask : out.mask)[j] = m;
  }
}

// Level lists of both directions, one launch: the first `in_blocks` workgroups
// list the in-direction's items, the others the out-direction's.  An item is
// listed on every level it has a row on (levels >= 31 share list 31).
// Positions come from one global atomic per workgroup, level and kind (the
// waves take their slots in the workgroup's share from an LDS counter).
constexpr unsigned kListBlock = 1024;  // workgroup of k_level_lists

__global__ __launch_bounds__(kListBlock) void k_level_lists(LevelItems in, LevelItems out,
                                                            uint32_t in_blocks) {
  constexpr uint32_t kWaves = kListBlock / 64;
  __shared__ uint32_t bcount[2][32], bbase[2][32], woff[2][kWaves][32];
  const bool first = blockIdx.x < in_blocks;
  const LevelItems& d = first ? in : out;
  const uint64_t i =
      uint64_t(first ? blockIdx.x : blockIdx.x - in_blocks) * kListBlock + threadIdx.x;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t mk[2] = {0, 0}, wm[2];
  if (i < d.n) {
    const uint32_t m = d.mask[i];
    const bool is_long = d.items[i].npieces != 0;
    mk[0] = is_long ? m : 0;
    mk[1] = is_long ? 0 : m;
  }
  if (threadIdx.x < 64) bcount[threadIdx.x >> 5][threadIdx.x & 31] = 0;
  __syncthreads();
  // the wave's slot in the workgroup's share of each level's list
#pragma unroll
  for (int k = 0; k < 2; k++) {
    wm[k] = mk[k];
    for (int o = 32; o > 0; o >>= 1) wm[k] |= __shfl_xor(wm[k], o, 64);
    for (uint32_t x = wm[k]; x; x &= x - 1) {
      const uint32_t l = uint32_t(__builtin_ctz(x));
      const uint64_t b = __ballot((mk[k] >> l) & 1u);
      if (lane == uint32_t(__builtin_ctzll(b)))
        woff[k][wave][l] = atomicAdd(&bcount[k][l], uint32_t(__popcll(b)));
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint32_t k = threadIdx.x >> 5, l = threadIdx.x & 31;
    if (bcount[k][l]) bbase[k][l] = atomicAdd(&(k ? d.nshort : d.nlong)[l], bcount[k][l]);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; k++) {
    for (uint32_t x = wm[k]; x; x &= x - 1) {
      const uint32_t l = uint32_t(__builtin_ctz(x));
      const uint64_t b = __ballot((mk[k] >> l) & 1u);
      if ((mk[k] >> l) & 1u) {
        const uint64_t below = lane ? (b & (~0ull >> (64 - lane))) : 0ull;
        const uint64_t p = bbase[k][l] + woff[k][wave][l] + uint32_t(__popcll(below));
        d.list[uint64_t(l) * d.n + (k ? d.n - 1 - p : p)] = uint32_t(i);
      }
    }
  }
}

__global__ void k_fill_f32(float* p, uint64_t n, float x) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = x;
}

}  // namespace

}  // namespace llgpu

extern "C" {

int ll_gpu_bc(ll_gpu_graph* g, int level, const int64_t* sources, int64_t n, float* bc_out) {
  if (!g) return LL_GPU_EINVAL;
  using namespace llgpu;
  try {
    LLG_HIP(hipSetDevice(g->ctx->device));
    ll_gpu_ctx* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint64_t V = g->V;
    const int64_t ns = sources ? n : int64_t(V);
    LLG_CHECK(!sources || n >= 0, LL_GPU_EINVAL, "bad source count");
    for (int64_t i = 0; sources && i < n; i++)
      LLG_CHECK(sources[i] >= 0 && uint64_t(sources[i]) < V, LL_GPU_EINVAL,
                "source outside [0, max_nodes)");
    const BfsPrepared bfs = bfs_prepare(g, level);
    const Csr& out = *bfs.out;
    const Csr& in = *bfs.in;
    const RowBlocks& in_rb = ensure_rowblocks(g, LL_GPU_DIR_IN, level, kCap, kBcPiece);
    const RowBlocks& out_rb = ensure_rowblocks(g, LL_GPU_DIR_OUT, level, kCap, kBcPiece);
    const uint64_t nin = std::max<uint64_t>(in_rb.n, 1), nout = std::max<uint64_t>(out_rb.n, 1);
    DevBuf lv, bfs_ws, st, bc, part, in_mask, out_mask, in_list, out_list, cnt, hub;
    lv.alloc(V * 4, s);
    bfs_ws.alloc(bfs_work_bytes(V), s);
    st.alloc(V * sizeof(VState), s);
    bc.alloc(V * 4, s);
    part.alloc(std::max(nin, nout) * 4, s);
    in_mask.alloc(nin * 4, s);
    out_mask.alloc(nout * 4, s);
    in_list.alloc(32 * nin * 4, s);
    out_list.alloc(32 * nout * 4, s);
    cnt.alloc(4 * 32 * 4, s);  // in and out, each long rows' pieces and others
    k_fill_f32<<<grid_for(V, 256), 256, 0, s>>>(bc.as<float>(), V, 0.0f);
    uint32_t* c = cnt.as<uint32_t>();
    const LevelItems li{in_rb.items.as<RowItem>(), in_rb.n, in_mask.as<uint32_t>(),
                        in_list.as<uint32_t>(), c, c + 32};
    const LevelItems lo{out_rb.items.as<RowItem>(), out_rb.n, out_mask.as<uint32_t>(),
                        out_list.as<uint32_t>(), c + 64, c + 96};
    const unsigned source_grid = unsigned(std::min<uint64_t>(
        grid_for((li.n + lo.n) * 64, kBlock), 8u * unsigned(ctx->num_cus)));
    const unsigned in_blocks = unsigned(grid_for(li.n, kListBlock));
    const unsigned out_blocks = unsigned(grid_for(lo.n, kListBlock));
    for (int64_t i = 0; i < ns; i++) {
      const uint32_t src = uint32_t(sources ? sources[i] : i);
      // the search's step count bounds the deepest level (a last step may
      // find nothing): a level without rows has an empty list
      const int32_t D = bfs_single_ws(g, bfs, src, bfs_ws.p, lv.as<int32_t>(), true).levels;
      k_bc_source<<<source_grid, kBlock, 0, s>>>(lv.as<int32_t>(), st.as<VState>(), V, src, li,
                                                 lo, c);
      k_level_lists<<<in_blocks + out_blocks, kListBlock, 0, s>>>(li, lo, in_blocks);
      LLG_HIP(hipGetLastError());
      LLG_HIP(hipMemcpyAsync(ctx->readback, c, 4 * 32 * 4, hipMemcpyDeviceToHost, s));
      LLG_HIP(hipStreamSynchronize(s));
      uint32_t h[4][32];
      std::memcpy(h, ctx->readback, sizeof(h));
      // long rows' terms by out-edge position, allocated when a source first
      // reaches one
      for (int l = 0; l < 32 && !hub.p; l++)
        if (h[2][l]) hub.alloc(out.E * 4, s);
      BcArgs a;
      a.st = st.as<VState>();
      a.bc = bc.as<float>();
      a.part = part.as<float>();
      a.hub = hub.as<float>();
      a.source = src;
      a.items = in_rb.items.as<RowItem>();
      a.ofs = in.ofs.as<uint64_t>();
      a.adj = in.adj.as<uint32_t>();
      for (int32_t d = 1; d <= D; d++) {
        const uint32_t l = uint32_t(std::min(d, 31));
        const LevelList lst{li.list + l * li.n, uint32_t(li.n), h[0][l]};
        if (h[0][l] + h[1][l] == 0) continue;
        a.d = d;
        {
          TimedLaunch t(ctx, "k_bc_pass");
          k_bc_pass<true><<<h[0][l] + h[1][l], kBlock, 0, s>>>(a, lst);
        }
        if (h[0][l] && in_rb.nsplit)
          k_bc_fixup<<<grid_for(h[0][l], kBlock / 64), kBlock, 0, s>>>(a, lst);
      }
      a.items = out_rb.items.as<RowItem>();
      a.ofs = out.ofs.as<uint64_t>();
      a.adj = out.adj.as<uint32_t>();
      // level 0 is the source alone, whose dependency is never added
      for (int32_t d = D - 1; d >= 1; d--) {
        const uint32_t l = uint32_t(std::min(d, 31));
        const LevelList lst{lo.list + l * lo.n, uint32_t(lo.n), h[2][l]};
        if (h[2][l] + h[3][l] == 0) continue;
        a.d = d;
        if (h[2][l]) {
          TimedLaunch t(ctx, "k_bc_hub_terms");
          k_bc_hub_terms<<<h[2][l], kBlock, 0, s>>>(a, lst);
        }
        TimedLaunch t(ctx, "k_bc_pass");
        k_bc_pass<false><<<h[2][l] + h[3][l], kBlock, 0, s>>>(a, lst);
      }
      LLG_HIP(hipGetLastError());
    }
    if (bc_out) copy_to_host(ctx, bc_out, bc.p, V * 4);
    LLG_HIP(hipStreamSynchronize(s));
    return LL_GPU_OK;
  } catch (const Error& e) {
    g->ctx->err = e.msg;
    return e.code;
  } catch (...) {
    return llgpu::api_exception(g->ctx);
  }
}

}  // extern "C"
