// Weighted PageRank and its adjoint over the snapshot (no reference
// counterpart; the forward is the weighted form of ll_b_pagerank_pull_ext,
// pagerank.h:98-182, the adjoint is the transposed sweep, i.e. the push
// pattern of ll_b_pagerank_push_ext, pagerank.h:217-360, computed as a pull
// over out-edges so it needs no atomics).
//
// Weights w[e] are given per live out-edge in the snapshot's out-edge order.
//   forward:  r0 = p,  r' = (1-d) p + d W^T r            (pull over in-edges)
//   adjoint:  l0 = g,  l' = g + d W l                     (pull over out-edges)
//             dL/dw[e=(u,v)] = d r[u] l[v],  dL/dp = (1-d) l
// Either direction is one sweep kernel over a CSR, with a permutation where
// entries are not in out-edge order that brings w into theirs once per call;
// sums are FP64.  Large skewed graphs number rows and columns by descending
// degree, so that hot columns sit in an LDS table (kTableV, kHotShare).  Bytes
// per sweep: 8 per edge (column, weight) + 20 per vertex (row offset, x, base,
// y), and a gather of x per edge that misses the table.
#include "ll_gpu_internal.h"
#include "rowblocks.h"

namespace llgpu {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kGradCap = 1024;          // row blocks of the edge gradient
constexpr int kSpBlock = 1024;
constexpr uint32_t kCap = 512;               // stream-item capacity of the row blocks
constexpr uint32_t kEnt = kCap + kCap / 2;   // entries of an item, at most
constexpr uint32_t kWPiece = kEnt;           // entries of one piece of a long row
constexpr uint32_t kHot = 24576;             // entries of x kept in LDS
constexpr uint32_t kThreadRow = 32;          // longest row a single lane sums
constexpr uint32_t kRowLanes = 8;            // lanes of a longer one

// One item of a sweep: a wave's work.
struct SpItem {
  uint32_t row;   // first row; of a split row's piece, its place in `part`
  uint32_t meta;  // entries | rows << 12 | kind << 24
  uint64_t e0;    // first entry
};
static_assert(sizeof(SpItem) == 16 && kEnt < 4096 && kRowsPerItem < 4096, "SpItem fields");
constexpr uint32_t kRun = 0, kOneRow = 1, kSplit = 2;
// A row cut into several pieces.
struct SpSplit {
  uint32_t row, part, pieces;
};

struct SpArgs {
  const SpItem* items;
  uint64_t nitems;
  const SpSplit* splits;
  uint32_t nsplits;
  const uint64_t* ofs;
  const uint32_t* col;
  const float* val;
  const float* x;
  uint64_t nx;
  const float* base;      // y = base_scale * base + d * (matrix * x)
  float base_scale, d;
  float* y;
  double* part;           // sums of the pieces of split rows
};

// Make a wave's LDS writes visible to its other lanes before they read them.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One sweep: a fixed grid of waves taking items in turn, each wave on its own
// (no workgroup barrier past the table's).
//
// Bound by load latency (with the table, waves wait for 61% of their cycles
// and the vector units issue for 27%): a CU keeps few enough gathers of x from
// L2 in flight that they, not the 8 bytes streamed per edge, set the pace.
// kTable: rows and columns are numbered by descending degree, the first kHot
// entries of x, which take most of the gathers of a skewed graph, are copied
// to LDS once per workgroup, and the others lie close together.  Everything
// else an item needs (entries, row offsets, base) is loaded while the wave's
// item before it is summed.  Without: workgroups of four waves, sixteen of
// them where LDS allowed one.
//
// A run of short rows: the products are staged in LDS and summed in FP64, rows
// of up to kThreadRow entries by a lane each, longer ones by kRowLanes lanes
// each.  A long row is cut into pieces, a wave each; k_wspmv_split adds them
// in a fixed order, so the result does not depend on the schedule.
//
// R-MAT 2^20 vertices, 16.8 M edges, with the table: 69 us a sweep (2.0 TB/s of
// streamed bytes); 106 without, 120 with one workgroup per item, 83 with the
// columns but not the rows renumbered (y and base then scattered), 196 with
// workgroup-wide items and the same LDS table.  Lanes per row 8 / rows of
// 32 by a lane: 7.94 ms for 100 sweeps, 16 / 16: 8.22, 8 / 8: 8.14; a table of
// 8192 entries: 8.87.
template <bool kTable>
__global__ __launch_bounds__(kTable ? kSpBlock : kBlock) void k_wspmv(SpArgs a) {
  constexpr uint32_t kPer = kEnt / 64;
  constexpr uint32_t kThreads = kTable ? kSpBlock : kBlock;
  constexpr uint32_t kWaves = kThreads / 64;
  constexpr uint32_t kRowPer = kRowsPerItem / 64;
  __shared__ float hot[kTable ? kHot : 1];
  __shared__ float s_vals[kWaves][kEnt];
  __shared__ uint16_t s_rofs[kWaves][kRowsPerItem + 1];
  __shared__ uint16_t s_list[kWaves][kEnt / kThreadRow];  // rows left to lane groups
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  float* vals = s_vals[wave];
  uint16_t* rofs = s_rofs[wave];
  uint16_t* list = s_list[wave];
  const uint64_t stride = uint64_t(gridDim.x) * kWaves;
  uint64_t i = uint64_t(blockIdx.x) * kWaves + wave;
  uint32_t idx[kPer], ro[kRowPer];
  float wv[kPer], rb[kRowPer];
  auto load = [&](const SpItem& it) {
    const uint32_t ne = it.meta & 0xfffu, nrows = (it.meta >> 12) & 0xfffu;
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t q = lane + 64 * k;
      idx[k] = q < ne ? a.col[it.e0 + q] : 0u;
      wv[k] = q < ne ? a.val[it.e0 + q] : 0.f;
    }
#pragma unroll
    for (uint32_t k = 0; k < kRowPer; k++) {
      const uint32_t q = lane + 64 * k;
      ro[k] = q < nrows ? uint32_t(a.ofs[it.row + q] - it.e0) : 0u;
      rb[k] = q < nrows ? a.base[it.row + q] : 0.f;
    }
  };
  auto fetch = [&](uint64_t q) { return q < a.nitems ? a.items[q] : SpItem{0u, 0u, 0ull}; };
  auto uniform = [](SpItem t) {
    t.row = uint32_t(__builtin_amdgcn_readfirstlane(int(t.row)));
    t.meta = uint32_t(__builtin_amdgcn_readfirstlane(int(t.meta)));
    const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(t.e0))));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(t.e0 >> 32))));
    t.e0 = uint64_t(hi) << 32 | lo;
    return t;
  };
  SpItem cur = uniform(fetch(i)), nxt = uniform(fetch(i + stride));
  load(cur);
  if (kTable) {
    for (uint32_t q = threadIdx.x; q < kHot; q += kThreads) hot[q] = q < a.nx ? a.x[q] : 0.f;
    __syncthreads();
  }
  for (; i < a.nitems; i += stride) {
    const uint32_t ne = cur.meta & 0xfffu, nrows = (cur.meta >> 12) & 0xfffu;
    const uint32_t kind = cur.meta >> 24;
    const SpItem after = fetch(i + 2 * stride);
    float xv[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) xv[k] = !kTable || idx[k] >= kHot ? a.x[idx[k]] : 0.f;
    if (kTable) {
#pragma unroll
      for (uint32_t k = 0; k < kPer; k++)
        if (idx[k] < kHot) xv[k] = hot[idx[k]];
    }
    if (kind == kRun) {
#pragma unroll
      for (uint32_t k = 0; k < kPer; k++)
        if (lane + 64 * k < ne) vals[lane + 64 * k] = wv[k] * xv[k];
      float yb[kRowPer];
#pragma unroll
      for (uint32_t k = 0; k < kRowPer; k++) {
        if (lane + 64 * k < nrows) rofs[lane + 64 * k] = uint16_t(ro[k]);
        yb[k] = a.base_scale * rb[k];
      }
      if (lane == 0) rofs[nrows] = uint16_t(ne);
      wave_sync();
      load(nxt);
      // rows past kThreadRow entries, their sums left at their first product
      uint32_t lo[kRowPer], n[kRowPer], nl = 0;
#pragma unroll
      for (uint32_t k = 0; k < kRowPer; k++) {
        const uint32_t r = lane + 64 * k;
        lo[k] = n[k] = 0;
        if (r < nrows) {
          lo[k] = rofs[r];
          n[k] = rofs[r + 1] - lo[k];
        }
        const uint64_t m = __ballot(n[k] > kThreadRow);
        if (n[k] > kThreadRow)
          list[nl + uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1)))] = uint16_t(r);
        nl += uint32_t(__popcll(m));
      }
      wave_sync();
      for (uint32_t q0 = 0; q0 < nl; q0 += 64 / kRowLanes) {
        const uint32_t q = q0 + lane / kRowLanes;
        double S = 0;
        uint32_t first = 0;
        if (q < nl) {
          const uint32_t r = list[q], hi = rofs[r + 1];
          first = rofs[r];
#pragma unroll 4
          for (uint32_t j = first + lane % kRowLanes; j < hi; j += kRowLanes)
            S += double(vals[j]);
        }
        for (int o = kRowLanes / 2; o > 0; o >>= 1) S += __shfl_down(S, o, kRowLanes);
        if (q < nl && lane % kRowLanes == 0) vals[first] = float(S);
      }
      wave_sync();
#pragma unroll
      for (uint32_t k = 0; k < kRowPer; k++) {
        if (64 * k >= nrows) break;
        double S = 0;
        const uint32_t hi = lo[k] + (n[k] > kThreadRow ? 1u : n[k]);
#pragma unroll 4
        for (uint32_t j = lo[k]; j < hi; j++) S += double(vals[j]);
        if (lane + 64 * k < nrows) a.y[cur.row + lane + 64 * k] = yb[k] + a.d * float(S);
      }
      wave_sync();  // vals, rofs and list are rewritten for the next item
    } else {
      double S = 0;
#pragma unroll
      for (uint32_t k = 0; k < kPer; k++)
        if (lane + 64 * k < ne) S += double(wv[k] * xv[k]);
      load(nxt);
      for (int o = 32; o > 0; o >>= 1) S += __shfl_down(S, o, 64);
      if (lane == 0) {
        if (kind == kOneRow) a.y[cur.row] = a.base_scale * a.base[cur.row] + a.d * float(S);
        else a.part[cur.row] = S;
      }
    }
    cur = nxt;
    nxt = uniform(after);
  }
}

// Split rows: kSplitLanes lanes add a row's pieces, always in the same order.
constexpr uint32_t kSplitLanes = 16;
__global__ void k_wspmv_split(SpArgs a) {
  const uint32_t q = (blockIdx.x * blockDim.x + threadIdx.x) / kSplitLanes;
  const uint32_t lane = threadIdx.x % kSplitLanes;
  if (q >= a.nsplits) return;  // whole lane groups
  const SpSplit t = a.splits[q];
  double S = 0;
#pragma unroll 4
  for (uint32_t p = lane; p < t.pieces; p += kSplitLanes) S += a.part[t.part + p];
  for (int o = kSplitLanes / 2; o > 0; o >>= 1) S += __shfl_down(S, o, kSplitLanes);
  if (lane == 0) a.y[t.row] = a.base_scale * a.base[t.row] + a.d * float(S);
}

// Sweep items and split rows (counted in *cnt) of row blocks.
__global__ void k_sweep_items(const RowItem* items, const uint32_t* pslot, uint64_t n,
                              const uint64_t* ofs, SpItem* out, SpSplit* splits, uint32_t* cnt) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const RowItem it = items[i];
  uint64_t e0 = ofs[it.row_begin], e1 = ofs[it.row_end];
  SpItem t;
  t.row = it.row_begin;
  uint32_t kind = kRun, nrows = it.row_end - it.row_begin;
  if (it.npieces) {
    e0 += uint64_t(it.piece) * kWPiece;
    e1 = min(e1, e0 + kWPiece);
    kind = kOneRow;
    nrows = 0;
    if (it.npieces > 1) {
      kind = kSplit;
      t.row = pslot[i];
      if (it.piece == 0) splits[atomicAdd(cnt, 1u)] = SpSplit{it.row_begin, t.row, it.npieces};
    }
  }
  t.meta = uint32_t(e1 - e0) | nrows << 12 | kind << 24;
  t.e0 = e0;
  out[i] = t;
}

__global__ void k_zero_u32(uint32_t* p) { *p = 0; }

// Tail of every out-edge, a wave per row.
__global__ void k_edge_tails(const uint64_t* ofs, uint64_t V, uint32_t* tail) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t nw = uint64_t(gridDim.x) * (blockDim.x / 64);
  for (uint64_t u = uint64_t(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6); u < V; u += nw)
    for (uint64_t e = ofs[u] + lane, end = ofs[u + 1]; e < end; e += 64) tail[e] = uint32_t(u);
}

// In-degrees counted over the out-edges' heads.
__global__ void k_count_heads(const uint32_t* adj, uint64_t n, uint32_t* deg) {
  const uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e < n) atomicAdd(&deg[adj[e]], 1u);
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Edge e's row (its number in `slot` when given) as the sort key, e as the value.
__global__ void k_row_keys(const uint32_t* row, const uint32_t* slot, uint32_t* key,
                           uint32_t* pos, uint64_t n) {
  const uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= n) return;
  key[e] = slot ? slot[row[e]] : row[e];
  pos[e] = uint32_t(e);
}

// Row offsets of the sorted rows, a thread per row (rows without entries come
// in one run, the vertices of degree 0: filled by the entry that follows them,
// 2 M took 114 ms of one thread).
__global__ void k_row_offsets(const uint32_t* rows, uint64_t m, uint64_t V, uint64_t* ofs) {
  const uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (x > V) return;
  uint64_t lo = 0, hi = m;  // first entry of a row >= x
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (rows[mid] < x) lo = mid + 1;
    else hi = mid;
  }
  ofs[x] = lo;
}

// col[i] = column of edge perm[i] (its number in `slot` when given).
__global__ void k_columns(const uint32_t* perm, const uint32_t* column, const uint32_t* slot,
                          uint32_t* col, uint64_t n) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t c = column[perm[i]];
  col[i] = slot ? slot[c] : c;
}

// Length of every row by its number.
__global__ void k_row_lengths(const uint64_t* ofs, const uint32_t* slot, uint64_t V,
                              uint32_t* len) {
  const uint64_t u = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (u < V) len[slot[u]] = uint32_t(ofs[u + 1] - ofs[u]);
}

// Every edge to its row's new place, its column numbered; perm names its old
// position.  A thread per edge: a wave per row spent 80 ms on one row of 7.6 M
// edges.
__global__ void k_move_entries(const uint64_t* ofs, const uint32_t* adj, const uint32_t* tail,
                               const uint32_t* slot, const uint64_t* new_ofs, uint32_t* perm,
                               uint32_t* col, uint64_t n) {
  const uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const uint32_t u = tail[e];
  const uint64_t to = new_ofs[slot[u]] + (e - ofs[u]);
  perm[to] = uint32_t(e);
  col[to] = slot[adj[e]];
}

// xs[slot[v]] = x[v].
__global__ void k_to_slots(const float* x, const uint32_t* slot, float* xs, uint64_t n) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) xs[slot[i]] = x[i];
}

// x[v] = xs[slot[v]].
__global__ void k_from_slots(const float* xs, const uint32_t* slot, float* x, uint64_t n) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) x[i] = xs[slot[i]];
}

__global__ void k_gather_w(const float* w, const uint32_t* perm, float* out, uint64_t n) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = w[perm[i]];
}

__global__ void k_scale(const float* x, float* y, uint64_t n, float s) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) y[i] = s * x[i];
}

// dL/dw over out-edges: rows u, edges (u, v).
__global__ __launch_bounds__(kBlock) void k_edge_grad(const RowItem* items, const uint64_t* ofs,
                                                      const uint32_t* adj, const float* r,
                                                      const float* lam, float d, float* dw) {
  __shared__ uint64_t rofs[kRowsPerItem + 1];
  const RowItem it = items[blockIdx.x];
  if (it.npieces == 0) {
    const uint32_t nrows = it.row_end - it.row_begin;
    for (uint32_t i = threadIdx.x; i <= nrows; i += kBlock) rofs[i] = ofs[it.row_begin + i];
    __syncthreads();
    const uint64_t e0 = rofs[0], e1 = rofs[nrows];
    for (uint64_t e = e0 + threadIdx.x; e < e1; e += kBlock) {
      uint32_t lo = 0, hi = nrows;  // row k with rofs[k] <= e < rofs[k+1]
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (rofs[mid] <= e) lo = mid; else hi = mid;
      }
      dw[e] = d * r[it.row_begin + lo] * lam[adj[e]];
    }
  } else {
    const uint32_t u = it.row_begin;
    const uint64_t lo = ofs[u] + uint64_t(it.piece) * kPiece;
    const uint64_t hi = min(ofs[u + 1], lo + kPiece);
    const float ru = d * r[u];
    for (uint64_t e = lo + threadIdx.x; e < hi; e += kBlock) dw[e] = ru * lam[adj[e]];
  }
}

// The sweep items of matrix `c`.
void build_sweep_items(ll_gpu_ctx* ctx, const Csr& c, WprMatrix& m) {
  hipStream_t s = ctx->stream;
  RowBlocks rb;
  build_rowblocks(ctx, c, kCap, kWPiece, rb);
  DevBuf cnt;
  cnt.alloc(4, s);
  m.items.alloc(std::max<uint64_t>(rb.n, 1) * sizeof(SpItem), s);
  m.splits.alloc(std::max<uint64_t>(rb.nsplit, 1) * sizeof(SpSplit), s);
  k_zero_u32<<<1, 1, 0, s>>>(cnt.as<uint32_t>());
  k_sweep_items<<<grid_for(rb.n, 256), 256, 0, s>>>(
      rb.items.as<RowItem>(), rb.slots.as<uint32_t>(), rb.n, c.ofs.as<uint64_t>(),
      m.items.as<SpItem>(), m.splits.as<SpSplit>(), cnt.as<uint32_t>());
  LLG_HIP(hipGetLastError());
  if (rb.nsplit) {
    LLG_HIP(hipMemcpyAsync(ctx->readback, cnt.p, 4, hipMemcpyDeviceToHost, s));
    LLG_HIP(hipStreamSynchronize(s));
    m.nsplits = *static_cast<const uint32_t*>(ctx->readback);
  }
  m.n = rb.n;
  m.nparts = rb.nsplit;
}

// Whether x's hottest entries are worth an LDS table: they hold kHotShare of
// the columns, and the graph is large enough, and its rows long enough, for 96
// KiB copied per workgroup and rows numbered anew.  50 iterations forward and back, ms with table /
// plain (first call on a snapshot in brackets): R-MAT of 16 edges a vertex
// (share) 24576 vertices 1.8 / 1.1; 200003 (0.85) 2.54 / 2.48 [5.9 / 4.7];
// 400000 (0.75) 3.5 / 4.1; 2^20 (0.65) 7.7 / 10.6 [17.5 / 16.0]; 2^22 (0.47)
// 39 / 69 [55 / 78].  Even degrees: 2^20 (0.04) 12.5 / 10.7 [21.6 / 16.2], 24577
// 1.5 / 0.8.  Power laws whose IDs already ascend by degree: 2^20 (0.29) 10.8 /
// 10.4, (0.39) 10.3 / 9.8, (0.59) 9.6 / 9.1, 2^22 (0.36) 57 / 53: there the
// table loses 5%, with IDs in any order it wins as on R-MAT.
constexpr uint64_t kTableV = uint64_t(1) << 18;
constexpr double kHotShare = 0.3;

// The matrix of one direction of the sweeps.  forward: rows = heads, columns =
// tails; adjoint: rows = tails, columns = heads.  Entries of a row in out-edge
// order.  With a table, rows and columns are numbered by descending degree on
// the column side; else they keep their IDs, and the adjoint's matrix is the
// out-CSR itself (also past 2^32 edges, where no u32 permutation exists).
const WprMatrix& ensure_wpr_matrix(ll_gpu_graph* g, int level, bool forward) {
  level = resolve_level(g, level);
  WprMatrix& m = g->wpr[forward ? 0 : 1];
  if (m.level == level) return m;
  ll_gpu_ctx* ctx = g->ctx;
  hipStream_t s = ctx->stream;
  const Csr& out = ensure_csr(g, LL_GPU_DIR_OUT, level);
  const uint64_t V = g->V, E = out.E;
  const bool fits = E < (uint64_t(1) << 32);
  LLG_CHECK(fits || !forward, LL_GPU_ERANGE, "weighted PageRank needs E < 2^32");
  m = WprMatrix();
  if (fits && V >= kTableV && E / 4 >= V) {
    DevBuf counted;
    const uint32_t* deg;
    if (!forward && g->slcsr && !g->sl[LL_GPU_DIR_IN].valid) {
      // a single-level CSR may hold the out-edges alone
      counted.alloc(V * 4, s);
      k_fill_u32<<<grid_for(V, 256), 256, 0, s>>>(counted.as<uint32_t>(), V, 0u);
      k_count_heads<<<grid_for(E, 256), 256, 0, s>>>(out.adj.as<uint32_t>(), E,
                                                     counted.as<uint32_t>());
      LLG_HIP(hipGetLastError());
      deg = counted.as<uint32_t>();
    } else {
      deg = ensure_degrees(g, forward ? LL_GPU_DIR_OUT : LL_GPU_DIR_IN, level);
    }
    m.table = double(top_degree_sum(ctx, deg, nullptr, V, kHot)) >= kHotShare * double(E);
    if (m.table) degree_slots(ctx, deg, V, m.slot);
  }
  if (!forward && !m.table) {
    build_sweep_items(ctx, out, m);
    m.level = level;
    return m;
  }
  const uint32_t* slot = m.slot.as<uint32_t>();
  const uint32_t* heads = out.adj.as<uint32_t>();
  const uint64_t n = std::max<uint64_t>(E, 1);
  m.perm.alloc(n * 4, s);
  m.csr.ofs.alloc((V + 1) * 8, s);
  m.csr.adj.alloc(n * 4, s);
  DevBuf tail;  // the forward's sort keys first
  tail.alloc(n * 4, s);
  auto edge_tails = [&]() {
    k_edge_tails<<<unsigned(std::min<uint64_t>((V + 3) / 4, uint64_t(ctx->num_cus) * 32)), 256, 0,
                   s>>>(out.ofs.as<uint64_t>(), V, tail.as<uint32_t>());
  };
  if (forward) {
    DevBuf pos, rows;
    pos.alloc(n * 4, s);
    rows.alloc(n * 4, s);
    k_row_keys<<<grid_for(E, 256), 256, 0, s>>>(heads, slot, tail.as<uint32_t>(),
                                                pos.as<uint32_t>(), E);
    LLG_HIP(hipGetLastError());
    int bits = 1;
    while (bits < 32 && ((V - 1) >> bits) != 0) bits++;
    sort_pairs_u32_u32(tail.as<uint32_t>(), rows.as<uint32_t>(), pos.as<uint32_t>(),
                       m.perm.as<uint32_t>(), E, bits, s, false);
    edge_tails();
    k_row_offsets<<<grid_for(V + 1, 256), 256, 0, s>>>(rows.as<uint32_t>(), E, V,
                                                       m.csr.ofs.as<uint64_t>());
    k_columns<<<grid_for(E, 256), 256, 0, s>>>(m.perm.as<uint32_t>(), tail.as<uint32_t>(), slot,
                                               m.csr.adj.as<uint32_t>(), E);
  } else {
    // the rows are the out-CSR's, whole, in another order: nothing to sort
    DevBuf len;
    len.alloc(V * 4, s);
    edge_tails();
    k_row_lengths<<<grid_for(V, 256), 256, 0, s>>>(out.ofs.as<uint64_t>(), slot, V,
                                                   len.as<uint32_t>());
    scan_u32_to_u64(len.as<uint32_t>(), m.csr.ofs.as<uint64_t>(), V, s);
    k_move_entries<<<grid_for(E, 256), 256, 0, s>>>(
        out.ofs.as<uint64_t>(), heads, tail.as<uint32_t>(), slot, m.csr.ofs.as<uint64_t>(),
        m.perm.as<uint32_t>(), m.csr.adj.as<uint32_t>(), E);
  }
  LLG_HIP(hipGetLastError());
  m.csr.valid = true;
  m.csr.level = level;
  m.csr.V = V;
  m.csr.E = E;
  build_sweep_items(ctx, m.csr, m);
  m.level = level;
  return m;
}

// iters >= 1 sweeps y = base_scale * base + d * (matrix * y) from y = base;
// the last y, by vertex, in `out`.
void wpr_sweeps(ll_gpu_graph* g, int level, bool forward, const float* w, const float* base,
                float base_scale, float d, int iters, float* out, const char* name) {
  ll_gpu_ctx* ctx = g->ctx;
  hipStream_t s = ctx->stream;
  const WprMatrix& m = ensure_wpr_matrix(g, level, forward);
  const Csr& c = m.csr.valid ? m.csr : ensure_csr(g, LL_GPU_DIR_OUT, level);
  const uint64_t V = g->V;
  const uint32_t* slot = m.slot.as<uint32_t>();
  DevBuf w_in, base_in, buf[2], part;
  if (m.perm.p) {
    w_in.alloc(std::max<uint64_t>(c.E, 1) * 4, s);
    k_gather_w<<<grid_for(c.E, 256), 256, 0, s>>>(w, m.perm.as<uint32_t>(), w_in.as<float>(), c.E);
    w = w_in.as<float>();
  }
  if (slot) {
    base_in.alloc(V * 4, s);
    k_to_slots<<<grid_for(V, 256), 256, 0, s>>>(base, slot, base_in.as<float>(), V);
    base = base_in.as<float>();
  }
  LLG_HIP(hipGetLastError());
  buf[0].alloc(V * 4, s);
  buf[1].alloc(V * 4, s);
  part.alloc(m.nparts * 8, s);
  SpArgs a{};
  a.items = m.items.as<SpItem>();
  a.nitems = m.n;
  a.splits = m.splits.as<SpSplit>();
  a.nsplits = m.nsplits;
  a.ofs = c.ofs.as<uint64_t>();
  a.col = c.adj.as<uint32_t>();
  a.val = w;
  a.x = base;
  a.nx = V;
  a.base = base;
  a.base_scale = base_scale;
  a.d = d;
  a.part = part.as<double>();
  const uint64_t per = (m.table ? kSpBlock : kBlock) / 64;  // waves of a workgroup
  // with a table one workgroup fits a CU and its copy is to be shared by many
  // items; else as many as there are items, up to many a CU (8 a CU: 5% slower)
  const unsigned grid = unsigned(std::min<uint64_t>(
      (m.n + per - 1) / per, uint64_t(ctx->num_cus) * (m.table ? 1 : 64)));
  for (int it = 0; it < iters; it++) {
    a.y = it == iters - 1 && !slot ? out : buf[it & 1].as<float>();
    {
      TimedLaunch t(ctx, name);
      if (m.table) k_wspmv<true><<<grid, kSpBlock, 0, s>>>(a);
      else k_wspmv<false><<<grid, kBlock, 0, s>>>(a);
    }
    if (a.nsplits) k_wspmv_split<<<grid_for(uint64_t(a.nsplits) * kSplitLanes, 64), 64, 0, s>>>(a);
    LLG_HIP(hipGetLastError());
    a.x = a.y;
  }
  if (slot) k_from_slots<<<grid_for(V, 256), 256, 0, s>>>(a.x, slot, out, V);
  LLG_HIP(hipGetLastError());
}

}  // namespace

// Forward: iters sweeps from r0 = p; result in r_out (device).
void wpr_forward_device(ll_gpu_graph* g, int level, const float* w, const float* p, int iters,
                        double d, float* r_out) {
  if (iters > 0) {
    wpr_sweeps(g, level, true, w, p, float(1.0 - d), float(d), iters, r_out, "k_wspmv_fwd");
  } else {
    ensure_wpr_matrix(g, level, true);
    LLG_HIP(hipMemcpyAsync(r_out, p, g->V * 4, hipMemcpyDeviceToDevice, g->ctx->stream));
  }
}

void wpr_adjoint_device(ll_gpu_graph* g, int level, const float* w, const float* r,
                        const float* gr, int iters, double d, float* dw, float* dp) {
  ll_gpu_ctx* ctx = g->ctx;
  hipStream_t s = ctx->stream;
  const Csr& out = ensure_csr(g, LL_GPU_DIR_OUT, level);
  const RowBlocks& rb = ensure_rowblocks(g, LL_GPU_DIR_OUT, level, kGradCap, kPiece);
  const uint64_t V = g->V;
  DevBuf lam_v;
  const float* lam = gr;
  if (iters > 0) {
    lam_v.alloc(V * 4, s);
    wpr_sweeps(g, level, false, w, gr, 1.0f, float(d), iters, lam_v.as<float>(), "k_wspmv_adj");
    lam = lam_v.as<float>();
  }
  if (dw) {
    TimedLaunch t(ctx, "k_edge_grad");
    k_edge_grad<<<unsigned(rb.n), kBlock, 0, s>>>(rb.items.as<RowItem>(), out.ofs.as<uint64_t>(),
                                                  out.adj.as<uint32_t>(), r, lam, float(d), dw);
  }
  if (dp) k_scale<<<grid_for(V, 256), 256, 0, s>>>(lam, dp, V, float(1.0 - d));
  LLG_HIP(hipGetLastError());
}

}  // namespace llgpu

extern "C" {

int ll_gpu_wpr_forward(ll_gpu_graph* g, int level, const float* edge_w, const float* teleport,
                       int iters, double damping, float* r_out) {
  if (!g) return LL_GPU_EINVAL;
  try {
    LLG_HIP(hipSetDevice(g->ctx->device));
    LLG_CHECK(edge_w && teleport && r_out, LL_GPU_EINVAL, "NULL device pointer");
    LLG_CHECK(iters >= 0 && damping >= 0 && damping <= 1, LL_GPU_EINVAL, "bad iters/damping");
    llgpu::wpr_forward_device(g, level, edge_w, teleport, iters, damping, r_out);
    LLG_HIP(hipStreamSynchronize(g->ctx->stream));
    return LL_GPU_OK;
  } catch (const llgpu::Error& e) {
    g->ctx->err = e.msg;
    return e.code;
  } catch (...) {
    return llgpu::api_exception(g->ctx);
  }
}

int ll_gpu_wpr_adjoint(ll_gpu_graph* g, int level, const float* edge_w, const float* r,
                       const float* dl_dr, int iters, double damping, float* dl_dw_out,
                       float* dl_dteleport_out) {
  if (!g) return LL_GPU_EINVAL;
  try {
    LLG_HIP(hipSetDevice(g->ctx->device));
    LLG_CHECK(edge_w && r && dl_dr, LL_GPU_EINVAL, "NULL device pointer");
    LLG_CHECK(iters >= 0 && damping >= 0 && damping <= 1, LL_GPU_EINVAL, "bad iters/damping");
    llgpu::wpr_adjoint_device(g, level, edge_w, r, dl_dr, iters, damping, dl_dw_out,
                              dl_dteleport_out);
    LLG_HIP(hipStreamSynchronize(g->ctx->stream));
    return LL_GPU_OK;
  } catch (const llgpu::Error& e) {
    g->ctx->err = e.msg;
    return e.code;
  } catch (...) {
    return llgpu::api_exception(g->ctx);
  }
}

}  // extern "C"
