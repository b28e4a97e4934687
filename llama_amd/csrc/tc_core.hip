// Triangle counting over a DAG whose vertices are numbered by degree.
//
// Arcs go from lower to higher (degree, ID), as in tc.hip; here that order is
// the numbering itself, so the neighbours of a list are its hubs-to-be and the
// kCore highest numbers (the core) hold nearly every list entry of a skewed
// graph.  A row a sets the bits of N+(a) within the core in an LDS bitmap (4
// KiB a wave); the core part of every N+(b), b in N+(a), is then streamed as
// 16-bit offsets and each entry costs one LDS bit test.  Entries outside the
// core -- only neighbours of a b that is itself outside -- pass a hashed bit
// filter and are confirmed by a binary search of N+(a).
#include "ll_gpu_internal.h"

namespace llgpu {

namespace {

constexpr uint32_t kCore = 32768;       // core numbers fit 16 bits
constexpr uint32_t kNone = kCore;       // stands for no entry: its bit is never set
constexpr uint32_t kFilterBits = 2048;  // filter of a row's neighbours outside the core
constexpr int kWaves = 8;               // waves per workgroup, a row each
constexpr int kGroup = 8;               // pieces of 64 entries in flight per wave

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline uint32_t lane_val(uint32_t x, int lane) {
  return uint32_t(__builtin_amdgcn_readlane(int(x), lane));
}
__device__ inline uint64_t lane_val(uint64_t x, int lane) {
  const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(x)), lane));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(x >> 32)), lane));
  return uint64_t(hi) << 32 | lo;
}

__global__ void k_degree_keys(const uint32_t* dout, const uint32_t* din, uint32_t* key,
                              uint32_t* id, uint64_t V) {
  const uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (v >= V) return;
  key[v] = uint32_t(min(uint64_t(dout[v]) + din[v], uint64_t(0xffffffffu)));
  id[v] = uint32_t(v);
}

__global__ void k_number(const uint32_t* sorted_ids, uint32_t* num, uint64_t V) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < V) num[sorted_ids[i]] = uint32_t(i);
}

__global__ void k_zero_ull(unsigned long long* p, uint32_t n) {
  if (threadIdx.x < n) p[threadIdx.x] = 0;
}

// The key of a self-loop: all ones, past every arc's.
__host__ __device__ inline uint64_t no_arc(uint32_t vb) {
  return vb >= 32 ? ~uint64_t(0) : (uint64_t(1) << (2 * vb)) - 1;
}

// Arc key of every live edge, a wave per vertex row: lower number << vb |
// higher number.
__global__ __launch_bounds__(256) void k_arc_keys(const uint64_t* ofs, const uint32_t* adj,
                                                  const uint32_t* num, uint64_t V, uint32_t vb,
                                                  uint64_t* keys) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t nw = uint64_t(gridDim.x) * (blockDim.x / 64);
  const uint64_t none = no_arc(vb);
  for (uint64_t u = uint64_t(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6); u < V;
       u += nw) {
    const uint64_t ru = num[u];
    for (uint64_t e = ofs[u] + lane, end = ofs[u + 1]; e < end; e += 64) {
      const uint64_t rv = num[adj[e]];
      keys[e] = ru == rv ? none : ru < rv ? ru << vb | rv : rv << vb | ru;
    }
  }
}

// Row offsets of the sorted arc keys, a thread per row (runs of rows without
// arcs are long here: the vertices of degree 0 come first).
__global__ void k_arc_rows(const uint64_t* keys, uint64_t m, uint64_t V, uint32_t vb,
                           uint64_t* ofs) {
  const uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (x > V) return;
  uint64_t lo = 0, hi = m;  // first arc of a row >= x
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if ((keys[mid] >> vb) < x) lo = mid + 1;
    else hi = mid;
  }
  ofs[x] = lo;
}

// Higher ends of the arcs and their core offsets (arcs into the core).
__global__ void k_arc_ends(const uint64_t* keys, uint64_t m, uint32_t vb, uint32_t core0,
                           uint32_t* nbr, uint16_t* nbc) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const uint32_t b = uint32_t(keys[i] & ((uint64_t(1) << vb) - 1));
  nbr[i] = b;
  nbc[i] = uint16_t(b - core0);
}

// Arcs of each row that end outside the core (the row's first ones).
__global__ void k_outside(const uint64_t* ofs, const uint32_t* nbr, uint64_t V, uint32_t core0,
                          uint32_t* nout) {
  const uint64_t a = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (a >= V) return;
  const uint64_t a0 = ofs[a];
  uint64_t lo = a0, hi = ofs[a + 1];
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (nbr[mid] < core0) lo = mid + 1;
    else hi = mid;
  }
  nout[a] = uint32_t(lo - a0);
}

__device__ inline uint32_t filter_bit(uint32_t x) {
  return (x * 2654435761u) >> 21;  // 11 bits
}
static_assert(kFilterBits == 2048, "filter_bit gives 11 bits");

struct TcCoreArgs {
  const uint64_t* ofs;
  const uint32_t* nbr;
  const uint16_t* nbc;
  const uint32_t* nout;
  uint64_t V;
  unsigned long long* out;  // triangles, W, largest row element count
};

// A wave per row, from the highest number down (the rows of one wave then mix
// heavy and light ones), 64 rows looked at together.  Bound by instruction
// issue: about 12 vector and 12 scalar instructions per piece of 64 entries
// (90% full on R-MAT graphs); the vector units issue for 74% of the kernel's
// cycles, the LDS of the bit tests for 35%.  2^20 vertices, 4.4 G entries: 2.0
// ms (10.8 with a bucketed search of N+(a) per entry).  A core of 65536
// numbers: 3.7 ms (half the waves fit a CU) and 16384: 3.2 against 3.1 of
// 32768; then 32-bit positions and loads past a piece's end instead of masked
// ones: 2.3; workgroups of 8 waves instead of 4: 2.2; more of them: 2.0.
// I: type of an arc position.
template <typename I>
__global__ __launch_bounds__(kWaves * 64, 8) void k_tc_core(TcCoreArgs a) {
  __shared__ uint32_t s_bits[kWaves][kCore / 32 + 1];
  __shared__ uint32_t s_filter[kWaves][kFilterBits / 32];
  __shared__ unsigned long long red[3][kWaves];
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  uint32_t* bits = s_bits[wave];
  uint32_t* filter = s_filter[wave];
  for (uint32_t i = lane; i <= kCore / 32; i += 64) bits[i] = 0;
  for (uint32_t i = lane; i < kFilterBits / 32; i += 64) filter[i] = 0;
  wave_sync();
  unsigned long long count = 0, work = 0, maxrow = 0;
  const uint64_t nw = uint64_t(gridDim.x) * kWaves;
  for (uint64_t r0 = uint64_t(blockIdx.x) * kWaves + wave; r0 < a.V; r0 += 64 * nw) {
    // the wave's next 64 rows, a lane each; those of one arc close no triangle
    // and are done there
    const uint64_t mine = r0 + lane * nw;
    uint64_t mine_a0 = 0;
    uint32_t mine_na = 0, mine_out = 0;
    if (mine < a.V) {
      const uint64_t row = a.V - 1 - mine;
      mine_a0 = a.ofs[row];
      mine_na = uint32_t(a.ofs[row + 1] - mine_a0);
      if (mine_na == 1) {
        const uint32_t b = a.nbr[mine_a0];
        const unsigned long long el = a.ofs[b + 1] - a.ofs[b];
        work += el + 1;
        maxrow = el > maxrow ? el : maxrow;
      } else if (mine_na > 1) {
        mine_out = a.nout[row];
      }
    }
    for (uint64_t todo_rows = __ballot(mine_na > 1); todo_rows; todo_rows &= todo_rows - 1) {
      const int rj = __ffsll((long long)todo_rows) - 1;
      const uint64_t a0 = lane_val(mine_a0, rj);
      const uint64_t na = lane_val(mine_na, rj), a1 = a0 + na;
      const uint32_t outside = lane_val(mine_out, rj);
      const uint64_t c0 = a0 + outside;
      for (uint64_t e = c0 + lane; e < a1; e += 64) {
        const uint32_t x = a.nbc[e];
        atomicOr(&bits[x >> 5], 1u << (x & 31));
      }
      for (uint64_t e = a0 + lane; e < c0; e += 64) {
        const uint32_t h = filter_bit(a.nbr[e]);
        atomicOr(&filter[h >> 5], 1u << (h & 31));
      }
      wave_sync();
      uint32_t c = 0;
      unsigned long long el = 0;
      for (uint64_t i0 = 0; i0 < na; i0 += 64) {
        const uint64_t i = i0 + lane;
        I start = 0, ostart = 0;
        uint32_t len = 0, olen = 0;
        if (i < na) {
          const uint32_t b = a.nbr[a0 + i];
          const uint64_t b0 = a.ofs[b], b1 = a.ofs[b + 1];
          const uint32_t bo = a.nout[b];
          el += b1 - b0;
          start = I(b0 + bo);
          len = uint32_t(b1 - b0) - bo;
          if (i < outside && outside > 1) {
            ostart = I(b0);
            olen = bo;
          }
        }
        // the core parts of the 64 lists, in pieces of 64 entries
        uint64_t todo = __ballot(len != 0);
        I at = 0;
        uint32_t left = 0;
        while (todo || left) {
          uint32_t n[kGroup];
          uint16_t w[kGroup];
#pragma unroll
          for (int q = 0; q < kGroup; q++) {
            if (left == 0 && todo) {
              const int j = __ffsll((long long)todo) - 1;
              todo &= todo - 1;
              at = lane_val(start, j);
              left = lane_val(len, j);
            }
            n[q] = min(left, 64u);
            w[q] = (a.nbc + at)[lane];  // past the piece: other entries, or the padding
            at += n[q];
            left -= n[q];
          }
#pragma unroll
          for (int q = 0; q < kGroup; q++) {
            const uint32_t x = lane < n[q] ? uint32_t(w[q]) : kNone;
            c += (bits[x >> 5] >> (x & 31)) & 1u;
          }
        }
        // the entries outside the core of the lists of vertices outside it
        for (uint64_t om = __ballot(olen != 0); om; om &= om - 1) {
          const int j = __ffsll((long long)om) - 1;
          const I s0 = lane_val(ostart, j);
          const uint32_t n = lane_val(olen, j);
          for (uint32_t t = lane; t < n; t += 64) {
            const uint32_t w = a.nbr[s0 + t];
            const uint32_t h = filter_bit(w);
            if (!((filter[h >> 5] >> (h & 31)) & 1u)) continue;
            uint64_t lo = a0, hi = c0;
            while (lo < hi) {
              const uint64_t mid = (lo + hi) >> 1;
              if (a.nbr[mid] < w) lo = mid + 1;
              else hi = mid;
            }
            c += lo < c0 && a.nbr[lo] == w ? 1u : 0u;
          }
        }
      }
      wave_sync();
      for (uint64_t e = c0 + lane; e < a1; e += 64) bits[a.nbc[e] >> 5] = 0;
      for (uint64_t e = a0 + lane; e < c0; e += 64) filter[filter_bit(a.nbr[e]) >> 5] = 0;
      wave_sync();
      count += c;
      work += el + (lane == 0 ? na * na : 0);  // na arcs of d+(a) each, and every d+(b)
      for (int o = 32; o > 0; o >>= 1) el += __shfl_xor(el, o, 64);
      maxrow = el > maxrow ? el : maxrow;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    count += __shfl_down(count, o, 64);
    work += __shfl_down(work, o, 64);
    const unsigned long long m = __shfl_down(maxrow, o, 64);
    maxrow = m > maxrow ? m : maxrow;
  }
  if (lane == 0) {
    red[0][wave] = count;
    red[1][wave] = work;
    red[2][wave] = maxrow;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0, w = 0, m = 0;
    for (int i = 0; i < kWaves; i++) {
      t += red[0][i];
      w += red[1][i];
      m = red[2][i] > m ? red[2][i] : m;
    }
    if (t) atomicAdd(a.out, t);
    if (w) atomicAdd(a.out + 1, w);
    if (m) atomicMax(a.out + 2, m);
  }
}

}  // namespace

// Builds (or reuses) the numbered DAG; false when the core would hold too
// little of the graph, and tc.hip's form by vertex ID is used instead.
bool ensure_tc_core(ll_gpu_graph* g, int level) {
  level = resolve_level(g, level);
  TcCore& t = g->tc_core;
  if (t.level == level) return t.usable;
  ll_gpu_ctx* ctx = g->ctx;
  hipStream_t s = ctx->stream;
  const uint64_t V = g->V;
  const Csr& out = ensure_csr(g, LL_GPU_DIR_OUT, level);
  const uint32_t* dout = ensure_degrees(g, LL_GPU_DIR_OUT, level);
  const uint32_t* din = ensure_degrees(g, LL_GPU_DIR_IN, level);
  const uint64_t E = out.E;
  t = TcCore();
  DevBuf num;
  const uint32_t core0 = uint32_t(V > kCore ? V - kCore : 0);
  if (core0) {
    // Entries outside the core cost several times a bit test.  With a share
    // x of the edge ends outside, x^2 of the arcs lie wholly outside (and
    // fewer of the list entries, the more skewed the graph).  Milliseconds of
    // a count, this form / by vertex ID, at x^2, [first call on a snapshot]:
    // R-MAT of 16 edges a vertex 2^20 vertices (0.10) 2.2 / 10.8 [8.2 / 16.2],
    // 2^22 (0.23) 11.8 / 55 [22 / 67], 2^24 123 / 308; even degrees 90000
    // vertices, 64 edges (0.36) 0.67 / 0.67 [2.8 / 3.7], 100000 (0.41) 0.80 /
    // 0.72 [2.9 / 3.8], 120000 (0.49) 1.18 / 0.79 [3.3 / 4.0].
    // With hubs among many small vertices the lists end in the core all the
    // same: R-MAT 2^20 and uniform edges, half as many (0.28) 3.1 / 11.4, as
    // many (0.41) 4.1 / 11.9, twice (0.56) 8.3 / 13.4, four times (0.70) 29 /
    // 17.9; 2^22 half (0.42) 16 / 58, as many (0.54) 22 / 60, twice (0.67) 45 /
    // 67, four times (0.79) 142 / 87.  So the limit is higher where the core's
    // vertices have 16 times the mean degree (2^22: 23 to 67), and not as high
    // as it could be: R-MAT 2^26 in 11 levels (0.59) 1.53 / 1.84 s, 2^27 in 20
    // (0.66) 5.2 / 4.5.  The share comes from a histogram of the degrees, before
    // any sort (a rejected graph of 4 M vertices paid 2.1 ms for one).
    const double in_core = double(top_degree_sum(ctx, dout, din, V, kCore));
    const double x = E ? 1.0 - in_core / (2.0 * double(E)) : 0.0;
    const double hub = (1.0 - x) * double(V) / kCore;  // mean degree of the core over all
    if (x * x > (hub >= 16 ? 0.5 : 0.42)) {
      t.level = level;
      t.usable = false;
      return false;
    }
  }
  {
    DevBuf key, id, skey, sid;
    key.alloc(V * 4, s);
    id.alloc(V * 4, s);
    skey.alloc(V * 4, s);
    sid.alloc(V * 4, s);
    num.alloc(V * 4, s);
    k_degree_keys<<<grid_for(V, 256), 256, 0, s>>>(dout, din, key.as<uint32_t>(),
                                                   id.as<uint32_t>(), V);
    sort_pairs_u32_u32(key.as<uint32_t>(), skey.as<uint32_t>(), id.as<uint32_t>(),
                       sid.as<uint32_t>(), V, 32, s);
    k_number<<<grid_for(V, 256), 256, 0, s>>>(sid.as<uint32_t>(), num.as<uint32_t>(), V);
    LLG_HIP(hipGetLastError());
  }
  uint32_t vb = 1;
  while (vb < 32 && ((V - 1) >> vb) != 0) vb++;
  const uint64_t n = std::max<uint64_t>(E, 1);
  DevBuf keys, sorted;
  keys.alloc(n * 8, s);
  sorted.alloc(n * 8, s);
  {
    TimedLaunch tl(ctx, "k_orient");
    const unsigned go = unsigned(std::min<uint64_t>(std::max<uint64_t>((V + 3) / 4, 1),
                                                    uint64_t(ctx->num_cus) * 32));
    k_arc_keys<<<go, 256, 0, s>>>(out.ofs.as<uint64_t>(), out.adj.as<uint32_t>(),
                                  num.as<uint32_t>(), V, vb, keys.as<uint64_t>());
  }
  LLG_HIP(hipGetLastError());
  sort_keys_u64(keys.as<uint64_t>(), sorted.as<uint64_t>(), E, int(2 * vb), s, false);
  uint64_t m = unique_u64(sorted.as<uint64_t>(), keys.as<uint64_t>(), E, s);
  if (m > 0) {  // the self-loops' key, if any, is the last
    uint64_t last = 0;
    copy_to_host(ctx, &last, keys.as<uint64_t>() + (m - 1), 8);
    if (last == no_arc(vb)) m--;
  }
  sorted.release();
  t.ofs.alloc((V + 1) * 8, s);
  t.nbr.alloc(std::max<uint64_t>(m, 1) * 4, s);
  t.nbc.alloc((m + 64) * 2, s);  // a piece loads 64 entries whatever its length
  t.nout.alloc(V * 4, s);
  k_arc_rows<<<grid_for(V + 1, 256), 256, 0, s>>>(keys.as<uint64_t>(), m, V, vb,
                                                  t.ofs.as<uint64_t>());
  k_arc_ends<<<grid_for(m, 256), 256, 0, s>>>(keys.as<uint64_t>(), m, vb, core0,
                                              t.nbr.as<uint32_t>(), t.nbc.as<uint16_t>());
  k_outside<<<grid_for(V, 256), 256, 0, s>>>(t.ofs.as<uint64_t>(), t.nbr.as<uint32_t>(), V, core0,
                                             t.nout.as<uint32_t>());
  LLG_HIP(hipGetLastError());
  t.arcs = m;
  t.level = level;
  t.usable = true;
  return true;
}

void tc_core_count(ll_gpu_graph* g, uint64_t* triangles, uint64_t* work, uint64_t* maxrow) {
  ll_gpu_ctx* ctx = g->ctx;
  hipStream_t s = ctx->stream;
  const TcCore& t = g->tc_core;
  DevBuf out;
  out.alloc(24, s);
  k_zero_ull<<<1, 64, 0, s>>>(out.as<unsigned long long>(), 3);
  {
    TimedLaunch tl(ctx, "k_tc_core");
    // four workgroups fit a CU; more of them even out the rows of many arcs,
    // and each clears its bitmaps once more.  us a count by workgroups a CU 8 /
    // 16 / 32, R-MAT, vertices x edges per vertex: 300000 x 4 115 / 169 / -,
    // 100000 x 16 167 / 220 / 351, 2^20 x 4 400 / 380 / 414, 300000 x 16 442 /
    // 411 / 471, 700000 x 16 1210 / 1133 / 1113, 2^20 x 16 2214 / 2020 / 1981,
    // 2^22 x 16 13191 / 12253 / 11800 (64: 1964 and 11699 at the last two).
    // Fewer yet for few arcs: a star of 500000 32 us with 1954 workgroups, 57
    // with 4096, 20000 x 16 65 with 1220, 87 with 2048.
    const uint64_t cus = uint64_t(ctx->num_cus);
    const uint64_t per_cu = t.arcs > (uint64_t(1) << 23) ? 32 : t.arcs > (uint64_t(3) << 20) ? 16 : 8;
    const unsigned grid = unsigned(std::min<uint64_t>(
        {(g->V + kWaves - 1) / kWaves, cus * per_cu, std::max<uint64_t>(t.arcs / 256, cus * 4)}));
    const TcCoreArgs a{t.ofs.as<uint64_t>(), t.nbr.as<uint32_t>(), t.nbc.as<uint16_t>(),
                       t.nout.as<uint32_t>(), g->V, out.as<unsigned long long>()};
    if (t.arcs < (uint64_t(1) << 32)) k_tc_core<uint32_t><<<grid, kWaves * 64, 0, s>>>(a);
    else k_tc_core<uint64_t><<<grid, kWaves * 64, 0, s>>>(a);
  }
  LLG_HIP(hipGetLastError());
  uint64_t h[3];
  copy_to_host(ctx, h, out.p, sizeof h);
  *triangles = h[0];
  *work = h[1];
  *maxrow = h[2];
}

}  // namespace llgpu
