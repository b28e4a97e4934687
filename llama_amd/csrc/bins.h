// Device helper shared by the sweeps over the binned out-edge layout
// (pr_bins.hip builds it): vertices in bins of 2^bb consecutive IDs, every
// out-edge (u, v) owning one slot, the slots of destination bin b' grouped by
// the source's bin b into chunks (b', b), contiguous, and a chunk table by
// source bin, ct[b * nb + b'] = {first slot, slots}.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace llgpu {

// Bin sizes the layout is built for.
constexpr uint32_t kMinBinBits = 8;
constexpr uint32_t kMaxBinBits = 14;

// Workgroup of the sweeps that take one bin each.  1024 threads at every size:
// small bins then spread their few slots over 16 waves (2^8 vertices, 10^4
// vertices and 1.6*10^5 edges: 9.1 us per PageRank iteration against 13.9 us
// with 256 threads), large ones fill a CU with the one or two workgroups their
// LDS words leave room for (2^13: 243 us against 439 us at 4.2 M vertices,
// 67 M edges).
constexpr int kBinBlock = 1024;

// Calls f with the bin bits as a compile-time constant.
template <typename F>
inline void with_bin_bits(uint32_t bb, F&& f) {
  switch (bb) {
    case 8: f(std::integral_constant<uint32_t, 8>{}); break;
    case 9: f(std::integral_constant<uint32_t, 9>{}); break;
    case 10: f(std::integral_constant<uint32_t, 10>{}); break;
    case 11: f(std::integral_constant<uint32_t, 11>{}); break;
    case 12: f(std::integral_constant<uint32_t, 12>{}); break;
    case 13: f(std::integral_constant<uint32_t, 13>{}); break;
    default: f(std::integral_constant<uint32_t, 14>{}); break;
  }
}

// Writes the values of one source bin's vertices into the bin's chunks for
// every destination bin: slot k of a chunk gets cl[sidx[k]], where cl holds
// the bin's values by offset (LDS) and sidx names each slot's source offset.
// Every slot of the bin's chunks is written.
//
// Bound by the slot streams, as long as enough loads are in flight: the
// chunks are dealt evenly to the waves (with fewer chunks than waves, each is
// cut into equal parts), a wave holds 64 table entries in its lanes and walks
// them in pieces of 64 slots, kGroup pieces requested together whether they
// are kGroup short chunks or one long one.  The piece bounds are wave-uniform
// (scalar registers).
template <int kBlock, int kGroup, typename T>
__device__ __forceinline__ void scatter_chunks(const uint2* row, uint32_t nb,
                                               const uint16_t* sidx, const T* cl, T* out) {
  constexpr uint32_t kWaves = kBlock / 64;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  const uint32_t parts = nb < kWaves ? kWaves / nb : 1u;
  const uint32_t n = nb * parts;
  const uint32_t lo = uint32_t(uint64_t(n) * wave / kWaves);
  const uint32_t hi = uint32_t(uint64_t(n) * (wave + 1) / kWaves);
  for (uint32_t c0 = lo; c0 < hi; c0 += 64) {
    uint2 t = make_uint2(0u, 0u);
    if (c0 + lane < hi) {
      const uint32_t c = c0 + lane;
      t = row[c / parts];
      if (parts > 1) {
        const uint32_t k = c % parts;
        const uint32_t a = uint32_t(uint64_t(t.y) * k / parts);
        const uint32_t z = uint32_t(uint64_t(t.y) * (k + 1) / parts);
        t = make_uint2(t.x + a, z - a);
      }
    }
    uint64_t todo = __ballot(t.y != 0);  // entries not walked yet
    uint32_t at = 0, left = 0;           // the current entry's next slot, slots left
    while (todo || left) {
      uint32_t st[kGroup], len[kGroup];
#pragma unroll
      for (int q = 0; q < kGroup; q++) {
        if (left == 0 && todo) {
          const int j = __ffsll((long long)todo) - 1;
          todo &= todo - 1;
          at = uint32_t(__builtin_amdgcn_readlane(int(t.x), j));
          left = uint32_t(__builtin_amdgcn_readlane(int(t.y), j));
        }
        st[q] = at;
        len[q] = min(left, 64u);
        at += len[q];
        left -= len[q];
      }
      uint16_t s[kGroup];
#pragma unroll
      for (int q = 0; q < kGroup; q++) s[q] = lane < len[q] ? sidx[st[q] + lane] : uint16_t(0);
#pragma unroll
      for (int q = 0; q < kGroup; q++)
        if (lane < len[q]) out[st[q] + lane] = cl[s[q]];
    }
  }
}

}  // namespace llgpu
