// How the split gate/up (moe_gemm_split.hip) cuts the experts' sorted rows into
// chunks and deals them: the chunk table (built by one wave from the sort's
// expert counts), the chunk of a number, and a workgroup's share. Integer work
// and cross-lane operations only, so that the host test compiles this file with
// its own definitions of those (tests/split_table_host.cpp).
#pragma once
#include <cstdint>

namespace nksplit {

constexpr uint32_t kMaxE = 513;             // experts, the shared one included
constexpr uint32_t kPer = (kMaxE + 63) / 64;  // experts per lane of the scan

struct Table {
  uint32_t n[kMaxE];        // rows of each expert
  uint32_t off[kMaxE + 1];  // 64-row blocks before it << 16 | chunks before it; [Etot]: all of them
};

struct Chunk {
  uint32_t e, row0, tiles, first;  // expert, first sorted row, 16-row tiles, its number among all chunks
};

// The chunk table, by one wave (the caller puts a barrier behind it). Counts
// are clamped to T: an operation launched out of order may find another
// tensor's bytes there.
template <uint32_t RM>
__device__ __forceinline__ void build_table(Table& s, const int32_t* __restrict__ counts, uint32_t T, uint32_t Etot,
                                            uint32_t lane) {
  const uint32_t per = (Etot + 63u) / 64u;
  uint32_t n[kPer], c[kPer], b[kPer], cs = 0, bs = 0;
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    const uint32_t e = lane * per + i;
    n[i] = (uint32_t)counts[min(e, Etot - 1u)];  // unconditional: all in flight together
  }
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) n[i] = i < per && lane * per + i < Etot ? min(n[i], T) : 0u;
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    c[i] = ((n[i] + 15u) / 16u + RM - 1u) / RM;
    b[i] = (n[i] + 63u) / 64u;
    cs += c[i];
    bs += b[i];
  }
  uint32_t ci = cs, bi = bs;  // inclusive scans over the lanes
#pragma unroll
  for (uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t oc = __shfl_up(ci, off), ob = __shfl_up(bi, off);
    if (lane >= off) { ci += oc; bi += ob; }
  }
  if (lane == 63u) s.off[Etot] = bi << 16 | ci;
  ci -= cs;
  bi -= bs;
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    const uint32_t e = lane * per + i;
    if (i < per && e < Etot) {
      s.n[e] = n[i];
      s.off[e] = bi << 16 | ci;
      ci += c[i];
      bi += b[i];
    }
  }
}

__device__ __forceinline__ uint32_t all_chunks(const Table& s, uint32_t Etot) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)s.off[Etot]) & 0xffffu;
}

// Chunk number q (below the total, uniform, every lane active): the last
// expert whose chunks begin at or before q, by two ballots.
__device__ __forceinline__ Chunk locate(const Table& s, uint32_t q, uint32_t Etot, uint32_t lane) {
  const uint32_t per = (Etot + 63u) / 64u;
  const uint32_t l0 = lane * per;
  const unsigned long long m0 = __ballot(l0 < Etot && (s.off[min(l0, Etot - 1u)] & 0xffffu) <= q);
  const uint32_t base = ((uint32_t)__popcll(m0) - 1u) * per;
  const uint32_t l1 = base + lane;
  const unsigned long long m1 = __ballot(lane < per && l1 < Etot && (s.off[min(l1, Etot - 1u)] & 0xffffu) <= q);
  Chunk k;
  k.e = __builtin_amdgcn_readfirstlane((int)(base + (uint32_t)__popcll(m1) - 1u));
  const uint32_t off = __builtin_amdgcn_readfirstlane((int)s.off[k.e]), c0 = off & 0xffffu;
  const uint32_t nc = (__builtin_amdgcn_readfirstlane((int)s.off[k.e + 1u]) & 0xffffu) - c0;
  const uint32_t tiles = (__builtin_amdgcn_readfirstlane((int)s.n[k.e]) + 15u) / 16u;
  const uint32_t t0 = (q - c0) * tiles / nc, t1 = (q - c0 + 1u) * tiles / nc;
  k.row0 = (off >> 16) * 64u + t0 * 16u;
  k.tiles = t1 - t0;
  k.first = q;
  return k;
}

// This workgroup's share [lo, hi) of `total` positions, workgroups of an XCD
// (blockIdx % 8) side by side.
__device__ __forceinline__ void share(uint32_t total, uint32_t& lo, uint32_t& hi) {
  uint32_t w = blockIdx.x;
  if (gridDim.x % 8u == 0u) w = (w & 7u) * (gridDim.x / 8u) + (w >> 3);
  lo = (uint32_t)((uint64_t)w * total / gridDim.x);
  hi = (uint32_t)((uint64_t)(w + 1u) * total / gridDim.x);
}

}  // namespace nksplit
