// Compiles the split gate/up's chunk table (moe_split_table.h) for the host, 64
// threads standing in for a wave: stdin "T Etot RM grid blocks" and Etot counts;
// stdout every chunk "e row0 tiles", then every workgroup's share "lo hi" of
// chunks x blocks.
#include <pthread.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <thread>
#include <vector>

struct Dim { uint32_t x; };
static Dim blockIdx, gridDim;
static pthread_barrier_t wave_barrier;
static uint64_t slots[64];
static thread_local uint32_t me;

// every lane's value, then lane-wise use of it
template <class F>
static uint64_t exchange(uint64_t v, F use) {
  slots[me] = v;
  pthread_barrier_wait(&wave_barrier);
  const uint64_t r = use();
  pthread_barrier_wait(&wave_barrier);
  return r;
}
static uint32_t __shfl_up(uint32_t v, uint32_t off) {
  return (uint32_t)exchange(v, [&] { return slots[me >= off ? me - off : me]; });
}
static unsigned long long __ballot(bool p) {
  return exchange(p, [] { uint64_t m = 0; for (int i = 0; i < 64; ++i) m |= slots[i] << i; return m; });
}
static int readfirstlane(int v) { return (int)exchange((uint32_t)v, [] { return slots[0]; }); }
#define __popcll __builtin_popcountll
#define __builtin_amdgcn_readfirstlane readfirstlane
#define __device__
#define __forceinline__ inline
#define __restrict__ __restrict
using std::min;

#include "moe_split_table.h"

static nksplit::Table table;

template <uint32_t RM>
static void wave(uint32_t lane, const std::vector<int32_t>& counts, uint32_t T, std::vector<nksplit::Chunk>& out) {
  me = lane;
  const uint32_t Etot = (uint32_t)counts.size();
  nksplit::build_table<RM>(table, counts.data(), T, Etot, lane);
  pthread_barrier_wait(&wave_barrier);
  const uint32_t total = nksplit::all_chunks(table, Etot);
  for (uint32_t q = 0; q < total; ++q) {
    const nksplit::Chunk k = nksplit::locate(table, q, Etot, lane);
    if (lane == 0u) out.push_back(k);
  }
}

int main() {
  uint32_t T, Etot, RM, grid, blocks;
  if (std::scanf("%u %u %u %u %u", &T, &Etot, &RM, &grid, &blocks) != 5 || RM != 4u) return 1;
  std::vector<int32_t> counts(Etot);
  for (auto& c : counts)
    if (std::scanf("%d", &c) != 1) return 1;
  pthread_barrier_init(&wave_barrier, nullptr, 64);
  std::vector<nksplit::Chunk> chunks;
  std::vector<std::thread> lanes;
  for (uint32_t l = 0; l < 64; ++l) lanes.emplace_back([&, l] { wave<4>(l, counts, T, chunks); });
  for (auto& t : lanes) t.join();
  for (const auto& k : chunks) std::printf("%u %u %u\n", k.e, k.row0, k.tiles);
  gridDim.x = grid;
  for (blockIdx.x = 0; blockIdx.x < grid; ++blockIdx.x) {
    uint32_t lo, hi;
    nksplit::share((uint32_t)chunks.size() * blocks, lo, hi);
    std::printf("share %u %u\n", lo, hi);
  }
  return 0;
}
