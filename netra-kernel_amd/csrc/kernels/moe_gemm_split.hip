// Grouped gate/up with the expert weights streamed once and the work divided
// evenly over the chip, for experts of a few rows each: past the decode sizes
// of the merged kernel (T = 65 and up at 256 experts, top-8) to the sizes
// where the block-pair LDS kernel has rows enough to be compute-bound.
//
// An expert's n sorted rows are cut into chunks of at most four 16-row tiles
// (nc = ceil(ceil(n / 16) / 4) chunks of nearly equal tile counts). The
// 128-column blocks of h of all chunks, in expert order, are dealt in
// contiguous runs of equal length to one workgroup per CU (workgroups of one
// XCD side by side). What bounds it is the weight stream (one read of W13 at
// 6.5 TB/s: 83 us for the 540 MB of 257 experts at H 2048, I 512). The items
// of the stream kernel cover a 16-row tile of up to 512 columns each, so 260
// tiles on 256 workgroups ran two rounds, the second nearly empty, and the
// block-pair kernel ends an item with ~6 us in which it requests nothing.
// Measured on one MI355X, gate/up us, that kernel / this one: T = 80 88.1 /
// 82.2, 100 93.2 / 84.6, 128 112.8 / 89.3, 192 115.3 / 98, 256 120.9 / 100
// (stream); T = 257 109.2 / 93.5, 400 110.8 / 96.3 (block pairs). Skewed
// routing (Zipf 1.1): T = 100 33.6 / 28.0, 192 52.1 / 45.4, 400 46.8 / 42.8,
// but 512 46.0 / 53.0 (uniform routing there: 111 / 96): an expert of hundreds
// of rows is many chunks here, each with a K-split sum per 64 rows, and the
// block pairs serve it better. The engine's rule (engine.py, split_gate_up)
// ends at 13 routed rows per expert, and leaves few-row calls to the others.
//
//   netra_moe_gate_up_split_h<H>_{tiles|rows}_gfx950(xq, xs, w13, w13s,
//       sorted_ids, counts, hq, hs; T, I, Etot, CAP)   grid 256, block 512
//
// The chunk table comes from the sort's expert counts (a scan of at most 513
// entries by the first wave), the rows from sorted_ids; expert e's rows begin
// at 64 times the number of 64-row blocks before it.
//
// (reference: kernels/gfx950/templates/moe/decode/gate_up_mfma.inc:12-161,
// silu_quant.inc:16-236)
#pragma once
#include <type_traits>

#include "moe_ffn_decode.hip"
#include "moe_numerics.h"
#include "moe_split_table.h"

#define NK_KERNEL extern "C" __global__

namespace nksplit {

using nk::v4f;
using nk::v8i;
using nkstream::lds_barrier;

__device__ __forceinline__ float lane_f32(float v, uint32_t l) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), (int)l));
}

// ---------------------------------------------------------------------------
// The K blocks are split over the eight waves (wave w: K blocks KBW w ..), and
// every wave keeps its K slice of the chunk's activation rows in registers as MFMA operands for as long as the
// workgroup stays on the chunk: an item (16 gate and 16 up rows of W13 over
// all of K, 64 KiB at H = 2048) is read once, straight into registers, for up
// to 64 rows, and nothing but weights moves per item. The waves' split sums
// meet in LDS (two buffers, one barrier per item); one wave per row tile adds
// them in wave order, applies SiLU.mul and writes bf16 h to the LDS rows of
// the current 128-column block, which is requantised (1x128) when complete.
// (Chunks of eight tiles halve the weight reads of many-row experts but not
// the sums, 256 KiB of LDS traffic per item: 3.4 us per item against 2.5 us of
// weight stream, and the workgroups of the shared expert ended last: T = 192
// 143 us.)
//
// A position is two items, one per weight buffer; each half of a buffer is
// refilled for the next position right after its last MFMA, so 1.5 to 2 items
// per wave are in flight. Past the share's end in the chunk the resource has
// no bytes and the loads return zeros without an access (no load is under a
// branch). Weights are read non-temporally (98 us against 113 with ordinary
// loads at T = 192).
constexpr uint32_t kGuWaves = 8;
constexpr uint32_t RM = 4;  // 16-row tiles per chunk

template <uint32_t KBW>
struct GuBuf {
  v8i g[KBW], u[KBW];
  float ws;  // lanes 0 .. KBW - 1: gate block scales, KBW .. 2 KBW - 1: up
};

template <uint32_t KB, bool kHw, bool kRowMajor>
__device__ __forceinline__ void gate_up_split(
    const uint8_t* __restrict__ xq, const float* __restrict__ xs, const uint8_t* __restrict__ w13,
    const float* __restrict__ w13s, const int32_t* __restrict__ sorted_ids, const int32_t* __restrict__ counts,
    uint8_t* __restrict__ hq, float* __restrict__ hs, uint32_t T, uint32_t I, uint32_t Etot, uint32_t cap_blocks) {
  static_assert(KB % kGuWaves == 0, "a whole number of K blocks per wave");
  constexpr uint32_t KBW = KB / kGuWaves;
  constexpr uint32_t H = 128u * KB;
  constexpr uint32_t kBufF4 = kGuWaves * 2u * RM * 64u;  // float4 per split-sum buffer
  __shared__ Table s_tab;
  __shared__ __align__(16) float4 s_red[2u * kBufF4];
  constexpr uint32_t kHStride = 128u + 8u;                 // bf16 per LDS h row (+16 bytes rotates banks)
  __shared__ __align__(16) uint16_t s_h[RM * 16u * kHStride];  // a 128-column block of h
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = nkstream::wave_id();
  if (Etot == 0u || Etot > kMaxE) return;  // host-checked
  if (wave == 0) build_table<RM>(s_tab, counts, T, Etot, lane);
  __syncthreads();
  const uint32_t UP = I / 32u;  // positions per chunk
  uint32_t lo, hi;
  // (in whole 128-column blocks of h, which the workgroup requantises)
  constexpr uint32_t GP = 4u;  // positions per block
  share(all_chunks(s_tab, Etot) * (UP / GP), lo, hi);
  lo *= GP;
  hi *= GP;
  if (lo >= hi) return;  // uniform

  const uint32_t g4 = lane >> 4;
  const uint32_t kb0 = wave * KBW;
  Chunk ck = locate(s_tab, lo / UP, Etot, lane);
  const uint32_t scale_lane = lane < 2u * KBW ? lane : 0u;
  const uint32_t scale_row = (scale_lane < KBW ? 0u : I / 128u) * KB + kb0 + scale_lane % KBW;

  const __amdgpu_buffer_rsrc_t xr = nk::buffer_rsrc(xq, T * H), sr = nk::buffer_rsrc(xs, T * KB * 4u);
  uint32_t rot = 0, par = 0;  // rotation of the adding waves, split-sum buffer
  uint32_t pos = lo;
  auto run = [&](auto rc) __attribute__((always_inline)) {
    constexpr uint32_t R = decltype(rc)::value;
    const uint8_t* we = w13 + (size_t)ck.e * 2u * I * H;
    const float* wse = w13s + (size_t)ck.e * (2u * I / 128u) * KB + scale_row;
    const uint32_t end = min(hi, (ck.first + 1u) * UP);
    GuBuf<KBW> b0, b1;
    // column item 2 ip + j of the chunk into a buffer (its number opaque: with an
    // induction variable for every tile's offset a call measured 0.3% more)
    auto column = [&](uint32_t ip, uint32_t j) __attribute__((always_inline)) {
      uint32_t c = 2u * ip + j;
      asm("" : "+s"(c));
      return c;
    };
    auto issue_g = [&](GuBuf<KBW>& b, uint32_t ip, uint32_t j, bool live) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t r = nk::buffer_rsrc(we, live ? 2u * I * H : 0u);
      const uint32_t c = column(ip, j);
      b.ws = wse[(live ? c >> 3 : 0u) * KB];  // (ahead of the tiles it scales)
#pragma unroll
      for (uint32_t i = 0; i < KBW; ++i) b.g[i] = nk::load_tile_operand<false, true>(r, (2u * c * KB + kb0 + i) * 2048u, lane);
    };
    auto issue_u = [&](GuBuf<KBW>& b, uint32_t ip, uint32_t j, bool live) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t r = nk::buffer_rsrc(we, live ? 2u * I * H : 0u);
      const uint32_t c = column(ip, j);
#pragma unroll
      for (uint32_t i = 0; i < KBW; ++i) b.u[i] = nk::load_tile_operand<false, true>(r, ((2u * c + 1u) * KB + kb0 + i) * 2048u, lane);
    };
    // the chunk's rows: lane l holds row l & 15 of every tile
    v8i a[R][KBW];
    float as[R][KBW];
    uint32_t t[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
      t[r] = (uint32_t)sorted_ids[ck.row0 + 16u * min(r, ck.tiles - 1u) + (lane & 15u)] & 0xffffffu;
    __builtin_amdgcn_sched_barrier(0);
    auto first = [&]() __attribute__((always_inline)) {
      const uint32_t p = pos - ck.first * UP;
      issue_g(b0, p, 0u, true);
      issue_u(b0, p, 0u, true);
      issue_g(b1, p, 1u, true);
      issue_u(b1, p, 1u, true);
      __builtin_amdgcn_sched_barrier(0);
    };
    first();
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) t[r] = t[r] < T ? t[r] : 0u;  // padding rows: any row, their h is never used
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
#pragma unroll
      for (uint32_t i = 0; i < KBW; ++i) {  // (T * H below 2^31, host-checked: one 32-bit offset per row)
        const nk::u32x4 al = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(t[r] * H + g4 * 32u), (int)((kb0 + i) * 128u), 0);
        const nk::u32x4 ah = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(t[r] * H + g4 * 32u + 16u), (int)((kb0 + i) * 128u), 0);
        a[r][i] = v8i{(int)al.x, (int)al.y, (int)al.z, (int)al.w, (int)ah.x, (int)ah.y, (int)ah.z, (int)ah.w};
        as[r][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sr, (int)(t[r] * KB * 4u), (int)((kb0 + i) * 4u), 0));
      }
    // the rows have arrived (and the older weights with them) before the loop:
    // pending at its head, they would put a full drain into every iteration
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
#pragma unroll
      for (uint32_t i = 0; i < KBW; ++i) {
        asm volatile("" : "+v"(a[r][i]), "+v"(as[r][i]));
      }
#pragma unroll 1
    for (; pos < end; ++pos) {
      const uint32_t p = pos - ck.first * UP;
      const bool live = pos + 1u < end;
      auto item = [&](GuBuf<KBW>& b, uint32_t j) __attribute__((always_inline)) {
        float sg[KBW], su[KBW];
#pragma unroll
        for (uint32_t i = 0; i < KBW; ++i) {
          sg[i] = lane_f32(b.ws, i);
          su[i] = lane_f32(b.ws, KBW + i);
        }
        float4* const red = s_red + par * kBufF4;
        // two row tiles at a time: their MFMAs are issued back to back and
        // scaled while the next pair's run (one at a time the chain of MFMA,
        // scale and LDS write set the time of a many-tile chunk: 140 us for
        // the shared expert at T = 128, against 85 us for every other share)
        auto part = [&](const v8i (&w)[KBW], const float (&ws)[KBW], uint32_t gu) __attribute__((always_inline)) {
#pragma unroll
          for (uint32_t r = 0; r < R; r += 2u) {
            v4f d[2][KBW];
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h)
#pragma unroll
              for (uint32_t i = 0; i < KBW; ++i)
                if (r + h < R) d[h][i] = nk::mfma_e4m3_16x16x128(w[i], a[r + h][i]);
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
              if (r + h < R) {
                v4f acc;
#pragma unroll
                for (uint32_t i = 0; i < KBW; ++i) {
                  const float s = ws[i] * as[r + h][i];
#pragma unroll
                  for (uint32_t q = 0; q < 4; ++q) acc[q] = i == 0 ? s * d[h][i][q] : fmaf(s, d[h][i][q], acc[q]);
                }
                red[((wave * 2u + gu) * RM + r + h) * 64u + lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
              }
            }
          }
        };
        part(b.g, sg, 0u);
        __builtin_amdgcn_sched_barrier(0);
        issue_g(b, p + 1u, j, live);
        part(b.u, su, 1u);
        __builtin_amdgcn_sched_barrier(0);
        issue_u(b, p + 1u, j, live);
        lds_barrier();  // (the other buffer was read before the previous barrier)
        // one wave per row tile adds the split sums in order
        const uint32_t r = (wave - rot) & (kGuWaves - 1u);
        if (r < R) {
          v4f gs, us;
#pragma unroll
          for (uint32_t w = 0; w < kGuWaves; ++w) {
            const float4 x = red[((w * 2u) * RM + r) * 64u + lane];
            const float4 y = red[((w * 2u + 1u) * RM + r) * 64u + lane];
            const v4f xv = {x.x, x.y, x.z, x.w}, yv = {y.x, y.y, y.z, y.w};
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
              gs[q] = w == 0 ? xv[q] : gs[q] + xv[q];
              us[q] = w == 0 ? yv[q] : us[q] + yv[q];
            }
            // (a few reads in flight: all sixteen would take 64 registers)
            if (w % 4u == 3u) asm volatile("" : "+v"(gs), "+v"(us) : : "memory");
          }
#pragma unroll
          for (uint32_t q = 0; q < 4; ++q) us[q] = (kHw ? nk::silu_hw(gs[q]) : nk::silu(gs[q])) * us[q];
          const uint32_t col = ((2u * p + j) & 7u) * 16u + g4 * 4u;
          *reinterpret_cast<uint2*>(&s_h[(r * 16u + (lane & 15u)) * kHStride + col]) =
              make_uint2(nk::bf16x2_hw(us[0], us[1]), nk::bf16x2_hw(us[2], us[3]));
        }
        rot += R;
        par ^= 1u;
      };
      item(b0, 0u);
      item(b1, 1u);
      if ((p + 1u) % GP == 0u) {  // uniform: a 128-column block of h is complete
        lds_barrier();
        if (wave < R) {  // (its rows are read before the next item's barrier, and written after it)
          const uint4* src = reinterpret_cast<const uint4*>(&s_h[(wave * 16u + (lane & 15u)) * kHStride + g4 * 32u]);
          uint32_t raw[16];
#pragma unroll
          for (uint32_t q = 0; q < 4; ++q) {
            const uint4 v = src[q];
            raw[4 * q] = v.x; raw[4 * q + 1] = v.y; raw[4 * q + 2] = v.z; raw[4 * q + 3] = v.w;
          }
          uint4 qlo, qhi;
          float scale;
          nkffn::quant_block(raw, qlo, qhi, scale);
          const size_t row = ck.row0 + 16u * wave;
          const uint32_t kb = p / GP, KBI = I / 128u;
          if constexpr (kRowMajor) {
            uint8_t* d = hq + (row + (lane & 15u)) * I + kb * 128u + g4 * 32u;
            *reinterpret_cast<uint4*>(d) = qlo;
            *reinterpret_cast<uint4*>(d + 16) = qhi;
            if (lane < 16u) hs[(row + lane) * KBI + kb] = scale;
          } else {
            uint8_t* d = hq + ((row >> 4) * KBI + kb) * 2048u + lane * 16u;
            *reinterpret_cast<uint4*>(d) = qlo;
            *reinterpret_cast<uint4*>(d + 1024) = qhi;
            if (lane < 16u) hs[((row >> 4) * KBI + kb) * 16u + lane] = scale;
          }
        }
      }
    }
  };
#pragma unroll 1
  while (pos < hi) {
    // malformed counts; uniform
    if (ck.tiles - 1u >= RM || ck.row0 + ck.tiles * 16u > cap_blocks * 64u) return;
    switch (ck.tiles) {
      case 1: run(std::integral_constant<uint32_t, 1>{}); break;
      case 2: run(std::integral_constant<uint32_t, 2>{}); break;
      case 3: run(std::integral_constant<uint32_t, 3>{}); break;
      default: run(std::integral_constant<uint32_t, 4>{}); break;
    }
    if (pos < hi) ck = locate(s_tab, ck.first + 1u, Etot, lane);
  }
}

}  // namespace nksplit

#define NK_GATE_UP_SPLIT(HV, NAME, HW, ROWS)                                                        \
  NK_KERNEL __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))                          \
  void netra_moe_gate_up_split_h##HV##_##NAME##_gfx950(                                             \
      const uint8_t* __restrict__ xq, const float* __restrict__ xs, const uint8_t* __restrict__ w13, \
      const float* __restrict__ w13s, const int32_t* __restrict__ sorted_ids,                       \
      const int32_t* __restrict__ counts, uint8_t* __restrict__ hq, float* __restrict__ hs,         \
      uint32_t T, uint32_t I, uint32_t Etot, uint32_t cap_blocks) {                                 \
    nksplit::gate_up_split<HV / 128, HW, ROWS>(xq, xs, w13, w13s, sorted_ids, counts, hq, hs, T, I, \
                                               Etot, cap_blocks);                                   \
  }
// _tiles: h in the stream path's layout; _rows: row-major, as the tile path's
NK_GATE_UP_SPLIT(2048, tiles, false, false)
NK_GATE_UP_SPLIT(2048, rows, true, true)
