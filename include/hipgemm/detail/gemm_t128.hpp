// hipgemm -- the 128 x 128 tile schedule (gfx950): the tile schedule of
// gemm_tile.hpp on its smallest tile, with four LDS stages, and the kernel
// that sums its K-slices.  For grids the larger tiles leave underfilled: a 256
// x 256 tile per workgroup leaves most CUs idle when M x N has few tiles
// (2048^3: 64 tiles for 256 CUs).  No reference counterpart:
// fp8_4wave.hpp:334-567 has 256 x 256 tiles only.
#pragma once

#include "gemm_tile.hpp"

namespace hipgemm {
namespace detail {

using CfgT128 = CfgTile<128, 128, 4>;

template <bool kVec, bool kExt = false, int kFmt = 0, int kAct = kActNone,
          int kOut = kOutBf16, bool kSplit = false, bool kMx = false>
__device__ __forceinline__ void gemm_t128_body(const GemmArgs& g, lds_u8* lds) {
  gemm_tile_body<CfgT128, kVec, kExt, kFmt, kAct, kOut, kSplit, kMx>(g, lds);
}

// Sum of the K-slice partials of gemm_t128_body<..., kSplit = true>, in
// slice order 0, 1, ... (the result does not depend on which unit finished
// first), then the epilogue (per-tensor, or the extended one with the
// activation and output type chosen at run time) and the C stores.  One
// wave per workgroup, 16 x tiles workgroups: workgroup b takes rows
// 16 (b % 4) .. + 15 of quadrant (b / 4) % 4 of tile b / 16 (one row of
// four 16 x 16 blocks).  Its loads go out kBatch slices at a time (4 KiB per
// slice and wave), so that a wave has 32 KiB in flight instead of one
// slice: the partials come back from the device-level cache, and with one
// slice in flight per wave (4 waves per tile) the sum of 128 x 8192 x 8192's
// 16 MiB of partials took 11.1 us.  Slices past the last read as +0 (out of
// range), which leaves every sum unchanged (a sum that starts at +0 is never
// -0).  Launched right after the split kernel on the same stream, which makes
// its partials visible.  kVec8: one store per lane and block (N and ldc
// multiples of 4, C aligned to four elements), else one per element.
template <bool kVec8, bool kExt>
__device__ __forceinline__ void gemm_t128_reduce_body(const GemmArgs& g) {
  using Cfg = CfgT128;
  constexpr int kBatch = 8;
  const int lane = lane_id();
  const int M = g.M, N = g.N;
  const int tiles_m = (M + Cfg::kBM - 1) / Cfg::kBM;
  const int tiles_n = (N + Cfg::kBN - 1) / Cfg::kBN;
  const int tiles = tiles_m * tiles_n;
  const int w = (blockIdx.x >> 2) & 3, i = blockIdx.x & 3, t = blockIdx.x >> 4;
  if (t >= tiles) return;
  const int wm = w >> 1, wn = w & 1;
  const TileCoord tc = grouped_tile_u(t, tiles_m, tiles_n, g.group_m);
  const int row0 = tc.m * Cfg::kBM + wm * 64, col0 = tc.n * Cfg::kBN + wn * 64;
  const float s = (g.scale_a ? *g.scale_a : 1.0f) * (g.scale_b ? *g.scale_b : 1.0f);
  EpiVec<4, 4> ev;
  if constexpr (kExt) ev.load(g.epi, M, N, row0, col0, s, lane);
  const int slices = g.split.slices;
  const __amdgpu_buffer_rsrc_t rp = make_rsrc(
      g.split.partial, (uint32_t)tiles * (uint32_t)slices * 65536u);
  f32x4 sum[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] = f32x4{};
  for (int q0 = 0; q0 < slices; q0 += kBatch) {
    f32x4 v[kBatch][4];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int q = q0 + b;
      const uint32_t base =
          q < slices ? (uint32_t)(((q * tiles + t) * 4 + w) * 16384 + 4 * i * 1024 +
                                  lane * 16)
                     : kOobOffset;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[b][j] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, base + j * 1024, 0, 0));
    }
#pragma unroll
    for (int b = 0; b < kBatch; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += v[b][j];
  }
  const int rows_left = M - row0, cols_left = N - col0;
  auto oob_unless = [](int x, int limit) -> uint32_t {
    return (uint32_t)((limit - 1 - x) >> 31) & kOobOffset;
  };
  const int es = kExt ? out_bytes(ev.out) : 2;  // bytes per C element
  const int wrows = min(64, rows_left), wcols = min(64, cols_left);
  const __amdgpu_buffer_rsrc_t rc = make_rsrc(
      reinterpret_cast<uint8_t*>(g.C) + ((size_t)row0 * g.ldc + col0) * es,
      wrows > 0 && wcols > 0 ? (uint32_t)(((wrows - 1) * g.ldc + wcols) * es) : 0u);
  const int r16 = lane & 15, grp = lane >> 4;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4 a = sum[j];
    const int r = 16 * i + r16, col = 16 * j + 4 * grp;
    const uint32_t rb = (uint32_t)((r * g.ldc + col) * es) | oob_unless(r, rows_left);
    if constexpr (kExt) {
      store_out4<kVec8>(ev, a[0], a[1], a[2], a[3], i, j, rc, rb, col, cols_left);
      continue;
    }
    const u32x2 pk = u32x2{pack_bf16x2(a[0] * s, a[1] * s), pack_bf16x2(a[2] * s, a[3] * s)};
    if constexpr (kVec8) {
      __builtin_amdgcn_raw_buffer_store_b64(pk, rc, rb | oob_unless(col, cols_left),
                                            0, 0);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t x = (e < 2 ? pk.x : pk.y) >> (16 * (e & 1));
        __builtin_amdgcn_raw_buffer_store_b16(
            (unsigned short)x, rc, (rb | oob_unless(col + e, cols_left)) + 2 * e, 0, 0);
      }
    }
  }
}

}  // namespace detail
}  // namespace hipgemm
