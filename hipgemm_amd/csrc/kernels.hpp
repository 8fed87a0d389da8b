// Kernel lookup across the library's translation units.  Each schedule's
// instantiations live in their own file (compiled in parallel); the C ABI
// (hipgemm.hip) asks here for the entry point of one configuration.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "hipgemm/detail/gemm_8wave.hpp"
#include "hipgemm/detail/gemm_skinny.hpp"
#include "hipgemm/detail/gemm_strip.hpp"
#include "hipgemm/detail/gemm_t128.hpp"

namespace hipgemm {
namespace kernels {

// One configuration: operand formats (bit 0 A, bit 1 B_T), extended
// epilogue, its activation and output type, the store width (16 bytes per
// lane for the tiled schedules, 8 for the skinny one), and whether C's rows
// start on 128-byte lines (the 4-wave schedule's overlapped epilogue).
struct Key {
  int fmt = 0;
  bool ext = false;
  int act = 0;
  int out = 0;
  bool vec = true;
  bool line = false;
};

// Entry points (host handles for hipLaunchKernel), nullptr for a
// configuration that is not built.
const void* four_wave_plain(int mf, const Key& k);  // k4wave_plain.hip
const void* four_wave_ext_bf16(const Key& k);       // k4wave_ext_bf16.hip
const void* four_wave_ext_f16(const Key& k);        // k4wave_ext_f16.hip
const void* four_wave_ext_f32(const Key& k);        // k4wave_ext_f32.hip
const void* four_wave_ext_f8(const Key& k);         // k4wave_ext_f8.hip
const void* eight_wave_plain(const Key& k);         // k8wave_plain.hip
const void* eight_wave_ext_bf16(const Key& k);      // k8wave_ext_bf16.hip
const void* eight_wave_ext_f16(const Key& k);       // k8wave_ext_f16.hip
const void* skinny_plain(int kmb, int kf, const Key& k);  // kskinny_plain.hip
const void* skinny_ext(int kmb, int kf, const Key& k);    // kskinny_ext.hip
const void* skinny_reduce(int kf, const Key& k);    // kskinny_plain.hip
const void* strip_plain(int kmb, int knb, const Key& k);  // kstrip_plain.hip
const void* strip_ext(int kmb, int knb, const Key& k);    // kstrip_ext.hip
const void* four_wave_mx(const Key& k);             // k4wave_mx.hip
const void* tile128_mx(const Key& k);               // k4wave_mx.hip
const void* tile128_split_mx(const Key& k);         // k4wave_mx.hip
const void* tile128_plain(const Key& k);            // kt128_plain.hip
const void* tile128_ext_narrow(const Key& k);       // kt128_ext.hip
const void* tile128_ext_wide(const Key& k);         // kt128_ext_wide.hip
inline const void* tile128_ext(const Key& k) {
  return k.out >= detail::kOutF32 ? tile128_ext_wide(k) : tile128_ext_narrow(k);
}
const void* tile128_split(const Key& k);            // kt128_plain.hip
const void* tile128_reduce(const Key& k);           // kt128_plain.hip
const void* split_plain(const Key& k);              // ksplit_plain.hip
const void* tile_plain(int tile, const Key& k);     // ktile_plain.hip
const void* tile_ext_narrow(int tile, const Key& k);  // ktile_ext.hip
const void* tile_ext_wide(int tile, const Key& k);    // ktile_ext_wide.hip
// 64-column tiles.  mode: one K-slice, one with B_T read once (kNt), or
// K-slices.
enum { kNarrowWhole = 0, kNarrowOnce = 1, kNarrowSplit = 2 };
const void* narrow_plain(int tile, int mode, const Key& k);       // knarrow_plain.hip
const void* narrow_ext(int tile, int mode, const Key& k);         // knarrow_ext.hip
const void* narrow_ext_wide(int tile, int mode, const Key& k);    // knarrow_ext_wide.hip
// hipgemm_gemm_noalloc's static scratch array on the current device
// (noalloc_scratch.hip): its address, looked up once per device (with that
// device current); at that first lookup its counter region is cleared on
// `stream` unless the stream is being captured.  nullptr with *err set on
// failure.
void* noalloc_scratch(hipStream_t stream, hipError_t* err);
// Per-row e4m3 quantisation (kquant.hip); type: HIPGEMM_IN_*.
hipError_t quantize_rows(const void* x, int type, int M, int K, long long ldx,
                         void* q, float* s, hipStream_t stream);
// Packs [rows][ceil(K/32)] E8M0 scales (row stride ld) into MxArgs' layout.
hipError_t mx_pack(const uint8_t* src, int rows, int K, int ld, uint8_t* dst,
                   hipStream_t stream);

// Runtime value -> integral_constant, for building the lookups.
template <int I>
using ic = std::integral_constant<int, I>;
template <class F>
const void* sel2(int v, F&& f) {
  return v ? f(ic<1>{}) : f(ic<0>{});
}
// Operand-format pairs: the four 8-bit pairs and fp4 x fp4 (kFmtPairFp4).
template <class F>
const void* sel_fmt(int v, F&& f) {
  switch (v) {
    case 0: return f(ic<0>{});
    case 1: return f(ic<1>{});
    case 2: return f(ic<2>{});
    case 3: return f(ic<3>{});
    case 4: return f(ic<4>{});
    default: return nullptr;
  }
}
// The pairs of sel_fmt and fp6 x fp6 (kFmtPairFp6 + 0..3): the 128 x 128
// schedule's, and the 4-wave schedule's with the per-tensor epilogue.
template <class F>
const void* sel_fmt_t128(int v, F&& f) {
  switch (v) {
    case 8: return f(ic<8>{});
    case 9: return f(ic<9>{});
    case 10: return f(ic<10>{});
    case 11: return f(ic<11>{});
    default: return sel_fmt(v, f);
  }
}
template <class F>
const void* sel4(int v, F&& f) {
  switch (v) {
    case 0: return f(ic<0>{});
    case 1: return f(ic<1>{});
    case 2: return f(ic<2>{});
    case 3: return f(ic<3>{});
    default: return nullptr;
  }
}

// The tiles between 128 x 128 and 256 x 256, and the 64-column ones.
struct TileShape {
  int bm, bn;
};
constexpr int kNumTiles = 3, kNumNarrow = 2;
constexpr TileShape kTiles[kNumTiles] = {{128, 256}, {192, 192}, {192, 128}};
constexpr TileShape kNarrow[kNumNarrow] = {{128, 64}, {64, 64}};
template <class F>
const void* sel_tile(int t, F&& f) {
  switch (t) {
    case 0: return f(detail::CfgTile<kTiles[0].bm, kTiles[0].bn, 3>{});
    case 1: return f(detail::CfgTile<kTiles[1].bm, kTiles[1].bn, 3>{});
    case 2: return f(detail::CfgTile<kTiles[2].bm, kTiles[2].bn, 3>{});
    default: return nullptr;
  }
}
// Six LDS stages (144 and 96 KiB): these tiles are streams over B_T.
template <class F>
const void* sel_narrow(int t, F&& f) {
  switch (t) {
    case 0: return f(detail::CfgTile<kNarrow[0].bm, kNarrow[0].bn, 6>{});
    case 1: return f(detail::CfgTile<kNarrow[1].bm, kNarrow[1].bn, 6>{});
    default: return nullptr;
  }
}
template <class F>
const void* sel3(int v, F&& f) {
  return v == 0 ? f(ic<0>{}) : v == 1 ? f(ic<1>{}) : v == 2 ? f(ic<2>{}) : nullptr;
}

}  // namespace kernels
}  // namespace hipgemm
