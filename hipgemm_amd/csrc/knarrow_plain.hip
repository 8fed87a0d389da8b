// Instantiations of the tile schedule (gemm_tile.hpp) on 64-column tiles,
// per-tensor epilogue, bf16 output: the 8-bit pairs.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

template <class Cfg, bool kVec, int kFmt, int kMode>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_narrow(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::kLdsBytes];
  gemm_tile_body<Cfg, kVec, false, kFmt, kActNone, kOutBf16, kMode == kNarrowSplit,
                 false, kMode == kNarrowOnce>(g, (lds_u8*)lds);
}

}  // namespace

const void* narrow_plain(int tile, int mode, const Key& k) {
  return sel_narrow(tile, [&](auto cfg) {
    return sel3(mode, [&](auto S) {
      return sel4(k.fmt, [&](auto F) {
        return sel2(k.vec, [&](auto V) {
          return (const void*)&k_fp8_gemm_narrow<decltype(cfg), decltype(V)::value == 1,
                                                 decltype(F)::value, decltype(S)::value>;
        });
      });
    });
  });
}

}  // namespace kernels
}  // namespace hipgemm
