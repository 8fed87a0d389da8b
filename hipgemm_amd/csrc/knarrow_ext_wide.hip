// Instantiations of the tile schedule (gemm_tile.hpp) on 64-column tiles,
// extended epilogue, fp32 and e4m3 output: the 8-bit pairs, with one store per
// lane and block, one K-slice.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

template <class Cfg, int kFmt, int kAct, int kOut, int kMode>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_narrow_ext_wide(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::kLdsBytes];
  gemm_tile_body<Cfg, true, true, kFmt, kAct, kOut, false, false,
                 kMode == kNarrowOnce>(g, (lds_u8*)lds);
}

}  // namespace

const void* narrow_ext_wide(int tile, int mode, const Key& k) {
  if (!k.vec || mode == kNarrowSplit) return nullptr;
  return sel_narrow(tile, [&](auto cfg) {
    return sel2(mode, [&](auto S) {
      return sel4(k.fmt, [&](auto F) {
        return sel4(k.act, [&](auto A) {
          return sel2(k.out - kOutF32, [&](auto O) {
            return (const void*)&k_fp8_gemm_narrow_ext_wide<
                decltype(cfg), decltype(F)::value, decltype(A)::value,
                decltype(O)::value + kOutF32, decltype(S)::value>;
          });
        });
      });
    });
  });
}

}  // namespace kernels
}  // namespace hipgemm
