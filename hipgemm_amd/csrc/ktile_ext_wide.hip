// Instantiations of the tile schedule (gemm_tile.hpp) between 128 x 128 and
// 256 x 256, extended epilogue, fp32 and e4m3 output: the 8-bit pairs, with
// one store per lane and block.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

template <class Cfg, int kFmt, int kAct, int kOut>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_tile_ext_wide(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::kLdsBytes];
  gemm_tile_body<Cfg, true, true, kFmt, kAct, kOut>(g, (lds_u8*)lds);
}

}  // namespace

const void* tile_ext_wide(int tile, const Key& k) {
  if (!k.vec) return nullptr;
  return sel_tile(tile, [&](auto cfg) {
    return sel4(k.fmt, [&](auto F) {
      return sel4(k.act, [&](auto A) {
        return sel2(k.out - kOutF32, [&](auto O) {
          return (const void*)&k_fp8_gemm_tile_ext_wide<decltype(cfg), decltype(F)::value,
                                                   decltype(A)::value,
                                                   decltype(O)::value + kOutF32>;
        });
      });
    });
  });
}

}  // namespace kernels
}  // namespace hipgemm
