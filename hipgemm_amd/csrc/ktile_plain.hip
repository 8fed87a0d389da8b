// Instantiations of the tile schedule (gemm_tile.hpp) between 128 x 128 and
// 256 x 256, per-tensor epilogue, bf16 output: the 8-bit pairs.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

template <class Cfg, bool kVec, int kFmt>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_tile(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::kLdsBytes];
  gemm_tile_body<Cfg, kVec, false, kFmt>(g, (lds_u8*)lds);
}

}  // namespace

const void* tile_plain(int tile, const Key& k) {
  return sel_tile(tile, [&](auto cfg) {
    return sel4(k.fmt, [&](auto F) {
      return sel2(k.vec, [&](auto V) {
        return (const void*)&k_fp8_gemm_tile<decltype(cfg), decltype(V)::value == 1,
                                             decltype(F)::value>;
      });
    });
  });
}

}  // namespace kernels
}  // namespace hipgemm
