// The schedules with MX block scales (per-tensor epilogue): the 4-wave
// 16x16x128 one and the 128 x 128 one, and the scale-packing kernel.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

template <bool kVec, int kFmt>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_4wave_mx(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg4w::kLdsBytes];
  gemm_4wave_body<kVec, 16, false, kFmt, kActNone, kOutBf16, true>(g, (lds_u8*)lds);
}

// The 128 x 128 schedule with MX block scales (per-tensor epilogue), for
// every operand-format pair including fp4 x fp4; whole K and K-slices.
template <bool kVec, int kFmt>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_t128_mx(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[CfgT128::kLdsBytes];
  gemm_t128_body<kVec, false, kFmt, kActNone, kOutBf16, false, true>(g, (lds_u8*)lds);
}
template <int kFmt>
__global__ __launch_bounds__(256, 1) void k_fp8_gemm_t128_split_mx(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[CfgT128::kLdsBytes];
  gemm_t128_body<true, false, kFmt, kActNone, kOutBf16, true, true>(g, (lds_u8*)lds);
}

// The packed layout (MxArgs): byte f of step st of lane l in (W, p) is the
// scale of row 128 W + 16 f + l % 16, K-block 4 (2 p + st) + l / 16; 127 (1.0)
// past the rows or blocks of the source.
// One wave per 1 KiB of the packed layout (128 rows W, step pair p): a lane
// loads the 8 scales of rows `lane` and lane + 64, scatters their bytes through
// the wave's 1 KiB of LDS and stores 16 bytes.  kRow8: rows hold eight scales, so
// that one load of eight, at any alignment (the hardware splits it), fetches a
// lane's share: at the end of a row the last eight, shifted.  Else one by one.
// kStore16: the packed buffer starts on 16 bytes.
// Bound by the launch up to about 4096 x 8192, then by the scattered rows'
// reads.  One thread per packed byte did two divisions for one scattered byte
// load; us per packing in a graph of 20, that -> this: 128 x 4096 2.1 level,
// 4096 x 8192 4.0 -> 2.4, 8192 x 8192 6.0 -> 2.7, 28672 x 8320 20.1 -> 7.0, 2048
// x 4160 (odd row starts) 2.4 -> 2.3; behind only by the second load's latency
// where little is packed: 512 x 4128 2.2 -> 2.3, 4096 x 128 2.1 -> 2.5.
template <bool kRow8, bool kStore16>
__global__ __launch_bounds__(256) void k_mx_pack(const uint8_t* src, int rows,
                                                 int kblocks, int ld, int pairs,
                                                 uint8_t* dst, int chunks) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[4 * 1024];
  const int lane = lane_id(), wave = wave_id();
  const int chunk = blockIdx.x * 4 + wave;
  if (chunk >= chunks) return;
  const int W = chunk / pairs, p = chunk % pairs;
  uint8_t* mine = lds + wave * 1024;
  const int left = kblocks - 8 * p;  // scales of a row from here on, at least one
  uint64_t v[2] = {0x7f7f7f7f7f7f7f7full, 0x7f7f7f7f7f7f7f7full};  // padding: 1.0
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 128 * W + 64 * h + lane;
    const uint8_t* s = src + (size_t)row * ld + 8 * p;
    if (row >= rows) continue;
    if constexpr (kRow8) {
      __builtin_memcpy(&v[h], s - (left < 8 ? 8 - left : 0), 8);
    } else {
      uint8_t one[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) one[b] = s[b < left ? b : 0];
      v[h] = 0;
#pragma unroll
      for (int b = 0; b < 8; ++b) v[h] |= (uint64_t)(b < left ? one[b] : 127) << (8 * b);
    }
  }
  if (kRow8 && left < 8) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      v[h] = v[h] >> (8 * (8 - left)) | 0x7f7f7f7f7f7f7f7full << (8 * left);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    // Block b of the pair: step b / 4, lane group b % 4.
    const int r = 64 * h + lane, f = r >> 4;
#pragma unroll
    for (int b = 0; b < 8; ++b)
      mine[((b & 3) * 16 + (r & 15)) * 16 + (b >> 2) * 8 + f] = (uint8_t)(v[h] >> (8 * b));
  }
  // The wave's own region: its LDS operations complete in order.
  compiler_fence();
  uint8_t* to = dst + (size_t)chunk * 1024;
  if constexpr (kStore16) {
    *reinterpret_cast<i32x4*>(to + lane * 16) = lds_read16((lds_u8*)mine + lane * 16);
  } else {
#pragma unroll
    for (int b = 0; b < 16; ++b) to[64 * b + lane] = mine[64 * b + lane];
  }
}

}  // namespace

const void* four_wave_mx(const Key& k) {
  // The 8-bit pairs and fp4 x fp4 (MXFP4).
  return sel_fmt(k.fmt, [&](auto F) {
    return sel2(k.vec, [&](auto V) {
      return (const void*)&k_fp8_gemm_4wave_mx<decltype(V)::value == 1,
                                               decltype(F)::value>;
    });
  });
}

const void* tile128_mx(const Key& k) {
  return sel_fmt(k.fmt, [&](auto F) {
    return sel2(k.vec, [&](auto V) {
      return (const void*)&k_fp8_gemm_t128_mx<decltype(V)::value == 1,
                                              decltype(F)::value>;
    });
  });
}

const void* tile128_split_mx(const Key& k) {
  return sel_fmt(k.fmt, [&](auto F) {
    return (const void*)&k_fp8_gemm_t128_split_mx<decltype(F)::value>;
  });
}

hipError_t mx_pack(const uint8_t* src, int rows, int K, int ld, uint8_t* dst,
                   hipStream_t stream) {
  const size_t n = mx_packed_bytes(rows, K);
  if (n == 0) return hipSuccess;
  int kblocks = (K + 31) / 32, pairs = mx_pairs(K), chunks = (int)(n / 1024);
  const void* fn = sel2(kblocks >= 8, [&](auto R) {
    return sel2(reinterpret_cast<uintptr_t>(dst) % 16 == 0, [&](auto S) {
      return (const void*)&k_mx_pack<decltype(R)::value == 1, decltype(S)::value == 1>;
    });
  });
  void* args[] = {&src, &rows, &kblocks, &ld, &pairs, &dst, &chunks};
  return hipLaunchKernel(fn, dim3((unsigned)((chunks + 3) / 4)), dim3(256), args, 0,
                         stream);
}

}  // namespace kernels
}  // namespace hipgemm
