// Per-row e4m3 quantisation: q = e4m3(clamp(x / s, +-448)), s = amax(|row|)
// / 448 (1 for rows whose largest magnitude is zero or NaN), for fp32, bf16
// and fp16 rows.
//
// What bounds it: one read of x and one write of q.  As tensor operations
// this was seven passes over memory (fp32 copy, abs, amax, the scale, divide,
// clamp, convert) of four bytes per element each; here a workgroup takes a
// row, keeps it in registers between the maximum and the conversion (rows of
// up to 256 * kCache 16-byte loads; longer ones are read again, from the L2),
// and reduces the maximum over its four waves through LDS.  bf16, us per call
// in a graph: 4096 x 8192 215.8 -> 20.2 (5.0 TB/s, what a large copy reaches),
// 2048 x 4096 73.8 -> 9.2, 32 x 4096 25.0 -> 2.8 (launch-bound).
//
// The arithmetic is that of the tensor operations, bit for bit: the scale is
// the maximum times fp32(1 / 448), the quotient a correctly rounded fp32
// division, the conversion rounds to nearest even.  The maximum runs on the
// bit patterns of |x| as integers, which orders NaN above infinity.
#include "kernels.hpp"

namespace hipgemm {
namespace kernels {
namespace {

using namespace detail;

constexpr int kThreads = 256;
constexpr int kCache = 8;  // 16-byte loads of a row a thread keeps
// Rows, and so workgroups, of a launch (one of 2^32 threads is refused).
constexpr int kMaxRows = 1 << 23;

struct QuantArgs {
  const uint8_t* x;
  uint8_t* q;
  float* s;
  int K;
  long long ldx;  // elements
};

template <int kType>  // 0 fp32, 1 bf16, 2 fp16
struct In {
  static constexpr int kBytes = kType == 0 ? 4 : 2;
  static constexpr int kPer = 16 / kBytes;  // elements of a 16-byte load
  __device__ static float one(const uint8_t* p) {
    if constexpr (kType == 0) {
      return *reinterpret_cast<const float*>(p);
    } else {
      const uint16_t b = *reinterpret_cast<const uint16_t*>(p);
      if constexpr (kType == 1) return __builtin_bit_cast(float, (uint32_t)b << 16);
      else return (float)__builtin_bit_cast(_Float16, b);
    }
  }
  __device__ static void eight(const i32x4& v, float (&f)[kPer]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t u = (uint32_t)v[w];
      if constexpr (kType == 0) {
        f[w] = __builtin_bit_cast(float, u);
      } else if constexpr (kType == 1) {
        f[2 * w] = __builtin_bit_cast(float, u << 16);
        f[2 * w + 1] = __builtin_bit_cast(float, u & 0xffff0000u);
      } else {
        f[2 * w] = (float)__builtin_bit_cast(_Float16, (uint16_t)u);
        f[2 * w + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
      }
    }
  }
};

__device__ __forceinline__ uint32_t abs_bits(float x) {
  return __builtin_bit_cast(uint32_t, x) & 0x7fffffffu;
}

// The workgroup's maximum of m, in every lane.
__device__ __forceinline__ uint32_t block_max(uint32_t m) {
  __shared__ uint32_t part[kThreads / kWave];
#pragma unroll
  for (int d = kWave / 2; d > 0; d /= 2)
    m = max(m, (uint32_t)__shfl_xor((int)m, d, kWave));
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / kWave; ++w) m = max(m, part[w]);
  return m;
}

__device__ __forceinline__ float row_scale(uint32_t m) {
  constexpr float kInv = 1.0f / 448.0f;
  return m == 0 || m > 0x7f800000u ? 1.0f : __builtin_bit_cast(float, m) * kInv;
}

// x / s clamped to +-448; a NaN stays one.
__device__ __forceinline__ float scaled(float x, float s) {
  const float v = x / s;
  return v > 448.0f ? 448.0f : v < -448.0f ? -448.0f : v;
}

// Whether a row with largest magnitude m and scale s takes the short division
// below: no Inf or NaN, s normal with room under it (a remainder that
// underflows then belongs to a quotient below 2^-20, which is +-0 in e4m3
// either way), and s's significand not all ones.
__device__ __forceinline__ bool short_division(uint32_t m, float s) {
  const uint32_t b = __builtin_bit_cast(uint32_t, s);
  return m < 0x7f800000u && s >= 0x1p-80f && (b & 0x7fffffu) != 0x7fffffu;
}
// Four x / s clamped and converted, y = 1 / s correctly rounded: the first
// quotient x y is within two ulp, one remainder step brings it within one, and
// the second then rounds x / s correctly (Markstein 1990; the significand of
// all ones, which the theorem leaves out, takes the hardware division).  The
// steps lose the sign of a zero, which is x's.  About 8 instructions per
// element against 25 for the division, clamp and NaN rules in general (with
// those 4096 x 8192 took 34.3 us, 2048 x 4096 13.2).
__device__ __forceinline__ uint32_t quant4(const float* x, float s, float y) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float q = x[e] * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, s, x[e]), y, q);
    q = __builtin_fmaf(__builtin_fmaf(-q, s, x[e]), y, q);
    v[e] = __builtin_copysignf(__builtin_amdgcn_fmed3f(q, -448.0f, 448.0f), x[e]);
  }
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], w, true);
}

// kVec: rows start on 16 bytes and hold a whole number of 16-byte loads, and
// q's rows a whole number of the matching stores.
template <int kType, bool kVec>
__global__ __launch_bounds__(kThreads) void k_quantize_rows(QuantArgs g) {
  using T = In<kType>;
  const uint8_t* x = g.x + (long long)blockIdx.x * g.ldx * T::kBytes;
  uint8_t* q = g.q + (long long)blockIdx.x * g.K;
  uint32_t m = 0;
  if constexpr (kVec) {
    const int n = g.K / T::kPer;  // 16-byte loads of the row
    auto load = [&](int i) { return *reinterpret_cast<const i32x4*>(x + 16ll * i); };
    auto amax = [&](const i32x4& v) {
      float f[T::kPer];
      T::eight(v, f);
#pragma unroll
      for (int e = 0; e < T::kPer; ++e) m = max(m, abs_bits(f[e]));
    };
    i32x4 v[kCache];
#pragma unroll
    for (int c = 0; c < kCache; ++c) {
      const int i = c * kThreads + (int)threadIdx.x;
      v[c] = i < n ? load(i) : i32x4{};
    }
#pragma unroll
    for (int c = 0; c < kCache; ++c) amax(v[c]);
    for (int i = kCache * kThreads + (int)threadIdx.x; i < n; i += kThreads) amax(load(i));
    m = block_max(m);
    const float s = row_scale(m);
    if (threadIdx.x == 0) g.s[blockIdx.x] = s;
    const bool fast = __builtin_amdgcn_readfirstlane((int)short_division(m, s));
    const float y = 1.0f / s;
    auto store = [&](const i32x4& w, int i) {
      float f[T::kPer];
      T::eight(w, f);
      uint32_t r[T::kPer / 4];
      if (fast) {
#pragma unroll
        for (int e = 0; e < T::kPer; e += 4) r[e / 4] = quant4(f + e, s, y);
      } else {
#pragma unroll
        for (int e = 0; e < T::kPer; e += 4)
          r[e / 4] = pack_e4m3x4(f32x4{scaled(f[e], s), scaled(f[e + 1], s),
                                       scaled(f[e + 2], s), scaled(f[e + 3], s)});
      }
      if constexpr (T::kPer == 8)
        *reinterpret_cast<u32x2*>(q + 8ll * i) = u32x2{r[0], r[1]};
      else
        *reinterpret_cast<uint32_t*>(q + 4ll * i) = r[0];
    };
#pragma unroll
    for (int c = 0; c < kCache; ++c) {
      const int i = c * kThreads + (int)threadIdx.x;
      if (i < n) store(v[c], i);
    }
    for (int i = kCache * kThreads + (int)threadIdx.x; i < n; i += kThreads)
      store(load(i), i);
  } else {
    // (unsigned: K may lie within kThreads of 2^31)
    for (unsigned k = threadIdx.x; k < (unsigned)g.K; k += kThreads)
      m = max(m, abs_bits(T::one(x + (long long)k * T::kBytes)));
    const float s = row_scale(block_max(m));
    if (threadIdx.x == 0) g.s[blockIdx.x] = s;
    for (unsigned k = threadIdx.x; k < (unsigned)g.K; k += kThreads) {
      const float f = scaled(T::one(x + (long long)k * T::kBytes), s);
      q[k] = (uint8_t)pack_e4m3x4(f32x4{f, f, f, f});
    }
  }
}

}  // namespace

hipError_t quantize_rows(const void* x, int type, int M, int K, long long ldx,
                         void* q, float* s, hipStream_t stream) {
  QuantArgs g{static_cast<const uint8_t*>(x), static_cast<uint8_t*>(q), s, K, ldx};
  const int es = type == 0 ? 4 : 2;
  const bool vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && ldx * es % 16 == 0 &&
                   K % (16 / es) == 0 &&
                   reinterpret_cast<uintptr_t>(q) % (16 / es) == 0;
  const void* fn = nullptr;
  switch (2 * type + vec) {
    case 0: fn = (const void*)&k_quantize_rows<0, false>; break;
    case 1: fn = (const void*)&k_quantize_rows<0, true>; break;
    case 2: fn = (const void*)&k_quantize_rows<1, false>; break;
    case 3: fn = (const void*)&k_quantize_rows<1, true>; break;
    case 4: fn = (const void*)&k_quantize_rows<2, false>; break;
    case 5: fn = (const void*)&k_quantize_rows<2, true>; break;
    default: return hipErrorInvalidValue;
  }
  void* args[] = {&g};
  // Launches of at most kMaxRows rows (a multiple of 16, so that q keeps its
  // alignment from one to the next).
  for (;;) {
    const int rows = M < kMaxRows ? M : kMaxRows;
    const hipError_t e =
        hipLaunchKernel(fn, dim3((unsigned)rows), dim3(kThreads), args, 0, stream);
    if (e != hipSuccess || (M -= rows) == 0) return e;
    g.x += rows * ldx * es;
    g.q += (long long)rows * K;
    g.s += rows;
  }
}

}  // namespace kernels
}  // namespace hipgemm
