// Symmetric quantization of activations: what the quantizer kernels
// (rnsmx_kernels.hip) and the one-launch decode layer (rnsmx_linear.hip) share.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "rnsmx_gemm.hpp"

namespace rnsmx {

struct QuantArgs {
  const void *x;
  int64_t count;
  int32_t vec;      // 1: x is 16-byte aligned, read in 16-byte vectors
  int32_t nparts;   // blocks of the amax pass
  float qmax, rcp;  // rcp = fl32(1 / qmax)
  float *partial;
  float *scale;
  void *q;
};

// Input element decoding: float32, or the bits of a float16 / bfloat16.
template <typename T>
struct QuantIn;
template <>
struct QuantIn<float> {
  __device__ static float get(float v) { return v; }
};
struct Bf16Bits {
  uint16_t bits;
};
template <>
struct QuantIn<__half> {
  __device__ static float get(uint16_t v) { return __half2float(__ushort_as_half(v)); }
};
template <>
struct QuantIn<Bf16Bits> {
  __device__ static float get(uint16_t v) { return __uint_as_float(static_cast<uint32_t>(v) << 16); }
};
template <typename T>
using QuantRaw = typename std::conditional<std::is_same<T, float>::value, float, uint16_t>::type;

// max(a, b) that propagates NaN, as torch's amax does (fmaxf drops it).
__device__ __forceinline__ float max_nan(float a, float b) {
  return (a != a || b != b) ? __builtin_nanf("") : fmaxf(a, b);
}

// max |x| over the elements this thread visits (tid, tid + stride, ...);
// NaN when any of them is NaN.
template <typename T>
__device__ __forceinline__ float quant_thread_amax(const QuantArgs &a, int64_t tid, int64_t stride) {
  using R = QuantRaw<T>;
  constexpr int V = 16 / sizeof(R);
  const R *x = static_cast<const R *>(a.x);
  const int64_t nvec = a.vec ? a.count / V : 0;
  float m = 0.0f;
  bool nan = false;
  auto visit = [&](float v) {
    m = fmaxf(m, fabsf(v));
    nan |= v != v;
  };
  for (int64_t i = tid; i < nvec; i += stride) {
    R v[V];
    *reinterpret_cast<uint4 *>(v) = reinterpret_cast<const uint4 *>(x)[i];
    static_for<V>([&](auto E) { visit(QuantIn<T>::get(v[decltype(E)::value])); });
  }
  for (int64_t i = nvec * V + tid; i < a.count; i += stride) visit(QuantIn<T>::get(x[i]));
  return nan ? __builtin_nanf("") : m;
}

// The scale from the largest |x|: amax / qmax as a multiply by fl32(1 / qmax),
// at least FLT_EPSILON; NaN stays NaN (torch.clamp keeps it, fmaxf would not).
__device__ __forceinline__ float quant_scale(float amax, float rcp) {
  return amax != amax ? amax : fmaxf(amax * rcp, 1.1920928955078125e-07f);
}

// clamp(rint(v / s), -qmax, qmax), the division correctly rounded.  A NaN
// quotient (v NaN, s NaN, or v and s infinite) quantizes to 0, the value the
// hardware's float-to-integer conversion gives NaN.
__device__ __forceinline__ float quant_value(float v, float s, float qmax) {
  const float r = rintf(v / s);
  return r != r ? 0.0f : fminf(fmaxf(r, -qmax), qmax);
}

// The decode layer in one launch (rnsmx_linear.hip): whether it serves a call,
// and its launch (g: shape, weight and epilogue; q: x, vec, qmax, rcp).
// aligned: the activations start on a 16-byte boundary.
bool linear_rows_fits(int64_t rows, int64_t k, int64_t n, const rnsmx_moduli_t &mods, int32_t quant_bits,
                      bool adaptive, bool aligned);
void launch_linear_rows(const GemmArgs &g, const QuantArgs &q, int32_t x_dtype, hipStream_t st);

// Requests of a few int8 rows in one launch (rnsmx_linear.hip): row[i] the
// 16-byte aligned row i < g.m, copied to staging [m][K] too.
bool request_rows_fits(int64_t rows, int64_t k, const rnsmx_moduli_t &mods, int32_t a_dtype);
void launch_request_rows(const GemmArgs &g, const int8_t *const *row, int8_t *staging, hipStream_t st);

}  // namespace rnsmx
