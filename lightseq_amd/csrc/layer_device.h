// Device functions of the quantised layer path, shared by its stand-alone operators (layer_ops.hip)
// and the epilogues and launches they are fused into (layer_gemm.hip, layer_fused.hip).
#pragma once
#include "ls_device.h"

namespace lsh {

constexpr float kQ = 127.0f;               // kernels.h:20
constexpr float kLnEps = 1e-8f;            // normalize_kernels.cu:12
constexpr float kSoftmaxEps = 1e-8f;       // softmax_kernels.cu:11

// kernels.h:425-435
__device__ __forceinline__ int clip_mask_bits(float v, float cmax, int bit, bool symmetry = true) {
  if (v >= cmax) return 1 << (bit - 1);
  if (symmetry && v <= -cmax) return 1 << bit;
  return 0;
}
// kernels.h:463-471
__device__ __forceinline__ int quantize_b(float x, float cmax, int& mask, int bit) {
  mask = clip_mask_bits(x, cmax, bit);
  const float scale = cmax / kQ;
  const float q = floorf(x / scale + 0.5f);
  return (int)fminf(fmaxf(q, -kQ), kQ);
}
// kernels.h:473-488
__device__ __forceinline__ float fake_quantize_b(float x, float cmax, int& mask, int bit,
                                                 bool symmetry) {
  mask = clip_mask_bits(x, cmax, bit, symmetry);
  float scale = cmax / kQ;
  if (!symmetry) scale /= 2;
  float f = x / scale;
  if (!symmetry) f -= kQ;
  float q = fminf(fmaxf(floorf(f + 0.5f), -kQ), kQ);
  return symmetry ? q * scale : (q + kQ) * scale;
}
// A quantiser whose scale many elements share: quantize_b and fake_quantize_b bit for bit, the
// division by the scale made of a correctly rounded reciprocal, taken once, and a residual
// correction -- 3 instructions instead of the 12 of a division, in launches that are bound by them.
// Elements and clip values are halfs, so that the codes can be compared one by one: over all finite
// clip values and all halfs (2 x 10^9 pairs, both quantisers) they are those of the division, as
// with a second correction; without any 27265 differ.
// The clamp comes first, on the element: an infinite one has no residual (inf - inf), and of an
// element inside the clip value the quotient is at most 127 in magnitude, whatever its rounding, so
// that none is needed behind it.  A NaN becomes the lesser bound there, code -127, as it does in
// quantize_b.  (A clip value of zero gives code 0 where a division by zero gives others; what they
// stand for is zero either way.)
struct Quantiser {
  float scale, inv, lo, hi;
  static __device__ __forceinline__ Quantiser of(float cmax, bool symmetry = true) {
    float s = cmax / kQ;
    if (!symmetry) s /= 2;
    return Quantiser{s, s != 0.f ? 1.0f / s : 0.f, symmetry ? -cmax : 0.f, cmax};
  }
  __device__ __forceinline__ float quotient(float x) const {
    x = __builtin_amdgcn_fmed3f(x, lo, hi);
    const float q = x * inv;
    return __builtin_fmaf(__builtin_fmaf(-scale, q, x), inv, q);
  }
  __device__ __forceinline__ float rounded(float x) const {  // -127 .. 127
    return floorf(quotient(x) + 0.5f);
  }
  // four codes of one word: the conversion floors and writes its byte
  __device__ __forceinline__ uint32_t pack4(float x0, float x1, float x2, float x3) const {
    return floor_pack4_i8(quotient(x0) + 0.5f, quotient(x1) + 0.5f, quotient(x2) + 0.5f, quotient(x3) + 0.5f);
  }
  __device__ __forceinline__ float fake(float x) const { return rounded(x) * scale; }
  // the unsigned quantiser (symmetry = false)
  __device__ __forceinline__ float fake_unsigned(float x) const {
    return (floorf((quotient(x) - kQ) + 0.5f) + kQ) * scale;
  }
};
// kernels.h:497-501
__device__ __forceinline__ float dequantize_b(int q, float cmax) {
  const float r = (float)q * (cmax / kQ);
  return fminf(fmaxf(r, -cmax), cmax);
}
// dequantise + bias as T adds them (half: rounded operand, half add)
template <typename T>
__device__ __forceinline__ float deq_bias(int q, float cmax, float bias) {
  return TT<T>::rnd(TT<T>::rnd(dequantize_b(q, cmax)) + bias);
}
template <typename T>
__device__ __forceinline__ float cm(const T* p, int i = 0) {
  return TT<T>::ld(p, i);
}

// dropout_kernels.cu:25-59: float GELU/ReLU for T=float, the half2 forms for T=half
template <typename T, int ACT>
__device__ __forceinline__ float act_b(float x) {
  if (ACT == 1) return fmaxf(x, 0.f);
  if (sizeof(T) == 2) {
    const float p3 = TT<T>::rnd(x * TT<T>::rnd(x * x));
    // 0.5 * (1 + tanh(u)) as 1 / (1 + exp(-2u)), two hardware functions: the half it is rounded to
    // is the same for 65381 of the 65536 halfs x, and for the others (all but two below -2,
    // where 1 + tanh(u) cancels) the nearer one.  With tanhf the epilogue of the first feed-forward
    // product took longer than its K loop: 3600 x 3072 x 768 39.5 us, 28.2 now.
    const float cdf = __builtin_amdgcn_rcpf(
        1.0f + __builtin_amdgcn_exp2f(-2.f * 0.7978845608028654f * 1.44269504088896340736f * (x + 0.044715f * p3)));
    return TT<T>::rnd(x * TT<T>::rnd(cdf));
  }
  return gelu_tanh(x);
}

}  // namespace lsh
