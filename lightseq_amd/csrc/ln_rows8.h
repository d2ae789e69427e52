// The row routine of the 8-wide layer-norm kernels (dequantise + residual (+ column sums) +
// LayerNorm + quantise of one token row held by LPR lanes), shared by the stand-alone kernel,
// the out-projection kernel that ends in it (ln_kernels.hip) and the per-XCD feed-forward
// segment (xcd_ffn_kernels.hip).  Replaces inference/kernels/transformerKernels_int8.cc.cu:
// 149-863.
#pragma once
#include "ls_device.h"
#include "tile_common.h"

namespace lsh {

enum LnMode {
  kLnFirst = 0,    // ker_norm_layer_resual_i8O      (:149-316)
  kLnResQuant = 1, // ker_residual_bias_ln_i{8,32}I_i8O (:318-705)
  kLnResOut = 2    // ker_residual_bias_ln_i32I      (:707-863)
};

// 8 consecutive elements per lane per step (one 16-byte load of fp16 data, 8 bytes of int8
// codes, two 16-byte loads of int32 accumulators); LPR lanes share a row, so a wavefront
// covers 64/LPR rows and a workgroup 4 * 64/LPR.  All loads of a lane are issued before the
// first reduction.  `nparts` int32 accumulator planes `part_stride` elements apart are
// summed first (the split-K form of the int32 GEMM); the sum of integers is exact.
// Preconditions (checked by the launcher): hidden % 8 == 0, hidden <= LPR * 8 * ITER,
// 16-byte aligned pointers.
__device__ __forceinline__ void ld8_acc(const int8_t* p, long i, float (&o)[8]) {
  uint2 w = *reinterpret_cast<const uint2*>(p + i);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    o[k] = (float)unpack_i8(w.x, k);
    o[4 + k] = (float)unpack_i8(w.y, k);
  }
}
__device__ __forceinline__ void ld8_acc(const int32_t* p, long i, int (&o)[8]) {
  int4 a = *reinterpret_cast<const int4*>(p + i);
  int4 b = *reinterpret_cast<const int4*>(p + i + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
  o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}
__device__ __forceinline__ void ld8(const float* p, long i, float (&o)[8]) {
  float a[4], b[4];
  ld4(p, i, a);
  ld4(p, i + 4, b);
#pragma unroll
  for (int k = 0; k < 4; ++k) { o[k] = a[k]; o[4 + k] = b[k]; }
}
__device__ __forceinline__ void ld8(const __half* p, long i, float (&o)[8]) {
  half8_t t = *reinterpret_cast<const half8_t*>(p + i);
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k] = __half2float(t.v[k]);
}
__device__ __forceinline__ void st8(float* p, long i, const float (&o)[8]) {
  *reinterpret_cast<float4*>(p + i) = make_float4(o[0], o[1], o[2], o[3]);
  *reinterpret_cast<float4*>(p + i + 4) = make_float4(o[4], o[5], o[6], o[7]);
}
__device__ __forceinline__ void st8(__half* p, long i, const float (&o)[8]) {
  half8_t t;
#pragma unroll
  for (int k = 0; k < 8; ++k) t.v[k] = __float2half_rn(o[k]);
  *reinterpret_cast<half8_t*>(p + i) = t;
}
// Eight consecutive elements as raw words (converted after every load of the row has been
// requested) and the statement that makes the words opaque to the compiler, which otherwise
// sinks a load into the branch that uses its values, where it is followed by its wait.
struct Raw8F { float4 a, b; };
struct Raw8H { uint4 a; };
struct Raw8I { int4 a, b; };
struct Raw8C { uint2 a; };
__device__ __forceinline__ Raw8F ld8_raw(const float* p, long i) {
  return Raw8F{*reinterpret_cast<const float4*>(p + i), *reinterpret_cast<const float4*>(p + i + 4)};
}
__device__ __forceinline__ Raw8H ld8_raw(const __half* p, long i) {
  return Raw8H{*reinterpret_cast<const uint4*>(p + i)};
}
__device__ __forceinline__ Raw8I ld8_raw(const int32_t* p, long i) {
  return Raw8I{*reinterpret_cast<const int4*>(p + i), *reinterpret_cast<const int4*>(p + i + 4)};
}
__device__ __forceinline__ Raw8C ld8_raw(const int8_t* p, long i) {
  return Raw8C{*reinterpret_cast<const uint2*>(p + i)};
}
__device__ __forceinline__ void pin8(Raw8F& r) {
  asm volatile("" : "+v"(r.a.x), "+v"(r.a.y), "+v"(r.a.z), "+v"(r.a.w), "+v"(r.b.x), "+v"(r.b.y),
               "+v"(r.b.z), "+v"(r.b.w));
}
__device__ __forceinline__ void pin8(Raw8H& r) {
  asm volatile("" : "+v"(r.a.x), "+v"(r.a.y), "+v"(r.a.z), "+v"(r.a.w));
}
__device__ __forceinline__ void pin8(Raw8I& r) {
  asm volatile("" : "+v"(r.a.x), "+v"(r.a.y), "+v"(r.a.z), "+v"(r.a.w), "+v"(r.b.x), "+v"(r.b.y),
               "+v"(r.b.z), "+v"(r.b.w));
}
__device__ __forceinline__ void pin8(Raw8C& r) { asm volatile("" : "+v"(r.a.x), "+v"(r.a.y)); }
__device__ __forceinline__ void cvt8(const Raw8F& r, float (&o)[8]) {
  o[0] = r.a.x; o[1] = r.a.y; o[2] = r.a.z; o[3] = r.a.w;
  o[4] = r.b.x; o[5] = r.b.y; o[6] = r.b.z; o[7] = r.b.w;
}
__device__ __forceinline__ void cvt8(const Raw8H& r, float (&o)[8]) {
  half8_t t;
  __builtin_memcpy(&t, &r.a, sizeof(t));
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k] = __half2float(t.v[k]);
}
__device__ __forceinline__ void cvt8(const Raw8I& r, int (&o)[8]) {
  o[0] = r.a.x; o[1] = r.a.y; o[2] = r.a.z; o[3] = r.a.w;
  o[4] = r.b.x; o[5] = r.b.y; o[6] = r.b.z; o[7] = r.b.w;
}
__device__ __forceinline__ void cvt8(const Raw8C& r, float (&o)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    o[k] = (float)unpack_i8(r.a.x, k);
    o[4 + k] = (float)unpack_i8(r.a.y, k);
  }
}
// Sum over the LPR (32 or 64) lanes of a row, every lane active: the additions of the
// shuffle tree lane ^ 32, 16, 8, 4, 2, 1 in that order, on exchanges that stay in the vector
// registers (a permute through LDS takes tens of cycles, six in a chain, twice a row).
template <int LPR>
__device__ __forceinline__ float row_sum(float v) {
  // the words of a swap go into scalars first: a bit cast of the element of a vector reads the
  // vector's first element, whatever the index
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  if constexpr (LPR == 64) {
    const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t lo = s[0], hi = s[1];
    v = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
  }
  const uint32_t w = __builtin_bit_cast(uint32_t, v);
  const auto s = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  const uint32_t lo = s[0], hi = s[1];
  v = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
  v += dpp_f<kDppRor8>(v);                         // lane ^ 8
  v += dpp_f<kDppXor3>(dpp_f<kDppHalfMirror>(v));  // lane ^ 7 ^ 3
  v += dpp_f<kDppXor2>(v);
  v += dpp_f<kDppXor1>(v);
  return v;
}
typedef _Float16 HalfPair __attribute__((ext_vector_type(2)));
// keep + bias in the storage type, where keep has just been rounded to it: a half addition
// (two roundings, to float and to half, of the sum of two halves are one: 24 >= 2 * 11 + 2)
__device__ __forceinline__ void add8_store(float* p, long i, const float (&keep)[8], const Raw8F& rb) {
  float b[8], w[8];
  cvt8(rb, b);
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = keep[k] + b[k];
  st8(p, i, w);
}
__device__ __forceinline__ void add8_store(__half* p, long i, const float (&keep)[8], const Raw8H& rb) {
  const uint32_t words[4] = {rb.a.x, rb.a.y, rb.a.z, rb.a.w};
  uint32_t out[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const HalfPair v = {(_Float16)keep[2 * k], (_Float16)keep[2 * k + 1]};
    out[k] = __builtin_bit_cast(uint32_t, v + __builtin_bit_cast(HalfPair, words[k]));
  }
  *reinterpret_cast<uint4*>(p + i) = make_uint4(out[0], out[1], out[2], out[3]);
}
__device__ __forceinline__ void zero8(Raw8F& r) { r.a = r.b = make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ void zero8(Raw8H& r) { r.a = make_uint4(0, 0, 0, 0); }

// One row of the 8-wide kernel: `sub` is the lane's index among the LPR lanes of the row,
// `live` false for a row beyond the tensor (its lanes still take part in the shuffles).
// gemm_out is read at gemm_out[row * hidden + column] and may point anywhere a flat load
// reaches (the fused GEMM + LayerNorm kernel passes a tile staged in LDS).
template <typename T, typename AccT, int MODE, int LPR, int ITER, bool FULL = false, bool REQ = false>
__device__ __forceinline__ void
ln_rows8_row(int row, bool live, int sub, const AccT* __restrict__ gemm_out, T* residual, T* out_t,
             int8_t* __restrict__ out_q, const T* __restrict__ scale, const T* __restrict__ bias,
             const T* __restrict__ residual_bias, const T* __restrict__ colsum, int width,
             float dequant_scale, float quant_scale, int is_post_ln, int nparts, long part_stride,
             const half8_t* pre_res = nullptr, int dead_row = 0, int blocked = 0, int in_row = -1,
             float requant = 0.f) {
  // pre_res (fp16 only): the lane's ITER residual chunks, already loaded by the caller.
  // dead_row: the row whose addresses a lane without a row reads (and drops); a caller that
  // hands over a staged tile names a row of the tile.
  // blocked: out_q is a blocked matrix.  in_row: the row of gemm_out and residual that row `row` of
  // out_t is made from, where that is another one (kLnResOut).
  // REQ: int32 sums that become int8 codes of the scale `requant` first.
  // FULL: the row fills its lanes' chunks, width == LPR * 8 * ITER.
  constexpr int kWidth = LPR * 8 * ITER;
  const int hidden = FULL ? kWidth : width;
  const long base = (long)(live ? (in_row >= 0 ? in_row : row) : dead_row) * hidden;
  const long out_base = (long)row * hidden;

  float x[ITER][8];
  // Every load of the row -- parameters, residual, accumulator, column sums -- is requested
  // before the first value is used: no branch around a load (columns beyond the row and rows
  // beyond the tensor are clamped, optional operands read through a pointer that is always
  // valid, and what they bring is dropped), a scheduling barrier after the last request, and
  // only then the statements that make the values visible to the arithmetic.  Written with
  // conditions around the loads, the compiler put each load next to its use: six to nine
  // memory round trips in a row instead of one.
  const bool has_rb = MODE != kLnResOut && residual_bias != nullptr;
  const bool has_cs = MODE != kLnFirst && colsum != nullptr;
  const bool own_res = !(sizeof(T) == 2 && pre_res != nullptr);
  const T* rbp = has_rb ? residual_bias : scale;
  const T* csp = has_cs ? colsum : scale;
  decltype(ld8_raw(scale, 0)) g_raw[ITER], b_raw[ITER], rb_raw[ITER], cs_raw[ITER], r_raw[ITER];
  decltype(ld8_raw(gemm_out, 0)) a_raw[ITER];
#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    const int e = FULL ? (it * LPR + sub) * 8 : min((it * LPR + sub) * 8, hidden - 8);
    g_raw[it] = ld8_raw(scale, e);
    b_raw[it] = ld8_raw(bias, e);
    rb_raw[it] = ld8_raw(rbp, e);
    cs_raw[it] = ld8_raw(csp, e);
    r_raw[it] = ld8_raw(own_res ? residual + base + e : scale, 0);
    if (MODE != kLnFirst) a_raw[it] = ld8_raw(gemm_out, base + e);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    pin8(g_raw[it]);
    pin8(b_raw[it]);
    pin8(rb_raw[it]);
    pin8(cs_raw[it]);
    pin8(r_raw[it]);
    if (MODE != kLnFirst) pin8(a_raw[it]);
  }
  float sum = 0.f;
#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    const int e = (it * LPR + sub) * 8;
    if (FULL || (e < hidden && live)) {
      float r[8];
      if (own_res) {
        cvt8(r_raw[it], r);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = __half2float(pre_res[it].v[k]);
      }
      if (MODE == kLnFirst) {
#pragma unroll
        for (int k = 0; k < 8; ++k) x[it][k] = TT<T>::safe(r[k]);
      } else {
        float a[8];
        if constexpr (sizeof(AccT) == 4) {
          // further planes in a rolled loop: launches of a few rows, where the planes come
          // from, use the row kernel, and this one stays small
          int acc[8];
          cvt8(a_raw[it], acc);
          for (int p = 1; p < nparts; ++p) {
            int more[8];
            ld8_acc(gemm_out + p * part_stride, base + e, more);
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] += more[k];
          }
#pragma unroll
          for (int k = 0; k < 8; ++k) a[k] = (float)(REQ ? requant_acc_fast(acc[k], requant) : acc[k]);
        } else {
          cvt8(a_raw[it], a);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) x[it][k] = a[k] * dequant_scale + TT<T>::safe(r[k]);
        if (has_cs) {
          float c[8];
          cvt8(cs_raw[it], c);
#pragma unroll
          for (int k = 0; k < 8; ++k) x[it][k] += TT<T>::safe(c[k]);
        }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) sum += x[it][k];
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) x[it][k] = 0.f;
    }
  }
  const float mean = row_sum<LPR>(sum) / (float)hidden;
  float var = 0.f;
#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    const int e = (it * LPR + sub) * 8;
    if (FULL || e < hidden) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float t = x[it][k] - mean;
        var += t * t;
      }
    }
  }
  const float rstd = rsqrtf(row_sum<LPR>(var) / (float)hidden + kLnEpsilon);
  if (!live) return;

#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    const int e = (it * LPR + sub) * 8;
    if (FULL || e < hidden) {
      float g[8], b[8], o[8];
      cvt8(g_raw[it], g);
      cvt8(b_raw[it], b);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        o[k] = (x[it][k] - mean) * rstd * TT<T>::safe(g[k]) + TT<T>::safe(b[k]);
      if (MODE == kLnResOut) {
        st8(out_t, out_base + e, o);
      } else {
        uint2 packed;
        packed.x = float2int8_pack4(o[0], o[1], o[2], o[3], quant_scale);
        packed.y = float2int8_pack4(o[4], o[5], o[6], o[7], quant_scale);
        *reinterpret_cast<uint2*>(out_q + code_offset(row, e, hidden, blocked)) = packed;
        if (!has_rb) zero8(rb_raw[it]);
        float keep[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) keep[k] = is_post_ln ? o[k] : x[it][k];
        if (MODE == kLnFirst && sizeof(T) == 2) {
          // the first norm's sum is a float's, rounded once
          float rb[8];
          cvt8(rb_raw[it], rb);
#pragma unroll
          for (int k = 0; k < 8; ++k) keep[k] += rb[k];
          st8(residual, base + e, keep);
        } else {
          add8_store(residual, base + e, keep, rb_raw[it]);
        }
      }
    }
  }
}

}  // namespace lsh
