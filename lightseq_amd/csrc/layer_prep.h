// The preparation of a quantised layer's matrices (device part), in units that a launch of their own or
// spare workgroups of another launch work through.
#pragma once
#include "layer_device.h"
#include "ls_launch.h"

namespace lsh {

// A unit is 16 rows x 512 columns, a quarter of it per wavefront (`wave`): a wavefront reads
// 128-byte pieces of 16 rows and writes 1 KB, the 16 rows x 64 bytes block; what a unit reads is
// requested before any of it is converted.
constexpr int kUnitK = 512;

__device__ __forceinline__ const __half* unit_row(const LayerPrepSection& s, int row) {
  const int r = min(row, s.rows - 1);
  if (s.n1 == 1) return s.src + (long)r * s.stride0;
  return s.src + (long)(r / s.n1) * s.stride0 + (long)(r % s.n1) * s.stride1;
}

__device__ __forceinline__ uint2 codes8(const Quantiser& of, const half8_t& x) {
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = __half2float(x.v[e]);
  return make_uint2(of.pack4(f[0], f[1], f[2], f[3]), of.pack4(f[4], f[5], f[6], f[7]));
}

__device__ __forceinline__ void unit_codes(const LayerPrepSection& s, int block, int wave) {
  const int per_row = (s.K + kUnitK - 1) / kUnitK;
  const int rb = block / per_row, kc = block - rb * per_row;
  const int lane = threadIdx.x & 63;
  const int row = rb * 16 + (lane & 15);
  const int k0 = kc * kUnitK + wave * 64 + (lane >> 4) * 16;
  const __half* src = unit_row(s, row);
  half8_t x[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      x[i][h] = *reinterpret_cast<const half8_t*>(src + min(k0 + i * 256 + h * 8, s.K - 8));  // K % 8 == 0
  const Quantiser of = Quantiser::of(cm(s.cmax));
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = k0 + i * 256;
    if (k >= s.k_pad) break;
    uint32_t w[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint2 q = codes8(of, x[i][h]);
      const bool on = row < s.rows && k + h * 8 < s.K;
      w[2 * h] = on ? q.x : 0u;
      w[2 * h + 1] = on ? q.y : 0u;
    }
    *reinterpret_cast<uint4*>(static_cast<int8_t*>(s.dst) + blocked_offset(row, k, s.k_pad)) =
        make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// fp16 -> blocked fp16 (64 bytes of K are 32 halfs), fake-quantised where `cmax` is set
__device__ __forceinline__ void unit_halfs(const LayerPrepSection& s, int block, int wave) {
  const int per_row = (s.K + kUnitK - 1) / kUnitK;
  const int rb = block / per_row, kc = block - rb * per_row;
  const int lane = threadIdx.x & 63;
  const int row = rb * 16 + (lane & 15);
  const int k0 = kc * kUnitK + wave * 32 + (lane >> 4) * 8;
  const __half* src = unit_row(s, row);
  half8_t x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const half8_t*>(src + min(k0 + i * 128, s.K - 8));
  const Quantiser of = Quantiser::of(s.cmax ? cm(s.cmax) : 1.f);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = k0 + i * 128;
    if (k >= s.k_pad) break;
    if (s.cmax) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[i].v[e] = __float2half_rn(of.fake(__half2float(x[i].v[e])));
    }
    if (row >= s.rows || k >= s.K) x[i] = half8_t{};
    *reinterpret_cast<half8_t*>(static_cast<char*>(s.dst) + blocked_offset(row, 2 * k, 2 * s.k_pad)) = x[i];
  }
}

// Matrices that ride in another launch: its workgroups from the first spare one on.  The weights of a
// layer's later products need not be ready before its first one, and what they wait behind is a
// chain of small launches that leave the memory idle.  Transformer-big decoder layer: preparation
// 14.8 -> 6.4 us, the four launches that take riders 20.2 -> 24.5 (16 x 61 rows); one decoding step
// 17.6 -> 10.0 and 18.6 -> 23.1 (64 rows).
__device__ __forceinline__ void ride_unit(const LayerRide& r, int block, int wave) {
  int i = 0, first = 0;
#pragma unroll
  for (int j = 1; j < kLayerRideMost; ++j)
    if (block >= r.first[j]) {
      i = j;
      first = r.first[j];
    }
  const LayerPrepSection& s = r.s[i];
  if (s.kind == kPrepCodes) unit_codes(s, block - first, wave);
  else unit_halfs(s, block - first, wave);
}

}  // namespace lsh
