// The layer norm of a generation step inside the product that reads it (device part; LnStep in
// ls_launch.h says what is normalised).
//
// A layer norm of a few rows is a launch of 3 us that keeps one compute unit busy, between two
// products that wait for it.  Here every workgroup of the product normalises the rows itself:
// its weights are on their way from the memory meanwhile (about 2 us), so the arithmetic of one
// to four rows -- some 170 instructions of each of the four wavefronts per row, 0.35 us -- costs less
// than the launch, and 2 of a layer's 7 launches go.  At hidden 1024: one row 3.0 + 3.6 -> 4.0 us
// with the QKV product, four rows 2.8 + 3.2 -> 5.4 us.
// The sums run exactly as in ln_row_wg_kernel: four consecutive elements per thread, the lanes
// of a wavefront pairwise, the wavefronts in ascending order.
#pragma once
#include "ls_device.h"
#include "ls_launch.h"
#include "tile_common.h"

namespace lsh {

constexpr int kLnRequant = -1;

// ROWS rows (those from `rows` on repeat the last one and leave nothing) on 256 threads, hidden a
// multiple of 256 up to 1024: 256 D, or not known at compile time (D = 0).  PLANES: 0 int8 codes,
// 1 one int32 plane, 4 up to four, kLnRequant one plane of sums that are requantised first (p.requant).
template <int PLANES, int ROWS, int D = 0>
struct LnStepRows {
  static constexpr bool I32 = PLANES != 0;
  static constexpr int NP = PLANES == kLnRequant ? 1 : PLANES;
  Raw4H g, b, rb, cs, r[ROWS];
  int4 m[ROWS][I32 ? NP : 1];
  uint32_t w[ROWS];

  // requests everything; t: thread of the 256
  __device__ __forceinline__ void load(const LnStep& p, int t, long row0, int rows, int width) {
    const int hidden = D ? D * 256 : width;
    const int e = t * 4 < hidden ? t * 4 : 0;
    g = ld4_raw(p.scale, e);
    b = ld4_raw(p.bias, e);
    // optional operands through a pointer that is always valid, dropped afterwards
    rb = ld4_raw(p.res_bias != nullptr ? p.res_bias : p.scale, e);
    cs = ld4_raw(p.colsum != nullptr ? p.colsum : p.scale, e);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const long at = (row0 + min(i, rows - 1)) * hidden + e;
      r[i] = ld4_raw(p.res_in, at);
      if constexpr (I32) {
#pragma unroll
        for (int u = 0; u < NP; ++u)
          m[i][u] = *reinterpret_cast<const int4*>(static_cast<const int32_t*>(p.acc) +
                                                   min(u, p.planes - 1) * p.plane_stride + at);
      } else {
        w[i] = *reinterpret_cast<const uint32_t*>(static_cast<const int8_t*>(p.acc) + at);
      }
    }
  }

  // The codes of row i as row i of a blocked matrix of 16 rows in LDS; `keep`: this workgroup will
  // store the residual stream (at its end: loads in flight are not to wait for the stores).  red: [2][ROWS][4] floats of LDS.  Two barriers; the caller's
  // third makes the codes visible.
  __device__ __forceinline__ void finish(const LnStep& p, int t, long row0, int rows, int width,
                                         int8_t* codes, float* red, bool keep) {
    const int hidden = D ? D * 256 : width;
    const int lane = t & 63, wid = t >> 6, wpr = hidden >> 8;
    const int e = t * 4;
    const bool on = D == 4 || e < hidden;
    float gf[4], bf[4], rbf[4], cf[4], x[ROWS][4];
    cvt4(g, gf);
    cvt4(b, bf);
    const bool has_cs = p.colsum != nullptr;
    if (p.res_bias == nullptr) rb.v = make_uint2(0u, 0u);
    cvt4(rb, rbf);
    cvt4(cs, cf);
    auto totals = [&](const float (&v)[ROWS], float* rr, float (&out)[ROWS]) {
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const float s = wave_sum_dpp(v[i]);
        if (lane == 0) rr[i * 4 + wid] = s;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const float4 q = *reinterpret_cast<const float4*>(rr + i * 4);
        float s = q.x;
        if (wpr > 1) s += q.y;
        if (wpr > 2) s += q.z;
        if (wpr > 3) s += q.w;
        out[i] = s;
      }
    };
    float part[ROWS], mean[ROWS], var[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      float rf[4], a[4];
      cvt4(r[i], rf);
      if constexpr (I32) {
        int4 acc = m[i][0];
#pragma unroll
        for (int u = 1; u < NP; ++u)
          if (u < p.planes) {
            acc.x += m[i][u].x; acc.y += m[i][u].y;
            acc.z += m[i][u].z; acc.w += m[i][u].w;
          }
        if constexpr (PLANES == kLnRequant) {
          acc.x = requant_acc_fast(acc.x, p.requant); acc.y = requant_acc_fast(acc.y, p.requant);
          acc.z = requant_acc_fast(acc.z, p.requant); acc.w = requant_acc_fast(acc.w, p.requant);
        }
        a[0] = (float)acc.x; a[1] = (float)acc.y; a[2] = (float)acc.z; a[3] = (float)acc.w;
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = (float)unpack_i8(w[i], k);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) x[i][k] = a[k] * p.dequant_scale + TT<__half>::safe(rf[k]);
      if (has_cs) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[i][k] += TT<__half>::safe(cf[k]);
      }
      if (!on) x[i][0] = x[i][1] = x[i][2] = x[i][3] = 0.f;
      part[i] = (x[i][0] + x[i][1]) + (x[i][2] + x[i][3]);
    }
    totals(part, red, mean);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      mean[i] = mean[i] / (float)hidden;
      float v = 0.f;
      if (on) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float d = x[i][k] - mean[i];
          v += d * d;
        }
      }
      part[i] = v;
    }
    totals(part, red + ROWS * 4, var);
    if (!on) return;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const float rstd = rsqrtf(var[i] / (float)hidden + kLnEpsilon);
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        o[k] = (x[i][k] - mean[i]) * rstd * TT<__half>::safe(gf[k]) + TT<__half>::safe(bf[k]);
      *reinterpret_cast<uint32_t*>(codes + (e >> 6) * 1024 + ((e >> 4) & 3) * 256 + i * 16 + (e & 15)) =
          float2int8_pack4(o[0], o[1], o[2], o[3], p.quant_scale);
      if (keep) {
        half4_t h;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          h.v[k] = __float2half_rn(TT<__half>::rnd(p.is_post_ln ? o[k] : x[i][k]) + rbf[k]);
        __builtin_memcpy(&r[i].v, &h, sizeof(h));
      }
    }
  }
  __device__ __forceinline__ void store(const LnStep& p, int t, long row0, int rows, int width) const {
    const int hidden = D ? D * 256 : width, e = t * 4;
    if (e >= hidden) return;
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if (i < rows) *reinterpret_cast<uint2*>(p.res_out + (row0 + i) * hidden + e) = r[i].v;
  }
};

}  // namespace lsh
