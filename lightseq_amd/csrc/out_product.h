// The out-projection of a decoder attention inside the launch that makes the context (device part).
//
//   acc[row][n] += sum over the 64 dimensions of one head: context code * W[n][head * 64 + dim]
//
// A workgroup of the attention holds a head's 64 context codes of one to four rows; their share of
// the projection is 64 of its K, all columns: 64 KB of weights at hidden 1024, requested with the
// first cache rows and in registers when the context is ready, one MFMA per 16 columns.  The
// shares of the heads meet in int32 sums by atomic adds, exact in any order, which the layer norm
// behind it requantises as the product's epilogue did: the same bytes as attention, product and
// layer norm.  us, hidden 1024, attention and product as launches and as one: one row, 200 cached steps
// 3.8 + 3.0 -> 4.2; 4 beams, cross attention included 3.9 + 2.7 + 6.2 + 2.7 -> 4.2 + 7.1; 16 rows, 600
// steps 7.0 + 3.0 -> 7.8; 64 rows (16 sentences), 4.4 + 3.0 + 7.6 + 3.0 -> 7.0 + 10.6, no less time but
// two launches fewer of 9.  Adds by 16 workgroups to 16 rows cost less than can be measured, to 64 rows 1.2 us.
//
// The sums of a launch start from zero: three buffers take turns, and a launch clears the one of the
// next (whose last reader, the layer norm behind the launch before the last, is done by then:
// with two the cross attention, which reads the self attention's sums, would clear them).
#pragma once
#include "gemm_kw.h"
#include "ls_launch.h"

namespace lsh {

// N fragments of 16 columns x 64 bytes per wavefront, blocks of columns first .. first + N - 1; those from
// `hidden` / 16 on repeat the last one and add nothing.  Eight wavefronts of 8 / N workgroups share the at
// most 64 blocks: with few workgroups a compute unit's own 64 KB would be what the launch waits for,
// so 2, 4 or 8 of them attend to the same rows and take a part of the columns each (4 beams of
// hidden 1024, us a launch with 1, 4, 8: self attention 6.3, 4.7, 4.2, cross attention 8.7, 7.1, 7.4;
// one row, 100 steps: 5.6, 4.8, 4.8).
template <int N>
struct OutFragments {
  static constexpr int SHARE = 8 / N;  // workgroups that share a head's columns
  v4i w[N];
  __device__ __forceinline__ void request(const int8_t* __restrict__ W, int head, int heads, int first, int lane) {
#pragma unroll
    for (int f = 0; f < N; ++f)
      w[f] = *reinterpret_cast<const v4i*>(W + ((long)min(first + f, heads * 4 - 1) * heads + head) * 1024 + lane * 16);
  }
  // ctx: [ROWS][64] codes in LDS; acc: the first row's sums
  template <int ROWS>
  __device__ __forceinline__ void add(const int8_t* ctx, int32_t* acc, int rows, int hidden, int first, int lane) {
    static_assert(ROWS == 1 || ROWS == 4, "one row, or up to four");
    const int l16 = lane & 15, kq = lane >> 4;
    // the columns of the activation operand repeat the rows, so that every lane has a sum to add
    const v4i a = *reinterpret_cast<const v4i*>(ctx + (ROWS == 4 ? (l16 & 3) * 64 : 0) + kq * 16);
    v4i c[N];
#pragma unroll
    for (int f = 0; f < N; ++f) {
      asm volatile("" : "+v"(w[f]));
      c[f] = KwI8::mma(w[f], a, (v4i)0);
    }
    // a lane holds columns 16 block + 4 kq + 0 .. 3 of (all the same, or four) rows
    auto pick = [](const v4i& v, int j) { return j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3]; };
    if constexpr (ROWS == 4) {
      const int row = l16 & 3, j = l16 >> 2;
#pragma unroll
      for (int f = 0; f < N; ++f)
        if ((first + f) * 16 < hidden && row < rows)
          __hip_atomic_fetch_add(acc + row * hidden + (first + f) * 16 + 4 * kq + j, pick(c[f], j),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      const int j = l16 & 3, fl = l16 >> 2;
#pragma unroll
      for (int f0 = 0; f0 < N; f0 += 4) {
        int v = pick(c[f0], j);
#pragma unroll
        for (int i = 1; i < 4; ++i)
          if (f0 + i < N) v = fl == i ? pick(c[f0 + i], j) : v;
        if (f0 + fl < N && (first + f0 + fl) * 16 < hidden)
          __hip_atomic_fetch_add(acc + (first + f0 + fl) * 16 + 4 * kq + j, v, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  // any number of rows, 16 at a time (those from `rows` on of the last 16 need not hold anything)
  __device__ __forceinline__ void add_rows(const int8_t* ctx, int32_t* acc, int rows, int hidden, int first,
                                           int lane) {
    const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int f = 0; f < N; ++f) asm volatile("" : "+v"(w[f]));
    for (int r0 = 0; r0 < rows; r0 += 16) {
      const v4i a = *reinterpret_cast<const v4i*>(ctx + (r0 + l16) * 64 + kq * 16);
#pragma unroll
      for (int f = 0; f < N; ++f) {
        // a lane holds column l16 of the block for rows 4 kq + 0 .. 3: an instruction adds to 64
        // consecutive bytes of four rows
        const v4i c = KwI8::mma(a, w[f], (v4i)0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if ((first + f) * 16 < hidden && r0 + 4 * kq + i < rows)
            __hip_atomic_fetch_add(acc + (long)(r0 + 4 * kq + i) * hidden + (first + f) * 16 + l16, c[i],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
};

// how many workgroups share a head's columns where `groups` would hold all of them
inline int out_product_share(int groups) {
  return groups * 8 <= cu_count() ? 8 : groups * 4 <= cu_count() ? 4 : groups * 2 <= cu_count() ? 2 : 1;
}

}  // namespace lsh
