// Epilogues of the generation steps' products (the QKV product with its cache append, the
// cross-attention query), shared by the row-major and the blocked kernels.
#pragma once
#include "ls_device.h"
#include "tile_common.h"

namespace lsh {

// n / d for 0 <= n < 2^24, d > 0, with inv = 1.0f / d from the host: the float product is
// within one of the quotient, the remainder decides.  A handful of instructions where the
// integer division is about forty -- in kernels whose length is their instruction count.
__device__ __forceinline__ int div_by(int n, int d, float inv) {
  int q = (int)((float)n * inv);
  const int r = n - q * d;
  if (r >= d) ++q;
  if (r < 0) --q;
  return q;
}

// Decode-step QKV product followed by ker_arrange_decself_qkv_i8I_i8O
// (inference/kernels/transformerKernels_int8.cc.cu:1432-1513; call sites
// model/quant_decoder.cc.cu:660-674, model/quant_gpt_encoder.cc.cu:640-653): the int8 code
// of the product is dequantised, biased and requantised with the cache scale; columns
// [0, H) go to new_q [M, H], [H, 2H) and [2H, 3H) to slot step_id of the K and V caches
// [M, heads, max_step, d].  Same float arithmetic as the stand-alone kernel (no fused
// multiply-add).
struct EpiDecQkvI8 {
  int8_t *new_q, *new_k, *new_v;
  const __half* bias;
  float alpha, dequant_scale, quant_scale;
  int hidden, head_num, dim_per_head, max_step, step_id;
  float inv_hidden, inv_dim;  // 1 / hidden, 1 / dim_per_head (for store1)
  // the 16 bias values of columns n .. n + 15: they do not depend on the product, so the
  // decode-step kernel requests them with its first weights
  struct Pre {
    half8_t b0, b1;
  };
  __device__ __forceinline__ Pre prefetch(int n) const {
    return Pre{*reinterpret_cast<const half8_t*>(bias + n),
               *reinterpret_cast<const half8_t*>(bias + n + 8)};
  }
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, bool full) const {
    store16_pre(m, n, N, c, full, prefetch(n));
  }
  __device__ __forceinline__ void store16_pre(long m, int n, int N, const v16i& c, bool,
                                              const Pre& pre) const {
#pragma clang fp contract(off)
    const int part = n / hidden, i = n - part * hidden;
    const half8_t b0 = pre.b0, b1 = pre.b1;
    int q[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float b = __half2float(k < 8 ? b0.v[k] : b1.v[k - 8]);
      const float val = (float)requant_acc(c[k], alpha) * dequant_scale + b;
      q[k] = float2int8(val, quant_scale);
    }
    int8_t* dst;
    if (part == 0) {
      dst = new_q + m * hidden + i;
    } else {
      const int head = i / dim_per_head, dim = i - head * dim_per_head;
      dst = (part == 1 ? new_k : new_v) +
            ((m * head_num + head) * max_step + step_id) * dim_per_head + dim;
    }
    uint4 o;
    o.x = pack4_i8(q[0], q[1], q[2], q[3]);
    o.y = pack4_i8(q[4], q[5], q[6], q[7]);
    o.z = pack4_i8(q[8], q[9], q[10], q[11]);
    o.w = pack4_i8(q[12], q[13], q[14], q[15]);
    *reinterpret_cast<uint4*>(dst) = o;
    (void)N;
  }
  // one element; its bias value is requested with the first weights
  struct Pre1 {
    __half b;
  };
  __device__ __forceinline__ Pre1 prefetch1(int n) const { return Pre1{bias[n]}; }
  // what the elements of one column share: the 16 columns of a block lie in one part and one
  // head (dim_per_head % 16 == 0), so the divisions run on the block's first column, the same
  // in every lane, once per block; an element's address is base + row * row_stride + add.
  // 32-bit offsets: this form serves the decode-step kernels only (at most 64 rows; the
  // launcher refuses caches of 2^31 bytes and more for them)
  struct Blk1 {
    int8_t* base;
    int row_stride, add;
  };
  __device__ __forceinline__ Blk1 block1(int n) const {
    const int nb = __builtin_amdgcn_readfirstlane(n & ~15);
    const int part = div_by(nb, hidden, inv_hidden), ib = nb - part * hidden;
    const int head = div_by(ib, dim_per_head, inv_dim), dim = ib - head * dim_per_head + (n & 15);
    if (part == 0) return Blk1{new_q, hidden, ib + (n & 15)};
    return Blk1{part == 1 ? new_k : new_v, head_num * max_step * dim_per_head,
                (head * max_step + step_id) * dim_per_head + dim};
  }
  __device__ __forceinline__ void store1(long m, Blk1 blk, int N, int acc, Pre1 pre,
                                         const int8_t*, int) const {
#pragma clang fp contract(off)
    const float val = (float)requant_acc_fast(acc, alpha) * dequant_scale + __half2float(pre.b);
    blk.base[(unsigned)((int)m * blk.row_stride + blk.add)] =
        (int8_t)float2int8(val, quant_scale);
    (void)N;
  }
  // four neighbouring columns of one head (gemm_kw.h)
  static constexpr bool kTable = false, kBlockedOut = false;
  struct Col {
    int8_t* base;
    int row_stride, add;
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    const int part = div_by(n, hidden, inv_hidden), i = n - part * hidden;
    const int head = div_by(i, dim_per_head, inv_dim), dim = i - head * dim_per_head;
    const half4_t b = *reinterpret_cast<const half4_t*>(bias + n);
    if (part == 0) return Col{new_q, hidden, i, b};
    return Col{part == 1 ? new_k : new_v, head_num * max_step * dim_per_head,
               (head * max_step + step_id) * dim_per_head + dim, b};
  }
  __device__ __forceinline__ void store4(int m, int, int, const Col& col, const v4i& c) const {
#pragma clang fp contract(off)
    int q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float val =
          (float)requant_acc_fast(c[k], alpha) * dequant_scale + __half2float(col.b.v[k]);
      q[k] = float2int8(val, quant_scale);
    }
    *reinterpret_cast<uint32_t*>(col.base + (long)m * col.row_stride + col.add) =
        pack4_i8(q[0], q[1], q[2], q[3]);
  }
  bool aligned() const {
    return ((reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(new_q) |
             reinterpret_cast<uintptr_t>(new_k) | reinterpret_cast<uintptr_t>(new_v)) & 7u) == 0;
  }
  bool vec_ok(int) const { return true; }
  static const char* name() { return "EpiDecQkvI8"; }
};

// QKV product of a GPT prompt pass followed by gpt_arrange_qkv_prefill_i8, with the same bits: code
// -> code * dq + bias -> requantised with the cache clip -> query codes [batch, head, seq, d], key
// and value codes into the caches [batch, head, max_step, d].  row_map: the position b * seq + s
// that a row holds, where the rows are those of a plan.  The stand-alone launch reads and writes
// all the codes once more and is one of nine launches of a layer: 10.3 us for 3072 rows of 3 x 1024.
struct EpiPromptQkvI8 {
  static constexpr bool kTable = false, kBlockedOut = false, kColumn16 = true, kFetch = true, kFetch16 = true;
  int8_t *q, *k, *v;
  const __half* bias;
  const int* row_map;
  float alpha, dequant_scale, quant_scale;
  int hidden, head_num, dim, max_step, seq;
  float inv_hidden, inv_dim, inv_seq;
  struct Col {
    int8_t* base;
    int head, steps;
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    const int part = div_by(n, hidden, inv_hidden), i = n - part * hidden;
    const int head = div_by(i, dim, inv_dim);
    return Col{(part == 0 ? q : part == 1 ? k : v) + (i - head * dim), head, part == 0 ? seq : max_step,
               *reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ int fetch(int m, int, int) const { return row_map != nullptr ? row_map[m] : m; }
  __device__ __forceinline__ int8_t* row_ptr(const Col& col, int p) const {
    const int b = div_by(p, seq, inv_seq), s = p - b * seq;
    return col.base + ((long)(b * head_num + col.head) * col.steps + s) * dim;
  }
  __device__ __forceinline__ float value(int acc, __half b) const {
#pragma clang fp contract(off)
    return floorf(requant_acc_clamped(acc, alpha)) * dequant_scale + __half2float(b);
  }
  __device__ __forceinline__ void store4(int, int, int, const Col& col, const v4i& c, int p) const {
    *reinterpret_cast<uint32_t*>(row_ptr(col, p)) =
        float2int8_pack4(value(c[0], col.b.v[0]), value(c[1], col.b.v[1]), value(c[2], col.b.v[2]),
                         value(c[3], col.b.v[3]), quant_scale);
  }
  // 16 columns of one head (dim % 16 == 0)
  struct Col16 {
    half8_t b[2];
  };
  __device__ __forceinline__ Col16 column16(int n) const {
    return Col16{{*reinterpret_cast<const half8_t*>(bias + n), *reinterpret_cast<const half8_t*>(bias + n + 8)}};
  }
  __device__ __forceinline__ int fetch16(int m, int, int) const { return fetch(m, 0, 0); }
  __device__ __forceinline__ void store16(long, int n, int, const v16i& c, const Col16& col, int p) const {
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const __half* b = &col.b[j >> 1].v[4 * (j & 1)];
      w[j] = float2int8_pack4(value(c[4 * j], b[0]), value(c[4 * j + 1], b[1]), value(c[4 * j + 2], b[2]),
                              value(c[4 * j + 3], b[3]), quant_scale);
    }
    const int part = div_by(n, hidden, inv_hidden), i = n - part * hidden, head = div_by(i, dim, inv_dim);
    const Col at{(part == 0 ? q : part == 1 ? k : v) + (i - head * dim), head, part == 0 ? seq : max_step, {}};
    *reinterpret_cast<uint4*>(row_ptr(at, p)) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  bool aligned() const {
    return ((reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(q) |
             reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15u) == 0;
  }
};

// Decode-step cross-attention query product followed by ker_arrange_encdec_q_i8I
// (inference/kernels/transformerKernels_int8.cc.cu:1596-1645; call site
// model/quant_decoder.cc.cu:745-760): code -> half(code * dq) + bias (a half add) -> fp16 q
// [batch, heads, beam, d].
struct EpiEncdecQF16 {
  __half* new_q;
  const __half* bias;
  float alpha, dequant_scale;
  int beam_size, head_num, dim_per_head;
  float inv_beam, inv_dim;  // 1 / beam_size, 1 / dim_per_head (for store1)
  struct Pre {  // the bias of columns n .. n + 15, requested ahead of the product
    half8_t b0, b1;
  };
  __device__ __forceinline__ Pre prefetch(int n) const {
    return Pre{*reinterpret_cast<const half8_t*>(bias + n),
               *reinterpret_cast<const half8_t*>(bias + n + 8)};
  }
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, bool full) const {
    store16_pre(m, n, N, c, full, prefetch(n));
  }
  __device__ __forceinline__ void store16_pre(long m, int n, int N, const v16i& c, bool,
                                              const Pre& pre) const {
    const int head = n / dim_per_head, dim = n - head * dim_per_head;
    const long batch_id = m / beam_size, beam_id = m - batch_id * beam_size;
    __half* dst = new_q + ((batch_id * head_num + head) * beam_size + beam_id) * dim_per_head + dim;
    const half8_t b0 = pre.b0, b1 = pre.b1;
    half8_t lo, hi;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      lo.v[k] = __float2half_rn(dequant_add_bias_h(requant_acc(c[k], alpha), dequant_scale,
                                                   __half2float(b0.v[k])));
      hi.v[k] = __float2half_rn(dequant_add_bias_h(requant_acc(c[8 + k], alpha), dequant_scale,
                                                   __half2float(b1.v[k])));
    }
    *reinterpret_cast<half8_t*>(dst) = lo;
    *reinterpret_cast<half8_t*>(dst + 8) = hi;
    (void)N;
  }
  struct Pre1 {
    __half b;
  };
  __device__ __forceinline__ Pre1 prefetch1(int n) const { return Pre1{bias[n]}; }
  struct Blk1 {
    int add;  // the column's share of the offset: head * beam_size * dim_per_head + dim
  };
  __device__ __forceinline__ Blk1 block1(int n) const {
    const int nb = __builtin_amdgcn_readfirstlane(n & ~15);
    const int head = div_by(nb, dim_per_head, inv_dim), dim = nb - head * dim_per_head + (n & 15);
    return Blk1{head * beam_size * dim_per_head + dim};
  }
  __device__ __forceinline__ void store1(long m, Blk1 blk, int N, int acc, Pre1 pre,
                                         const int8_t*, int) const {
    const int batch_id = div_by((int)m, beam_size, inv_beam), beam_id = (int)m - batch_id * beam_size;
    new_q[(unsigned)((batch_id * head_num * beam_size + beam_id) * dim_per_head + blk.add)] =
        __float2half_rn(dequant_add_bias_h(requant_acc_fast(acc, alpha), dequant_scale,
                                           __half2float(pre.b)));
    (void)N;
  }
  static constexpr bool kTable = false, kBlockedOut = false;
  struct Col {
    int add;
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    const int head = div_by(n, dim_per_head, inv_dim), dim = n - head * dim_per_head;
    return Col{head * beam_size * dim_per_head + dim, *reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ void store4(int m, int, int, const Col& col, const v4i& c) const {
    const int batch_id = div_by(m, beam_size, inv_beam), beam_id = m - batch_id * beam_size;
    half4_t o;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o.v[k] = __float2half_rn(dequant_add_bias_h(requant_acc_fast(c[k], alpha), dequant_scale,
                                                  __half2float(col.b.v[k])));
    *reinterpret_cast<half4_t*>(new_q + (long)(batch_id * head_num * beam_size + beam_id) * dim_per_head +
                                col.add) = o;
  }
  bool aligned() const {
    return ((reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(new_q)) & 7u) == 0;
  }
  bool vec_ok(int) const { return true; }
  static const char* name() { return "EpiEncdecQF16"; }
};

}  // namespace lsh
