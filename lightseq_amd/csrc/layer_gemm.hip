// The products of the quantised encoder and decoder layers with what follows each of them as the
// epilogue, on blocked operands (gemm_blocked.hip).
//
// A layer used to quantise, multiply to int8 codes, and read the codes back in a streaming kernel
// that dequantises, adds the bias and does what comes next.  Those kernels are a few
// microseconds of launch and memory round trip each at the sizes layers run at, so their
// arithmetic moved into the products: same formulas (layer_device.h), same rounding to fp16
// between the steps.  The clip values stay device scalars; an epilogue reads them once
// (request()), ahead of the first product.
//
// The second feed-forward product multiplies fake-quantised values in fp16, as it always did: the
// same codes multiplied in int8 give exact sums at half the bytes, but those differ from the
// sums of the fp16-rounded values by about one unit of fp16, which after a few layers has moved
// enough codes by one to be seen (4 % of a six-layer output).
//
// aligned() of these epilogues has nothing to ask: a layer call takes parameters, residual and output
// at any address, as the streaming kernels did (vector accesses to global memory need no
// alignment here); the operands are the layer's own buffers, which check_blk looks at.
#include "gemm_blk_dispatch.h"
#include "gemm_dec_epi.h"
#include "layer_device.h"

namespace lsh {

namespace {

__device__ __forceinline__ half4_t pack_half4(float a, float b, float c, float d) {
  half4_t o;
  o.v[0] = __float2half_rn(a);
  o.v[1] = __float2half_rn(b);
  o.v[2] = __float2half_rn(c);
  o.v[3] = __float2half_rn(d);
  return o;
}

// eight halfs as one 16-byte access; an LDS tile's lane holds sixteen neighbouring columns
__device__ __forceinline__ half8_t ld8(const __half* p) { return *reinterpret_cast<const half8_t*>(p); }
__device__ __forceinline__ void st8(void* p, const half8_t& x) { *reinterpret_cast<half8_t*>(p) = x; }
struct Half16 {
  half8_t h[2];
};
__device__ __forceinline__ Half16 ld16(const __half* p) { return Half16{{ld8(p), ld8(p + 8)}}; }

// clip values {input, weight, output} of an int8 product
struct ProductClips {
  const __half* cmax;
  float alpha, c_out, unit;
  struct Raw {
    __half in, weight, out;
  };
  __device__ __forceinline__ Raw request() const { return Raw{cmax[0], cmax[1], cmax[2]}; }
  __device__ __forceinline__ void finish(const Raw& r) {
    c_out = __half2float(r.out);
    unit = c_out / kQ;
    alpha = __half2float(r.in) * __half2float(r.weight) / (c_out * kQ);
  }
  // the element as the next operator reads it: int8 code, dequantised, bias added
  __device__ __forceinline__ float value(int acc, float bias) const {
    // (deq_bias; of three values the middle one is its clamp to +- c_out)
    const float r = __builtin_amdgcn_fmed3f((float)requant_acc_fast(acc, alpha) * unit, -c_out, c_out);
    return TT<__half>::rnd(TT<__half>::rnd(r) + bias);
  }
};

// where head h, position s of sequence b of part p goes: p's base + ((b heads + h) len + at + s) d
struct HeadPart {
  __half* base;
  int len, at;
};

// int8 [rows, parts * hidden] -> fp16 [part][b][head][position][d] with bias
// (opb_quant_bias_add_transform_20314); cache_cmax: fake-quantised like a cache entry
template <bool CACHE>
struct EpiHeads {
  static constexpr bool kTable = false, kBlockedOut = false, kClips = true, kColumn16 = true, kFetch16 = true;
  HeadPart p0, p1, p2;
  const __half *bias, *cache_cmax;
  ProductClips clips;
  Quantiser cache;
  int seq, heads, dim, hidden;
  float inv_seq, inv_hidden, inv_dim;
  struct Raw {
    ProductClips::Raw clips;
    __half cache;
  };
  __device__ __forceinline__ Raw request() const {
    Raw r{clips.request(), __half{}};
    if (CACHE) r.cache = cache_cmax[0];
    return r;
  }
  __device__ __forceinline__ EpiHeads finish(const Raw& r) const {
    EpiHeads e = *this;
    e.clips.finish(r.clips);
    if (CACHE) e.cache = Quantiser::of(__half2float(r.cache));
    return e;
  }
  struct Col {
    __half* base;
    int len, off, head;
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    const int part = div_by(n, hidden, inv_hidden), i = n - part * hidden;
    const int head = div_by(i, dim, inv_dim);
    const HeadPart p = part == 0 ? p0 : part == 1 ? p1 : p2;
    return Col{p.base, p.len, p.at * dim + (i - head * dim), head,
               *reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ float last(float x) const {
    return CACHE ? cache.fake(x) : x;
  }
  __device__ __forceinline__ __half* row_ptr(const Col& col, int m) const {
    const int b = div_by(m, seq, inv_seq), s = m - b * seq;
    return col.base + ((long)(b * heads + col.head) * col.len + s) * dim + col.off;
  }
  __device__ __forceinline__ void store4(int m, int, int, const Col& col, const v4i& c) const {
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = last(clips.value(c[k], __half2float(col.b.v[k])));
    *reinterpret_cast<half4_t*>(row_ptr(col, m)) = pack_half4(x[0], x[1], x[2], x[3]);
  }
  struct Col16 {
    Half16 b;
    __half* base;
    int head, len;
  };
  __device__ __forceinline__ Col16 column16(int n) const {
    const Col c = column(n, 0);
    return Col16{ld16(bias + n), c.base + c.off, c.head, c.len};
  }
  struct Row16 {
    int b, s;
  };
  __device__ __forceinline__ Row16 fetch16(int m, int, int) const {
    const int b = div_by(m, seq, inv_seq);
    return Row16{b, m - b * seq};
  }
  __device__ __forceinline__ void store16(long, int, int, const v16i& c, const Col16& col, const Row16& r) const {
    __half* p = col.base + ((long)(r.b * heads + col.head) * col.len + r.s) * dim;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8_t x;
#pragma unroll
      for (int k = 0; k < 8; ++k) x.v[k] = __float2half_rn(last(clips.value(c[8 * h + k], __half2float(col.b.h[h].v[k]))));
      st8(p + 8 * h, x);
    }
  }
  bool aligned() const { return true; }
};

// (dequantised code + bias) + residual (opb_quant_dropout_res_bias)
struct EpiResidual {
  static constexpr bool kTable = false, kBlockedOut = false, kClips = true, kFetch = true, kColumn16 = true,
                        kFetch16 = true;
  __half* out;
  const __half *bias, *residual;
  ProductClips clips;
  __device__ __forceinline__ ProductClips::Raw request() const { return clips.request(); }
  __device__ __forceinline__ EpiResidual finish(const ProductClips::Raw& r) const {
    EpiResidual e = *this;
    e.clips.finish(r);
    return e;
  }
  struct Col {
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    return Col{*reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ half4_t fetch(int m, int n, int N) const {
    return *reinterpret_cast<const half4_t*>(residual + (long)m * N + n);
  }
  __device__ __forceinline__ void store4(int m, int n, int N, const Col& col, const v4i& c, const half4_t& r) const {
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = clips.value(c[k], __half2float(col.b.v[k])) + __half2float(r.v[k]);
    *reinterpret_cast<half4_t*>(out + (long)m * N + n) = pack_half4(x[0], x[1], x[2], x[3]);
  }
  __device__ __forceinline__ Half16 column16(int n) const { return ld16(bias + n); }
  __device__ __forceinline__ Half16 fetch16(int m, int n, int N) const { return ld16(residual + (long)m * N + n); }
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, const Half16& b, const Half16& r) const {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8_t x;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        x.v[k] = __float2half_rn(clips.value(c[8 * h + k], __half2float(b.h[h].v[k])) + __half2float(r.h[h].v[k]));
      st8(out + m * N + n + 8 * h, x);
    }
  }
  bool aligned() const { return true; }
};

// activation(dequantised code + bias), fake-quantised, as the next product reads it: fp16, blocked
// (opb_quant_dropout_act_bias; in_cmax: that product's input clip)
template <bool RELU>
struct EpiAct {
  static constexpr bool kTable = false, kBlockedOut = true, kClips = true, kColumn16 = true;
  __half* out;
  int out_k;  // bytes of a row of `out`
  const __half *bias, *in_cmax;
  ProductClips clips;
  Quantiser in;
  struct Raw {
    ProductClips::Raw clips;
    __half in;
  };
  __device__ __forceinline__ Raw request() const { return Raw{clips.request(), in_cmax[0]}; }
  __device__ __forceinline__ EpiAct finish(const Raw& r) const {
    EpiAct e = *this;
    e.clips.finish(r.clips);
    e.in = Quantiser::of(__half2float(r.in), !RELU);
    return e;
  }
  struct Col {
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    return Col{*reinterpret_cast<const half4_t*>(bias + n)};
  }
  // (ReLU: the unsigned quantiser)
  __device__ __forceinline__ float value(int acc, __half b) const {
    const float x = act_b<__half, RELU ? 1 : 0>(clips.value(acc, __half2float(b)));
    return RELU ? in.fake_unsigned(x) : in.fake(x);
  }
  __device__ __forceinline__ half4_t four(const half4_t& b, int a0, int a1, int a2, int a3) const {
    return pack_half4(value(a0, b.v[0]), value(a1, b.v[1]), value(a2, b.v[2]), value(a3, b.v[3]));
  }
  __device__ __forceinline__ void store4(int m, int n, int, const Col& col, const v4i& c) const {
    *reinterpret_cast<half4_t*>(reinterpret_cast<char*>(out) + blocked_offset(m, 2 * n, out_k)) =
        four(col.b, c[0], c[1], c[2], c[3]);
  }
  __device__ __forceinline__ Half16 column16(int n) const { return ld16(bias + n); }
  __device__ __forceinline__ void store16(long m, int n, int, const v16i& c, const Half16& b) const {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8_t x;
#pragma unroll
      for (int k = 0; k < 8; ++k) x.v[k] = __float2half_rn(value(c[8 * h + k], b.h[h].v[k]));
      st8(reinterpret_cast<char*>(out) + blocked_offset(m, 2 * (n + 8 * h), out_k), x);
    }
  }
  bool aligned() const { return true; }
};

// second feed-forward product, fp16: (product, rounded as it was stored, + bias) + residual
// (opb_dropout_res_bias)
struct EpiFfn2 {
  static constexpr bool kTable = false, kBlockedOut = false, kFetch = true, kColumn16 = true, kFetch16 = true;
  __half* out;
  const __half *bias, *residual;
  struct Col {
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    return Col{*reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ half4_t fetch(int m, int n, int N) const {
    return *reinterpret_cast<const half4_t*>(residual + (long)m * N + n);
  }
  __device__ __forceinline__ void store4(int m, int n, int N, const Col& col, const v4f& c, const half4_t& r) const {
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = TT<__half>::rnd(TT<__half>::rnd(c[k]) + __half2float(col.b.v[k])) + __half2float(r.v[k]);
    *reinterpret_cast<half4_t*>(out + (long)m * N + n) = pack_half4(x[0], x[1], x[2], x[3]);
  }
  __device__ __forceinline__ Half16 column16(int n) const { return ld16(bias + n); }
  __device__ __forceinline__ Half16 fetch16(int m, int n, int N) const { return ld16(residual + (long)m * N + n); }
  __device__ __forceinline__ void store16(long m, int n, int N, const v16f& c, const Half16& b, const Half16& r) const {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8_t x;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        x.v[k] = __float2half_rn(TT<__half>::rnd(TT<__half>::rnd(c[8 * h + k]) + __half2float(b.h[h].v[k])) +
                                 __half2float(r.h[h].v[k]));
      st8(out + m * N + n + 8 * h, x);
    }
  }
  bool aligned() const { return true; }
};

// fp16 product [b * seq + s, 2 layers * hidden] -> keys (even parts) and values (odd parts)
// [b][head][s][d] of each layer, bias added in fp16 (opb_bias_add_transform_20314,
// arrange_encdec_kv)
struct EpiKv {
  static constexpr bool kTable = false, kBlockedOut = false, kColumn16 = true, kFetch16 = true;
  __half *k, *v;
  long layer_stride;
  const __half* bias;
  int seq, heads, dim, hidden;
  float inv_seq, inv_hidden, inv_dim;
  struct Col {
    __half* base;
    int head;
    half4_t b;
  };
  __device__ __forceinline__ Col column(int n, int) const {
    const int part = div_by(n, hidden, inv_hidden), i = n - part * hidden;
    const int head = div_by(i, dim, inv_dim);
    return Col{((part & 1) ? v : k) + (long)(part >> 1) * layer_stride + (i - head * dim), head,
               *reinterpret_cast<const half4_t*>(bias + n)};
  }
  __device__ __forceinline__ __half* row_ptr(const Col& col, int m) const {
    const int b = div_by(m, seq, inv_seq), s = m - b * seq;
    return col.base + ((long)(b * heads + col.head) * seq + s) * dim;
  }
  __device__ __forceinline__ half4_t four(const half4_t& b, float a0, float a1, float a2, float a3) const {
    return pack_half4(TT<__half>::rnd(a0) + __half2float(b.v[0]), TT<__half>::rnd(a1) + __half2float(b.v[1]),
                      TT<__half>::rnd(a2) + __half2float(b.v[2]), TT<__half>::rnd(a3) + __half2float(b.v[3]));
  }
  __device__ __forceinline__ void store4(int m, int, int, const Col& col, const v4f& c) const {
    *reinterpret_cast<half4_t*>(row_ptr(col, m)) = four(col.b, c[0], c[1], c[2], c[3]);
  }
  struct Col16 {
    Half16 b;
    __half* base;
    int head;
  };
  __device__ __forceinline__ Col16 column16(int n) const {
    const Col c = column(n, 0);
    return Col16{ld16(bias + n), c.base, c.head};
  }
  struct Row16 {
    int b, s;
  };
  __device__ __forceinline__ Row16 fetch16(int m, int, int) const {
    const int b = div_by(m, seq, inv_seq);
    return Row16{b, m - b * seq};
  }
  __device__ __forceinline__ void store16(long, int, int, const v16f& c, const Col16& col, const Row16& r) const {
    __half* p = col.base + ((long)(r.b * heads + col.head) * seq + r.s) * dim;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8_t x;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        x.v[k] = __float2half_rn(TT<__half>::rnd(c[8 * h + k]) + __half2float(col.b.h[h].v[k]));
      st8(p + 8 * h, x);
    }
  }
  bool aligned() const { return true; }
};

// The LDS tiles store 16 columns per lane: whole 16-byte pieces of one head only where heads are
// multiples of 16 (they are 32, 64 or 128 in layers).
bool bad_heads(int hidden, int heads, int rows) {
  return heads <= 0 || hidden % heads != 0 || (hidden / heads) % 16 != 0 || rows >= (1 << 22);
}

}  // namespace

template <bool CACHE>
static int heads_product(const int8_t* A, const int8_t* W, int rows, int parts, int hidden, int K,
                         const __half* bias, const __half* cmax, const __half* cache_cmax, int seq, int heads,
                         const HeadPart (&part)[3], hipStream_t s) {
  EpiHeads<CACHE> e{};
  e.p0 = part[0];
  e.p1 = part[1];
  e.p2 = part[2];
  e.bias = bias;
  e.cache_cmax = cache_cmax;
  e.clips.cmax = cmax;
  e.seq = seq;
  e.heads = heads;
  e.dim = hidden / heads;
  e.hidden = hidden;
  e.inv_seq = 1.0f / (float)seq;
  e.inv_hidden = 1.0f / (float)hidden;
  e.inv_dim = 1.0f / (float)e.dim;
  return dispatch_blk<KwI8, EpiHeads<CACHE>, true>(A, W, e, rows, parts * hidden, K, s);
}

int layer_gemm_heads(const int8_t* A, const int8_t* W, int rows, int parts, int hidden, int K,
                     const __half* bias, const __half* cmax, const __half* cache_cmax, int seq, int heads,
                     __half* const* base, const int* len, const int* at, hipStream_t s) {
  if (!bias || !cmax || !base || parts < 1 || parts > 3 || seq <= 0 || rows % seq != 0 ||
      bad_heads(hidden, heads, rows))
    return lsh_fail(LSH_ERR_INVALID, "layer_gemm_heads: bad arguments");
  HeadPart part[3] = {};
  for (int i = 0; i < parts; ++i) {
    if (!base[i] || at[i] < 0 || at[i] + seq > len[i])
      return lsh_fail(LSH_ERR_INVALID, "layer_gemm_heads: bad destination");
    part[i] = HeadPart{base[i], len[i], at[i]};
  }
  return cache_cmax ? heads_product<true>(A, W, rows, parts, hidden, K, bias, cmax, cache_cmax, seq, heads, part, s)
                    : heads_product<false>(A, W, rows, parts, hidden, K, bias, cmax, nullptr, seq, heads, part, s);
}

int layer_gemm_residual(const int8_t* A, const int8_t* W, int rows, int N, int K, const __half* bias,
                        const __half* cmax, const __half* residual, __half* out, hipStream_t s) {
  if (!bias || !cmax || !residual || !out) return lsh_fail(LSH_ERR_INVALID, "layer_gemm_residual: null pointer");
  EpiResidual e{};
  e.out = out;
  e.bias = bias;
  e.residual = residual;
  e.clips.cmax = cmax;
  return dispatch_blk<KwI8, EpiResidual, true>(A, W, e, rows, N, K, s);
}

template <bool RELU>
static int act(const int8_t* A, const int8_t* W, int rows, int N, int K, const __half* bias,
               const __half* cmax, const __half* in_cmax, __half* out, int out_k, hipStream_t s) {
  EpiAct<RELU> e{};
  e.out = out;
  e.out_k = 2 * out_k;
  e.bias = bias;
  e.in_cmax = in_cmax;
  e.clips.cmax = cmax;
  return dispatch_blk<KwI8, EpiAct<RELU>, true>(A, W, e, rows, N, K, s);
}
int layer_gemm_act(const int8_t* A, const int8_t* W, int rows, int N, int K, const __half* bias,
                   const __half* cmax, const __half* in_cmax, bool relu, __half* out, int out_k,
                   hipStream_t s) {
  if (!bias || !cmax || !in_cmax || !out || out_k < N || out_k % 32 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_gemm_act: bad arguments");
  return relu ? act<true>(A, W, rows, N, K, bias, cmax, in_cmax, out, out_k, s)
              : act<false>(A, W, rows, N, K, bias, cmax, in_cmax, out, out_k, s);
}

int layer_gemm_ffn2(const __half* A, const __half* W, int rows, int N, int K, const __half* bias,
                    const __half* residual, __half* out, hipStream_t s) {
  if (!bias || !residual || !out) return lsh_fail(LSH_ERR_INVALID, "layer_gemm_ffn2: null pointer");
  return dispatch_f16(reinterpret_cast<const int8_t*>(A),
                                            reinterpret_cast<const int8_t*>(W), EpiFfn2{out, bias, residual},
                                            rows, N, 2 * K, s);
}

int gemm_blk_kv_f16(const __half* A, const __half* W, int rows, int layers, int hidden, int K,
                    const __half* bias, int seq, int heads, __half* k, __half* v, long layer_stride,
                    hipStream_t s) {
  if (!bias || !k || !v || layers <= 0 || seq <= 0 || rows % seq != 0 || bad_heads(hidden, heads, rows) ||
      (long)layers * 2 * hidden >= (1 << 22))
    return lsh_fail(LSH_ERR_INVALID, "gemm_blk_kv_f16: bad arguments");
  EpiKv e{};
  e.k = k;
  e.v = v;
  e.layer_stride = layer_stride;
  e.bias = bias;
  e.seq = seq;
  e.heads = heads;
  e.dim = hidden / heads;
  e.hidden = hidden;
  e.inv_seq = 1.0f / (float)seq;
  e.inv_hidden = 1.0f / (float)hidden;
  e.inv_dim = 1.0f / (float)e.dim;
  return dispatch_f16(reinterpret_cast<const int8_t*>(A),
                                          reinterpret_cast<const int8_t*>(W), e, rows, layers * 2 * hidden,
                                          K * 2, s);
}

}  // namespace lsh
