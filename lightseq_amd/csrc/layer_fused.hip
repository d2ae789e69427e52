// What a quantised layer needs ahead of and between its products (layer_gemm.hip), in as few
// launches as there are dependencies: one that prepares everything the forward pass starts from,
// and the layer norm between two products.
#include "layer_prep.h"
#include "ls_launch.h"

#include <algorithm>
#include <type_traits>

namespace lsh {

namespace {

// ---- one launch for all of a layer's preparations -------------------------------------------
// The parameters belong to the caller and may have changed since the last call, so every forward
// pass quantises the weights (2 bytes read and 1 written per parameter: 10 MB for a
// Transformer-base layer).  As one launch per matrix that was 4 us each, six to nine times per
// layer; the sections below -- weights, the input, the mask, the copy of a decoding step's caches
// -- do not depend on one another, so they are ranges of workgroups of one grid (all of them, by the
// kernel trace: 8.0 us for a Transformer-base encoder layer, 10 MB, and 18 us for a step of a
// Transformer-big decoder layer, 64 MB with its caches, 3.6 TB/s).  Weights that only later products
// read ride in the launches between (layer_prep.h); the rest takes 4.0 and 9.5 us.
// eight normalised elements to where they go (`out`, `codes`: null where nobody reads them)
__device__ __forceinline__ void ln_store(const half8_t& x, const half8_t& g, const half8_t& b, float mean, float rstd,
                                         const Quantiser& of, __half* out, int8_t* codes) {
  half8_t o;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    o.v[k] = __float2half_rn((__half2float(x.v[k]) - mean) * rstd * __half2float(g.v[k]) + __half2float(b.v[k]));
  if (out) *reinterpret_cast<half8_t*>(out) = o;
  if (codes) *reinterpret_cast<uint2*>(codes) = codes8(of, o);
}

// Layer norm of one row by a wavefront (opb_layer_norm: var = E[x^2] - E[x]^2 + 1e-8), the row kept
// in registers where it is at most 512 IT elements; the codes of the fp16 result, blocked.
template <int IT>
__device__ __forceinline__ void ln_row(const __half* inp, __half* out, int8_t* codes, const __half* gamma,
                                       const __half* beta, const __half* cmax, int row, int hidden, int k_pad) {
  const int lane = threadIdx.x & 63;
  const long base = (long)row * hidden;
  half8_t raw[IT], g[IT], b[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int e = min(lane * 8 + it * 512, hidden - 8);
    raw[it] = *reinterpret_cast<const half8_t*>(inp + base + e);
    g[it] = *reinterpret_cast<const half8_t*>(gamma + e);
    b[it] = *reinterpret_cast<const half8_t*>(beta + e);
  }
  const Quantiser of = Quantiser::of(codes ? cm(cmax) : 1.f);
  float s = 0.f, s2 = 0.f;
#pragma unroll
  for (int it = 0; it < IT; ++it)
    if (lane * 8 + it * 512 < hidden) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = __half2float(raw[it].v[k]);
        s += x;
        s2 += x * x;
      }
    }
  const float mean = wave_sum(s) / (float)hidden;
  const float var = wave_sum(s2) / (float)hidden - mean * mean + kLnEps;
  const float rstd = rsqrtf(var);
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int e = lane * 8 + it * 512;
    if (e >= hidden) continue;
    ln_store(raw[it], g[it], b[it], mean, rstd, of, out ? out + base + e : nullptr,
             codes ? codes + blocked_offset(row, e, k_pad) : nullptr);
  }
}
// Rows that do not fit the registers are read twice, the second time from the cache (in place: a lane
// writes only what it has read itself).  Same sums in the same order.
__device__ __forceinline__ void ln_row_long(const __half* inp, __half* out, int8_t* codes, const __half* gamma,
                                            const __half* beta, const __half* cmax, int row, int hidden,
                                            int k_pad) {
  const int lane = threadIdx.x & 63;
  const long base = (long)row * hidden;
  float s = 0.f, s2 = 0.f;
  for (int e = lane * 8; e < hidden; e += 512) {
    const half8_t raw = *reinterpret_cast<const half8_t*>(inp + base + e);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float x = __half2float(raw.v[k]);
      s += x;
      s2 += x * x;
    }
  }
  const float mean = wave_sum(s) / (float)hidden;
  const float var = wave_sum(s2) / (float)hidden - mean * mean + kLnEps;
  const float rstd = rsqrtf(var);
  const Quantiser of = Quantiser::of(codes ? cm(cmax) : 1.f);
  for (int e = lane * 8; e < hidden; e += 512) {
    const half8_t raw = *reinterpret_cast<const half8_t*>(inp + base + e);
    ln_store(raw, *reinterpret_cast<const half8_t*>(gamma + e), *reinterpret_cast<const half8_t*>(beta + e), mean,
             rstd, of, out ? out + base + e : nullptr, codes ? codes + blocked_offset(row, e, k_pad) : nullptr);
  }
}
__device__ __forceinline__ void ln_row_any(const __half* inp, __half* out, int8_t* codes, const __half* gamma,
                                           const __half* beta, const __half* cmax, int row, int hidden,
                                           int k_pad) {
  if (hidden <= 512) ln_row<1>(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
  else if (hidden <= 1024) ln_row<2>(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
  else if (hidden <= 2048) ln_row<4>(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
  else if (hidden <= 4096) ln_row<8>(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
  else ln_row_long(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
}

// the additive fp16 mask of the layers, half(value * -1e8), from whatever the caller's mask is made of
__device__ __forceinline__ float mask_value(const void* p, int kind, long i) {
  switch (kind) {
    case kMaskF32: return static_cast<const float*>(p)[i];
    case kMaskF16: return __half2float(static_cast<const __half*>(p)[i]);
    case kMaskU8: return (float)static_cast<const unsigned char*>(p)[i];
    case kMaskI32: return (float)static_cast<const int*>(p)[i];
    default: return (float)static_cast<const long long*>(p)[i];
  }
}

// (arguments for as many sections as a call has, or a few more: a launch with 1.2 KB of them costs the
// host 3.1 us, with 0.3 KB 2.5)
template <int MOST>
struct LayerPrepArgs {
  int first[MOST];  // first workgroup of each section
  LayerPrepSection s[MOST];
};
template <int MOST>
__global__ void __launch_bounds__(256)
layer_prep_kernel(const LayerPrepArgs<MOST> a) {
  // the section that the workgroup belongs to: the first blocks are read together and compared, a
  // walk would be as many trips to the kernel arguments
  int i = 0, first = 0;
#pragma unroll
  for (int j = 1; j < MOST; ++j)
    if ((int)blockIdx.x >= a.first[j]) {
      i = j;
      first = a.first[j];
    }
  const int block = (int)blockIdx.x - first;
  const LayerPrepSection& s = a.s[i];
  switch (s.kind) {
    case kPrepCodes: unit_codes(s, block, (int)(threadIdx.x >> 6)); break;
    case kPrepHalfs: unit_halfs(s, block, (int)(threadIdx.x >> 6)); break;
    case kPrepNorm: {
      const int row = block * 4 + (int)(threadIdx.x >> 6);
      if (row < s.rows)
        ln_row_any(s.src, nullptr, static_cast<int8_t*>(s.dst), s.gamma, s.beta, s.cmax, row, s.K, s.k_pad);
      break;
    }
    case kPrepMask: {
      const long j = (long)block * 256 + threadIdx.x;
      if (j < s.rows)
        static_cast<__half*>(s.dst)[j] = __float2half_rn(mask_value(s.src, s.n1, j) * -1e8f);
      break;
    }
    default: {  // kPrepGrow: [rows, K] -> the first K of rows of stride1 elements, 2048 elements per block
      const long j = ((long)block * 256 + threadIdx.x) * 8;
      if (j < (long)s.rows * s.K) {
        const long r = j / s.K, c = j - r * s.K;
        *reinterpret_cast<half8_t*>(static_cast<__half*>(s.dst) + r * s.stride1 + c) =
            *reinterpret_cast<const half8_t*>(s.src + j);
      }
    }
  }
}

struct NoRide {};
template <typename Ride>
__global__ void __launch_bounds__(256)
layer_norm_codes_kernel(const __half* inp, __half* out, int8_t* codes, const __half* __restrict__ gamma,
                        const __half* __restrict__ beta, const __half* __restrict__ cmax, int rows,
                        int hidden, int k_pad, const Ride also) {
  const int row = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if constexpr (!std::is_same<Ride, NoRide>::value) {
    const int blocks = (rows + 3) >> 2;
    if ((int)blockIdx.x >= blocks) return ride_unit(also, (int)blockIdx.x - blocks, (int)(threadIdx.x >> 6));
  }
  if (row < rows) ln_row_any(inp, out, codes, gamma, beta, cmax, row, hidden, k_pad);
}

}  // namespace

int LayerPrep::add(const LayerPrepSection& s) {
  if (_n >= kLayerPrepMost) return lsh_fail(LSH_ERR_UNSUPPORTED, "layer_prep: too many sections");
  _s[_n++] = s;
  return LSH_OK;
}

static int prep_units(int rows, int K) { return (rows + 15) / 16 * ((K + kUnitK - 1) / kUnitK); }

int LayerPrep::codes(const __half* src, int8_t* dst, const __half* cmax, int rows, int K, int k_pad) {
  if (!src || !dst || !cmax || rows <= 0 || K <= 0 || K % 8 != 0 || k_pad < K || k_pad % 64 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_prep: bad matrix");
  LayerPrepSection s{};
  s.kind = kPrepCodes;
  s.blocks = prep_units(rows, K);
  s.src = src;
  s.dst = dst;
  s.cmax = cmax;
  s.rows = rows;
  s.K = K;
  s.k_pad = k_pad;
  s.n1 = 1;
  s.stride0 = K;
  return add(s);
}
int LayerPrep::halfs(const __half* src, __half* dst, const __half* cmax, int rows, int K, int k_pad, int n1,
                     long stride0, long stride1) {
  if (!src || !dst || rows <= 0 || K <= 0 || K % 8 != 0 || k_pad < K || k_pad % 32 != 0 || n1 <= 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_prep: bad fp16 matrix");
  LayerPrepSection s{};
  s.kind = kPrepHalfs;
  s.blocks = prep_units(rows, K);
  s.src = src;
  s.dst = dst;
  s.cmax = cmax;
  s.rows = rows;
  s.K = K;
  s.k_pad = k_pad;
  s.n1 = n1;
  s.stride0 = stride0;
  s.stride1 = stride1;
  return add(s);
}
int LayerPrep::norm(const __half* src, int8_t* dst, const __half* gamma, const __half* beta,
                    const __half* cmax, int rows, int hidden, int k_pad) {
  if (!src || !dst || !gamma || !beta || !cmax || rows <= 0 || hidden <= 0 || hidden % 8 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_prep: bad layer norm");
  LayerPrepSection s{};
  s.kind = kPrepNorm;
  s.blocks = (rows + 3) / 4;
  s.src = src;
  s.dst = dst;
  s.gamma = gamma;
  s.beta = beta;
  s.cmax = cmax;
  s.rows = rows;
  s.K = hidden;
  s.k_pad = k_pad;
  return add(s);
}
int LayerPrep::mask(const void* src, int kind, __half* dst, int count) {
  if (!src || !dst || count <= 0 || kind < kMaskF32 || kind > kMaskI64)
    return lsh_fail(LSH_ERR_INVALID, "layer_prep: bad mask");
  LayerPrepSection s{};
  s.kind = kPrepMask;
  s.blocks = (count + 255) / 256;
  s.src = static_cast<const __half*>(src);
  s.dst = dst;
  s.rows = count;
  s.n1 = kind;
  return add(s);
}
int LayerPrep::grow(const __half* src, __half* dst, int rows, int K, long dst_stride) {
  if (!src || !dst || rows <= 0 || K <= 0 || K % 8 != 0 || dst_stride < K || dst_stride % 8 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_prep: bad cache copy");
  LayerPrepSection s{};
  s.kind = kPrepGrow;
  s.blocks = (int)(((long)rows * K / 8 + 255) / 256);
  s.src = src;
  s.dst = dst;
  s.rows = rows;
  s.K = K;
  s.stride1 = dst_stride;
  return add(s);
}
int LayerPrep::ride(LayerRide* out) const {
  LayerRide r{};
  if (_n > kLayerRideMost) return lsh_fail(LSH_ERR_UNSUPPORTED, "layer_prep: too many sections to ride");
  for (int i = 0; i < kLayerRideMost; ++i) {
    r.first[i] = i < _n ? r.blocks : 0x7fffffff;
    if (i >= _n) continue;
    if (_s[i].kind != kPrepCodes && _s[i].kind != kPrepHalfs)
      return lsh_fail(LSH_ERR_UNSUPPORTED, "layer_prep: only matrices ride");
    r.s[i] = _s[i];
    r.blocks += _s[i].blocks;
  }
  if (r.blocks >= (1 << 26)) return lsh_fail(LSH_ERR_UNSUPPORTED, "layer_prep: too many workgroups");
  *out = r;
  return LSH_OK;
}

template <int MOST>
static int launch_prep(const LayerPrepSection* sections, int n, hipStream_t s) {
  LayerPrepArgs<MOST> args;
  long blocks = 0;
  for (int i = 0; i < MOST; ++i) {
    args.first[i] = i < n ? (int)std::min(blocks, 0x7fffffffL) : 0x7fffffff;
    if (i >= n) continue;
    args.s[i] = sections[i];
    blocks += sections[i].blocks;
  }
  if (blocks <= 0) return LSH_OK;
  if (blocks >= (1L << 30)) return lsh_fail(LSH_ERR_UNSUPPORTED, "layer_prep: too many workgroups");
  layer_prep_kernel<MOST><<<(unsigned)blocks, 256, 0, s>>>(args);
  return lsh_check_launch("layer_prep_kernel");
}
int LayerPrep::launch(hipStream_t s) const {
  if (_n <= 3) return launch_prep<3>(_s, _n, s);
  if (_n <= 5) return launch_prep<5>(_s, _n, s);
  return launch_prep<kLayerPrepMost>(_s, _n, s);
}

int layer_norm_codes(const __half* inp, __half* out, int8_t* codes, const __half* gamma, const __half* beta,
                     const __half* cmax, int rows, int hidden, int k_pad, hipStream_t s, const LayerPrep* also) {
  LayerRide ride{};
  if (also)
    if (int rc = also->ride(&ride)) return rc;
  if (!inp || (!out && !codes) || !gamma || !beta || (codes && !cmax) || rows <= 0 || hidden <= 0 ||
      hidden % 8 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer_norm_codes: bad arguments");
  const int blocks = (rows + 3) / 4;
  if (ride.blocks > 0)
    layer_norm_codes_kernel<LayerRide><<<blocks + ride.blocks, 256, 0, s>>>(inp, out, codes, gamma, beta, cmax, rows,
                                                                            hidden, k_pad, ride);
  else
    layer_norm_codes_kernel<NoRide><<<blocks, 256, 0, s>>>(inp, out, codes, gamma, beta, cmax, rows, hidden, k_pad,
                                                           NoRide{});
  return lsh_check_launch("layer_norm_codes_kernel");
}

}  // namespace lsh
