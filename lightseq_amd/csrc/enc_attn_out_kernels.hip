// Encoder self attention of a batch of few tokens with the out-projection behind it (out_product.h).
//
// For a handful of tokens the launch that multiplies QKV per (sequence, head) (qkv_attn_kernels.hip)
// waits for one compute unit to read a head's 147 to 196 KB of weights: 7.7 us for 16 tokens of
// hidden 768, and the out-projection takes 2.6 us behind it.  The QKV product spread over the chip takes 2.9 us,
// and this launch, which starts from its codes and ends in the out-projection's sums, 4.5 us.
// The sums of `rows` rows take heads * rows * hidden adds, so there is an end to it.  us of a call, fused
// launch and this route: 12 layers of 768 16 rows 288 and 247, 64 rows 301 and 276, 96 rows 322 and 300,
// 128 rows 325 and 319; 6 layers of 1024 160 and 134, 167 and 154, 180 and 176, 184 and 190.
#include "ls_launch.h"
#include "out_product.h"
#include "tile_common.h"

#include <algorithm>

namespace lsh {

// Eight wavefronts to a (head, sequence) pair, or to a share of its columns (blockIdx.z).  Codes to fp16 q,
// k and transposed v in LDS with the values the product's epilogue in qkv_attn_kernel leaves, a
// wavefront to 32 queries, the context codes to LDS, 16 N columns of the out-projection a wavefront.
// MAXB: the blocks of 32 tokens there can be.  clear: `clear_n` ints, dealt over the launch.
template <int MAXB, int N>
__global__ void __launch_bounds__(512)
enc_attn_out_kernel(const int8_t* __restrict__ qkv, const int* __restrict__ seq,
                    const _Float16* __restrict__ bias, const int* __restrict__ pad_mask,
                    const int8_t* __restrict__ W, int32_t* acc, int4* clear, int S, int head_num, int clear_n4,
                    float dq, float quant_scale, float alpha) {
  constexpr int D = 64, KSTR = attn_kstr(D), VSTR = kAttnVstr, CPT = (MAXB * 384 + 511) / 512;
  __shared__ __align__(16) _Float16 Qs[MAXB * 32 * KSTR], Ks[MAXB * 32 * KSTR], Vt[D * VSTR];
  __shared__ __align__(16) int8_t ctx[MAXB * 32 * D];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = (int)blockIdx.x, b = (int)blockIdx.y, hidden = head_num * D;
  const int l32 = lane & 31, g = lane >> 5, first = ((int)blockIdx.z * 8 + wave) * N;
  const int row0 = __builtin_amdgcn_readfirstlane(seq[2 * b]), len = __builtin_amdgcn_readfirstlane(seq[2 * b + 1]);
  {
    const int wgs = gridDim.x * gridDim.y * gridDim.z;
    const int wg = ((int)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    for (int i = wg * 512 + tid; i < clear_n4; i += wgs * 512) clear[i] = make_int4(0, 0, 0, 0);
  }
  if (len == 0) return;
  const int nblk = (len + 31) >> 5, chunks = nblk * 384;
  uint4 w[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = min(tid + i * 512, chunks - 1), row = c / 12, ch = c % 12;
    w[i] = *reinterpret_cast<const uint4*>(qkv + (long)(row0 + min(row, len - 1)) * 3 * hidden + (ch >> 2) * hidden +
                                           head * D + (ch & 3) * 16);
  }
  const int pm0 = pad_mask[(long)b * S + min(lane, len - 1)];
  const int pm1 = pad_mask[(long)b * S + min(lane + 64, len - 1)];
  __builtin_amdgcn_sched_barrier(0);
  OutFragments<N> out;
  out.request(W, head, head_num, first, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = tid + i * 512, row = c / 12, ch = c % 12, part = ch >> 2, d0 = (ch & 3) * 16;
    if (c >= chunks) continue;
    v8h lo, hi;
    dequant16_bias(w[i], bias + part * hidden + head * D + d0, dq, lo, hi);
    if (row >= len) lo = hi = (v8h)(_Float16)0;
    if (part == 2) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        Vt[(d0 + e) * VSTR + row] = lo[e];
        Vt[(d0 + 8 + e) * VSTR + row] = hi[e];
      }
    } else {
      _Float16* dst = (part == 0 ? Qs : Ks) + row * KSTR + d0;
      *reinterpret_cast<v8h*>(dst) = lo;
      *reinterpret_cast<v8h*>(dst + 8) = hi;
    }
  }
  __syncthreads();
  if (wave < nblk) {
    const int qi = wave * 32 + l32;
    v8h qreg[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
      qreg[ks] = *reinterpret_cast<const v8h*>(&Qs[qi * KSTR + ks * 16 + g * 8]);
    const bool padk0 = pm0 != 0 || lane >= len, padk1 = pm1 != 0 || lane + 64 >= len;
    const uint64_t pad_q = __ballot(wave < 2 ? padk0 : padk1);
    const bool q_pad = qi >= len || ((pad_q >> ((wave & 1) * 32 + l32)) & 1) != 0;
    int8_t* o = ctx + qi * D;
    if (MAXB >= 3 && nblk == 3)
      attend_block128<D, MAXB >= 3 ? 3 : 1>(Ks, Vt, qreg, padk0, padk1, q_pad, true, alpha, quant_scale, nullptr, o,
                                            l32, g);
    else if (MAXB >= 2 && nblk == 2)
      attend_block128<D, MAXB >= 2 ? 2 : 1>(Ks, Vt, qreg, padk0, padk1, q_pad, true, alpha, quant_scale, nullptr, o,
                                            l32, g);
    else
      attend_block128<D, 1>(Ks, Vt, qreg, padk0, padk1, q_pad, true, alpha, quant_scale, nullptr, o, l32, g);
  }
  __syncthreads();
  out.add_rows(ctx, acc + (long)row0 * hidden, len, hidden, first, lane);
}

bool enc_attention_out_supported(int batch, int seq_len, int head_num, int dim_per_head) {
  return dim_per_head == 64 && head_num >= 2 && head_num <= 16 && head_num % 2 == 0 && batch >= 1 && seq_len >= 1 &&
         (long)batch * seq_len <= kEncOutPositions;
}

int enc_attention_out(const int8_t* qkv, const __half* qkv_bias, float dequant_scale, const int* pad_mask,
                      const int8_t* W, int32_t* acc, int32_t* clear, int clear_rows, float quant_scale, int batch,
                      int seq_len, int head_num, hipStream_t s, const EncPack& pack) {
  if (!qkv || !qkv_bias || !pad_mask || !W || !acc || !clear || clear_rows <= 0 || !pack.seq ||
      (acc < clear + (long)clear_rows * head_num * 64 && clear < acc + (long)batch * seq_len * head_num * 64))
    return lsh_fail(LSH_ERR_INVALID, "enc_attention_out: bad arguments");
  if (!enc_attention_out_supported(batch, seq_len, head_num, 64))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "enc_attention_out: shape not covered");
  if (((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(qkv_bias) | reinterpret_cast<uintptr_t>(W) |
        reinterpret_cast<uintptr_t>(acc) | reinterpret_cast<uintptr_t>(clear)) & 15u) != 0)
    return lsh_fail(LSH_ERR_INVALID, "enc_attention_out: operands must be 16-byte aligned");
  const int hidden = head_num * 64, pairs = head_num * batch;
  const float alpha = __half2float(__float2half_rn(sqrtf(1.f / 64.f)));
  auto shares = [&](int n) { return (hidden / 16 + 8 * n - 1) / (8 * n); };
#define LSH_ENC_OUT_RUN(MAXB, N)                                                                              \
  enc_attn_out_kernel<MAXB, N><<<dim3(head_num, batch, shares(N)), 512, 0, s>>>(                              \
      qkv, pack.seq, reinterpret_cast<const _Float16*>(qkv_bias), pad_mask, W, acc,                           \
      reinterpret_cast<int4*>(clear), seq_len, head_num, clear_rows * hidden / 4, dequant_scale,      \
      quant_scale, alpha)
#define LSH_ENC_OUT(MAXB)                                            \
  do {                                                               \
    if (pairs * shares(1) <= cu_count()) LSH_ENC_OUT_RUN(MAXB, 1);   \
    else if (pairs * shares(2) <= cu_count()) LSH_ENC_OUT_RUN(MAXB, 2); \
    else if (pairs * shares(4) <= cu_count()) LSH_ENC_OUT_RUN(MAXB, 4); \
    else LSH_ENC_OUT_RUN(MAXB, 8);                                   \
  } while (0)
  if (seq_len <= 32) LSH_ENC_OUT(1);
  else if (seq_len <= 64) LSH_ENC_OUT(2);
  else LSH_ENC_OUT(3);
#undef LSH_ENC_OUT
#undef LSH_ENC_OUT_RUN
  return lsh_check_launch("enc_attn_out_kernel");
}

}  // namespace lsh
