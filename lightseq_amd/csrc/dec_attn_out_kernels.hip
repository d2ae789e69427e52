// Decoder self attention of a step with the out-projection behind it (out_product.h), heads of 64.
#include "dec_attend.h"
#include "ls_launch.h"
#include "out_product.h"

namespace lsh {

// Eight wavefronts.  ROWS == 1: one (row, head) pair on NWV of them, as decself_attn_wg_kernel;
// ROWS == 4: four rows of a head, a wavefront each, as decself_attn_pack_kernel does with caches
// that one wavefront's loads cover.  The same bodies and the same choice by cache length, hence the
// same context codes; they stay in LDS.  The other wavefronts bring weights meanwhile.
template <int NWV, int UN, int ROWS, int N, bool BY_BEAM>
__global__ void __launch_bounds__(512)
decself_out_kernel(const int8_t* __restrict__ q, const int8_t* __restrict__ k_cache,
                   const int8_t* __restrict__ v_cache, const int8_t* __restrict__ beam_from, int step_num,
                   int max_step, int head_num, int beam_stride, const int8_t* __restrict__ W, int32_t* acc,
                   int32_t* next_acc, int32_t* ffn_acc, int rows, float attn_scale, float dq, float quant_scale) {
  constexpr int D = 64, CH = D / 16, ATTEND = ROWS == 4 ? 4 : NWV;
  extern __shared__ __align__(16) float lds_f[];
  __shared__ __align__(16) int8_t ctx[ROWS * D];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int head = (int)blockIdx.x, row0 = (int)blockIdx.y * ROWS, hidden = head_num * D;
  const int first = ((int)blockIdx.z * 8 + wave) * N;  // block of columns
  OutFragments<N> out;
  if (wave < ATTEND) {
    const int slot = ROWS == 4 ? wave : 0, wid = ROWS == 4 ? 0 : wave;
    const int row = min(row0 + slot, rows - 1);
    const long bh = (long)row * head_num + head;
    const uint4 qv = *reinterpret_cast<const uint4*>(q + bh * D + (lane % CH) * 16);
    const int8_t *kb = k_cache + bh * (long)max_step * D, *vb = v_cache + bh * (long)max_step * D;
    uint4 kv[UN], vv[UN];
    if constexpr (BY_BEAM)
      decself_attend_load_rows<D, NWV, UN>(
          kb, vb, RowsByBeam<D>{beam_from + (long)row * beam_stride, step_num - 1, (long)head_num * max_step * D},
          step_num, wid, lane, kv, vv);
    else
      decself_attend_load_rows<D, NWV, UN>(kb, vb, RowsInPlace<D>{}, step_num, wid, lane, kv, vv);
    __builtin_amdgcn_sched_barrier(0);
    out.request(W, head, head_num, first, lane);
    __builtin_amdgcn_sched_barrier(0);
    // (three barriers)
    decself_attend_row_once_body<D, NWV, UN>(qv, kv, vv, ctx + slot * D, true, 16, step_num, attn_scale, dq,
                                             quant_scale, lds_f + slot * decself_group_floats<D, 1>(step_num), wid,
                                             lane);
  } else {
    out.request(W, head, head_num, first, lane);
    __syncthreads();
    __syncthreads();
    __syncthreads();
  }
  // the workgroup's share of the next launch's sums and the feed-forward block's: its rows, 64 columns
  if (blockIdx.z == 0 && (int)threadIdx.x < ROWS * 16) {
    const int r = row0 + ((int)threadIdx.x >> 4);
    const long at = (long)r * hidden + head * D + (threadIdx.x & 15) * 4;
    if (r < rows) {
      *reinterpret_cast<int4*>(next_acc + at) = make_int4(0, 0, 0, 0);
      *reinterpret_cast<int4*>(ffn_acc + at) = make_int4(0, 0, 0, 0);
    }
  }
  __syncthreads();
  out.template add<ROWS>(ctx, acc + (long)row0 * hidden, rows - row0, hidden, first, lane);
}

// The workgroups that fit one round of the chip: beyond it every one of them brings its head's weights
// again (64 KB each), and a product of that many rows reads them once.
bool decself_attention_out_supported(int rows, int head_num, int dim_per_head, int step_num) {
  if (dim_per_head != 64 || head_num < 2 || head_num > 16 || head_num % 2 != 0 || rows < 1 || step_num < 1 ||
      step_num > 1024)
    return false;
  return (step_num <= 128 ? (rows + 3) / 4 : rows) * head_num <= cu_count();
}

int decself_attention_out_i8(const int8_t* q, const int8_t* k_cache, const int8_t* v_cache, const int8_t* W,
                             int32_t* acc, int32_t* next_acc, int32_t* ffn_acc, int rows, int step_num, int max_step,
                             int head_num, float attn_scale, float dequant_scale, float quant_scale, hipStream_t s,
                             const CacheBeams* beams) {
  if (!q || !k_cache || !v_cache || !W || !acc || !next_acc || !ffn_acc || acc == next_acc || acc == ffn_acc || step_num > max_step ||
      (beams && (!beams->from || beams->stride < max_step)))
    return lsh_fail(LSH_ERR_INVALID, "decself_attention_out: bad arguments");
  if (!decself_attention_out_supported(rows, head_num, 64, step_num) || rows > 65535 || max_step > 4096)
    return lsh_fail(LSH_ERR_UNSUPPORTED, "decself_attention_out: shape not covered");
  if (((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) |
        reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(acc) |
        reinterpret_cast<uintptr_t>(next_acc) | reinterpret_cast<uintptr_t>(ffn_acc)) & 15u) != 0)
    return lsh_fail(LSH_ERR_INVALID, "decself_attention_out: operands must be 16-byte aligned");
  const CacheBeams by = beams ? *beams : CacheBeams{};
#define LSH_OUT_RUN(NWV, UN, ROWS, N, BY)                                                                      \
  decself_out_kernel<NWV, UN, ROWS, N, BY>                                                                     \
      <<<dim3(head_num, (rows + ROWS - 1) / ROWS, 8 / N), 512,                                                  \
         ROWS * decself_group_floats<64, NWV>(step_num) * sizeof(float), s>>>(                                 \
          q, k_cache, v_cache, by.from, step_num, max_step, head_num, by.stride, W, acc, next_acc, ffn_acc,    \
          rows, attn_scale, dequant_scale, quant_scale)
#define LSH_OUT_BY(NWV, UN, ROWS, N) \
  do { if (beams) LSH_OUT_RUN(NWV, UN, ROWS, N, true); else LSH_OUT_RUN(NWV, UN, ROWS, N, false); } while (0)
#define LSH_OUT(NWV, UN, ROWS)                                               \
  do {                                                                       \
    const int share = out_product_share((rows + ROWS - 1) / ROWS * head_num); \
    if (share == 8) LSH_OUT_BY(NWV, UN, ROWS, 1);                            \
    else if (share == 4) LSH_OUT_BY(NWV, UN, ROWS, 2);                         \
    else if (share == 2) LSH_OUT_BY(NWV, UN, ROWS, 4);                       \
    else LSH_OUT_BY(NWV, UN, ROWS, 8);                                       \
  } while (0)
  const int un8 = (step_num + 127) / 128;  // as decself_attention_i8 chooses
  if (step_num <= 64) LSH_OUT(1, 4, 4);
  else if (step_num <= 128) LSH_OUT(1, 8, 4);
  else if (step_num <= 256) LSH_OUT(4, 4, 1);
  else if (un8 <= 3) LSH_OUT(8, 3, 1);
  else if (un8 == 4) LSH_OUT(8, 4, 1);
  else if (un8 == 5) LSH_OUT(8, 5, 1);
  else if (un8 == 6) LSH_OUT(8, 6, 1);
  else LSH_OUT(8, 8, 1);
#undef LSH_OUT
#undef LSH_OUT_BY
#undef LSH_OUT_RUN
  return lsh_check_launch("decself_out_kernel");
}

}  // namespace lsh
