// int8 and fp16 products on blocked operands (blocked_offset in ls_device.h is the layout): what the models and
// layers run.  Weights are blocked once at load; activations are written blocked by the kernel
// that produces them (layer norm, attention, the table epilogue), so no product waits for a
// rearrangement.
//
// Two kernels: gemm_kw_kernel (gemm_kw.h) for outputs of up to a few rounds of small tiles, and
// the LDS tile loop of gemm_tile.h for the large ones.  The dispatch estimates both.
#include "gemm_blk_dispatch.h"
#include "gemm_dec_epi.h"
#include "ln_step.h"

namespace lsh {

// A product of one to four rows that makes its rows itself (ln_step.h): 16 columns per workgroup,
// a quarter of K per wavefront (D slices), its weights requested right behind the inputs of
// the layer norm and in flight while it runs.  Everything after the codes is gemm_kw_kernel's.
// us per generation step of a GPT-2 medium shape, batch 1: 573 -> 457.
template <typename Epi, int PLANES, int ROWS, int D>
__global__ void __launch_bounds__(256)
ln_gemm_kernel(const int8_t* __restrict__ W, int M, int N, int K, const LnStep ln, Epi epi) {
  extern __shared__ __align__(16) int8_t smem[];
  __shared__ __align__(16) float red_ln[2 * ROWS * 4];
  int8_t* codes = smem;           // [16 rows, K] blocked
  int8_t* part = smem + 16 * K;   // partial sums, then the table rows: as in gemm_kw_kernel
  int8_t* tab = part + 4 * 68 * 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  const int n0 = blockIdx.x * 16;
  // every argument in one batch of scalar loads
  asm volatile("" ::"s"(W), "s"(M), "s"(N), "s"(K), "s"(epi.alpha));
  LnStepRows<PLANES, ROWS, D> rows;
  rows.load(ln, tid, 0, M, K);
  __builtin_amdgcn_sched_barrier(0);
  const int8_t* wp = W + ((long)blockIdx.x * (K >> 6) + wave * D) * 1024 + lane * 16;
  v4i fw[D];
#pragma unroll
  for (int u = 0; u < D; ++u) fw[u] = *reinterpret_cast<const v4i*>(wp + u * 1024);
  v4i table = (v4i)0;  // through registers: the layer norm would wait for a DMA
  if constexpr (Epi::kTable)
    table = *reinterpret_cast<const v4i*>(epi.table() + min(n0 + (tid >> 4), N - 1) * 256 +
                                          (((tid ^ (tid >> 4)) & 15) << 4));
  const int quad = tid & 3, row = tid >> 2;
  const int n = n0 + 4 * quad;
  const typename Epi::Col col = epi.column(min(n, N - 4), N);
  __builtin_amdgcn_sched_barrier(0);
  rows.finish(ln, tid, 0, M, K, codes, red_ln, blockIdx.x == 0);
  if constexpr (Epi::kTable) *reinterpret_cast<v4i*>(tab + tid * 16) = table;
  __syncthreads();
  v4i acc = (v4i)0;
#pragma unroll
  for (int u = 0; u < D; ++u) {
    asm volatile("" : "+v"(fw[u]));
    const v4i a = *reinterpret_cast<const v4i*>(codes + (wave * D + u) * 1024 + lane * 16);
    acc = KwI8::mma(fw[u], a, acc);
  }
  v4i* cells = reinterpret_cast<v4i*>(part);
  cells[wave * 68 + kq * 17 + l16] = acc;
  __syncthreads();
  if (blockIdx.x == 0) rows.store(ln, tid, 0, M, K);
  if (row >= M || n >= N) return;
  const int cell = quad * 17 + row;
  const v4i c = (cells[cell] + cells[68 + cell]) + (cells[2 * 68 + cell] + cells[3 * 68 + cell]);
  if constexpr (Epi::kTable) epi.store4(row, n, N, col, c, tab + 4 * quad * 256);
  else epi.store4(row, n, N, col, c);
}

namespace {

template <typename Epi, int PLANES, int ROWS>
int launch_ln_rows(const LnStep& ln, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  const dim3 grid((N + 15) / 16);
  const size_t smem = 16 * (size_t)K + 4 * 68 * 16 + (Epi::kTable ? 16 * 256 : 0);
  switch (K >> 8) {
    case 1: return launch_blk<ln_gemm_kernel<Epi, PLANES, ROWS, 1>>(grid, 256, smem, s, W, M, N, K, ln, epi);
    case 2: return launch_blk<ln_gemm_kernel<Epi, PLANES, ROWS, 2>>(grid, 256, smem, s, W, M, N, K, ln, epi);
    case 3: return launch_blk<ln_gemm_kernel<Epi, PLANES, ROWS, 3>>(grid, 256, smem, s, W, M, N, K, ln, epi);
    default: return launch_blk<ln_gemm_kernel<Epi, PLANES, ROWS, 4>>(grid, 256, smem, s, W, M, N, K, ln, epi);
  }
}
template <typename Epi, int PLANES>
int launch_ln_planes(const LnStep& ln, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  if (!ln_step_supported(M, K) || N % 4 != 0 || ln.planes > 4)
    return lsh_fail(LSH_ERR_UNSUPPORTED, "layer norm + product: shape not covered");
  if (!ln.acc || !ln.res_in || !ln.res_out || ln.res_in == ln.res_out || !ln.scale || !ln.bias || !W ||
      !epi.aligned())
    return lsh_fail(LSH_ERR_INVALID, "layer norm + product: bad operands");
  const uintptr_t all = reinterpret_cast<uintptr_t>(ln.acc) | reinterpret_cast<uintptr_t>(ln.res_in) |
                        reinterpret_cast<uintptr_t>(ln.res_out) | reinterpret_cast<uintptr_t>(ln.scale) |
                        reinterpret_cast<uintptr_t>(ln.bias) | reinterpret_cast<uintptr_t>(ln.res_bias) |
                        reinterpret_cast<uintptr_t>(ln.colsum) | reinterpret_cast<uintptr_t>(W);
  if ((all & 15u) != 0 || ln.plane_stride % 4 != 0)
    return lsh_fail(LSH_ERR_INVALID, "layer norm + product: operands must be 16-byte aligned");
  if (M == 1) return launch_ln_rows<Epi, PLANES, 1>(ln, W, epi, M, N, K, s);
  if (M == 2) return launch_ln_rows<Epi, PLANES, 2>(ln, W, epi, M, N, K, s);
  return launch_ln_rows<Epi, PLANES, 4>(ln, W, epi, M, N, K, s);
}
// FROM_FFN: behind a second feed-forward product, whose planes are sums; otherwise behind an
// out-projection, which leaves codes or (with the attention, out_product.h) sums to requantise
template <typename Epi, bool FROM_FFN>
int launch_ln_gemm(const LnStep& ln, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  if (FROM_FFN != (ln.planes != 0 && ln.requant == 0.f) || (ln.requant != 0.f && ln.planes != 1))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "layer norm + product: operand not covered");
  if constexpr (FROM_FFN)
    return ln.planes == 1 ? launch_ln_planes<Epi, 1>(ln, W, epi, M, N, K, s)
                          : launch_ln_planes<Epi, 4>(ln, W, epi, M, N, K, s);
  else
    return ln.planes ? launch_ln_planes<Epi, kLnRequant>(ln, W, epi, M, N, K, s)
                     : launch_ln_planes<Epi, 0>(ln, W, epi, M, N, K, s);
}

}  // namespace

// Every workgroup repeats the rows' arithmetic, 0.35 us a row: beyond four rows it costs what the
// launch costs that it replaces.
bool ln_step_supported(int rows, int hidden) {
  return rows >= 1 && rows <= 4 && hidden % 256 == 0 && hidden >= 256 && hidden <= 1024;
}

const char* gemm_blk_kernel_name(int M, int N, int K, bool table) {
  const EpilogueCost epi = table ? EpilogueCost::kTable : EpilogueCost::kPlain;
  const LdsTile t = choose_lds_tile(M, N, K, cu_count(), epi);
  return t.tm != 0 && t.us < kw_choose_tile(M, N, K, 1, cu_count(), epi).us ? "gemm_blk_tile_kernel"
                                                                              : "gemm_kw_kernel";
}

int gemm_blk_i8o(const int8_t* A, const int8_t* W, int8_t* C, int M, int N, int K, float alpha,
                 hipStream_t s) {
  return dispatch_blk<KwI8, EpiI8, true>(A, W, EpiI8{C, alpha}, M, N, K, s);
}

int gemm_blk_i32o(const int8_t* A, const int8_t* W, int32_t* C, int M, int N, int K, int ksplit,
                  hipStream_t s) {
  return dispatch_blk<KwI8, EpiI32, true>(A, W, EpiI32{C}, M, N, K, s, ksplit);
}

int gemm_blk_i32_add(const int8_t* A, const int8_t* W, int32_t* C, int M, int N, int K, int ksplit, hipStream_t s) {
  return dispatch_blk<KwI8, EpiI32Add, false>(A, W, EpiI32Add{EpiI32{C}}, M, N, K, s, ksplit);
}

// Ranges of K (int32 planes, summed by the layer norm that reads them) for the few rows of a
// generation step, four at most: as many as make the estimate smallest, 0.1 us of it for a
// plane more to fetch.  16 x 1024 x 4096 with weights from memory: 4.6 us in one range, 3.5 in
// four.
int gemm_blk_preferred_ksplit(int M, int N, int K) {
  int best = 1;
  if (M > kKwColdRows) return best;
  float best_us = kw_choose_tile(M, N, K, 1, cu_count(), EpilogueCost::kPlain).us;
  for (int ks = 2; ks <= 4; ++ks) {
    if (K % (512 * ks) != 0) continue;
    const float us = kw_choose_tile(M, N, K / ks, ks, cu_count(), EpilogueCost::kPlain).us + 0.1f * ks;
    if (us < best_us) {
      best = ks;
      best_us = us;
    }
  }
  return best;
}

int gemm_blk_lut(const int8_t* A, const int8_t* W, int8_t* C, const int8_t* lut, int M, int N, int K,
                 float alpha, hipStream_t s, const LnStep* ln) {
  if (!lut) return lsh_fail(LSH_ERR_INVALID, "blocked gemm (table epilogue): null table");
  if (N % 64 != 0 || N >= (1 << 24))  // (table offsets of 32 bits)
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm (table epilogue): the output needs N % 64 == 0 and N < 2^24");
  if (ln) return launch_ln_gemm<EpiLutBlk, false>(*ln, W, EpiLutBlk{C, lut, alpha}, M, N, K, s);
  return dispatch_blk<KwI8, EpiLutBlk, true>(A, W, EpiLutBlk{C, lut, alpha}, M, N, K, s);
}

int gemm_blk_decself_qkv(const int8_t* A, const int8_t* W, const __half* qkv_bias, int8_t* new_q,
                         int8_t* new_k, int8_t* new_v, int step_token_num, int hidden, int K,
                         int head_num, int max_step, int step_id, float alpha, float dequant_scale,
                         float quant_scale, hipStream_t s, const LnStep* ln) {
  if (!qkv_bias || !new_q || !new_k || !new_v || head_num <= 0 || hidden <= 0 ||
      hidden % head_num != 0 || max_step <= 0)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm (decoder qkv): bad arguments");
  if (step_id < 0 || step_id >= max_step)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm (decoder qkv): step_id outside the cache");
  const int d = hidden / head_num;
  if (d % 4 != 0 || hidden >= (1 << 22) || (long)hidden * max_step >= (1L << 31))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm (decoder qkv): needs dim_per_head % 4 == 0");
  const EpiDecQkvI8 epi{new_q, new_k, new_v, qkv_bias, alpha, dequant_scale, quant_scale, hidden, head_num,
                        d, max_step, step_id, 1.0f / (float)hidden, 1.0f / (float)d};
  if (ln) return launch_ln_gemm<EpiDecQkvI8, true>(*ln, W, epi, step_token_num, 3 * hidden, K, s);
  return dispatch_blk<KwI8, EpiDecQkvI8, false>(A, W, epi, step_token_num, 3 * hidden, K, s);
}

int gemm_blk_prompt_qkv(const int8_t* A, const int8_t* W, const __half* qkv_bias, int8_t* q_codes,
                        int8_t* k_cache, int8_t* v_cache, int rows, int hidden, int batch, int seq_len,
                        int head_num, int max_step, const int* row_map, float alpha, float dequant_scale,
                        float quant_scale, hipStream_t s) {
  if (!qkv_bias || !q_codes || !k_cache || !v_cache || head_num <= 0 || hidden <= 0 ||
      hidden % head_num != 0 || batch <= 0 || seq_len <= 0 || seq_len > max_step ||
      rows > (long)batch * seq_len)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm (prompt qkv): bad arguments");
  const int d = hidden / head_num;
  if (d % 16 != 0 || hidden >= (1 << 20) || (long)batch * seq_len >= (1 << 22))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm (prompt qkv): needs dim_per_head % 16 == 0");
  const EpiPromptQkvI8 epi{q_codes, k_cache, v_cache, qkv_bias, row_map, alpha, dequant_scale, quant_scale,
                           hidden, head_num, d, max_step, seq_len, 1.0f / (float)hidden,
                           1.0f / (float)d, 1.0f / (float)seq_len};
  return dispatch_blk<KwI8, EpiPromptQkvI8, true>(A, W, epi, rows, 3 * hidden, hidden, s);
}

int gemm_blk_encdec_q(const int8_t* A, const int8_t* W, const __half* q_bias, __half* new_q,
                      int step_token_num, int hidden, int K, int beam_size, int head_num, float alpha,
                      float dequant_scale, hipStream_t s, const LnStep* ln) {
  if (!q_bias || !new_q || head_num <= 0 || hidden <= 0 || hidden % head_num != 0 ||
      beam_size <= 0 || step_token_num <= 0 || step_token_num % beam_size != 0)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm (cross-attention q): bad arguments");
  const int d = hidden / head_num;
  if (d % 4 != 0 || step_token_num >= (1 << 22))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm (cross-attention q): needs dim_per_head % 4 == 0");
  const EpiEncdecQF16 epi{new_q, q_bias, alpha, dequant_scale, beam_size, head_num, d,
                          1.0f / (float)beam_size, 1.0f / (float)d};
  if (ln) return launch_ln_gemm<EpiEncdecQF16, false>(*ln, W, epi, step_token_num, hidden, K, s);
  return dispatch_blk<KwI8, EpiEncdecQF16, false>(A, W, epi, step_token_num, hidden, K, s);
}

// [rows, K bytes] row-major -> blocked (rows beyond the matrix: zeros), or back.  A thread moves
// 16 bytes.
template <bool BACK>
__global__ void __launch_bounds__(256)
block_rows_kernel(const int8_t* __restrict__ in, int8_t* __restrict__ out, long chunks, int rows, int K) {
  const long chunk = (long)blockIdx.x * 256 + threadIdx.x;
  if (chunk >= chunks) return;
  const int lane = (int)(chunk & 63);
  const long blk = chunk >> 6;
  const int ks = (int)(blk % (K / 64));
  const long row = blk / (K / 64) * 16 + (lane & 15);
  const int k = ks * 64 + (lane >> 4) * 16;
  if (BACK) {
    if (row < rows)
      *reinterpret_cast<v4i*>(out + row * K + k) = *reinterpret_cast<const v4i*>(in + chunk * 16);
  } else {
    v4i v = (v4i)0;
    if (row < rows) v = *reinterpret_cast<const v4i*>(in + row * K + k);
    *reinterpret_cast<v4i*>(out + chunk * 16) = v;
  }
}

int block_rows(const void* in, void* out, int rows, int row_bytes, bool back, hipStream_t s) {
  if (!in || !out || in == out || rows <= 0 || row_bytes <= 0 || row_bytes % 64 != 0 ||
      ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) != 0)
    return lsh_fail(LSH_ERR_INVALID, "block_rows: needs row bytes % 64 == 0 and aligned pointers");
  const long chunks = (long)((rows + 15) / 16) * row_bytes;
  const unsigned grid = (unsigned)((chunks + 255) / 256);
  if (back)
    block_rows_kernel<true><<<grid, 256, 0, s>>>(static_cast<const int8_t*>(in), static_cast<int8_t*>(out),
                                                 chunks, rows, row_bytes);
  else
    block_rows_kernel<false><<<grid, 256, 0, s>>>(static_cast<const int8_t*>(in), static_cast<int8_t*>(out),
                                                  chunks, rows, row_bytes);
  return lsh_check_launch("block_rows_kernel");
}

}  // namespace lsh
