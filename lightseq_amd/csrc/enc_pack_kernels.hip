// Encoder calls without the padding of their batch: which rows are computed, and the embedding
// that fills them.
//
// Everything in an encoder stack but the attention works on single rows, and the attention of a
// padded query gives zeros, so all padded positions behind the end of their sequences carry the
// same row through the stack: embedding zero, context zero, the same products and norms.  One such
// row is computed, and the last layer norm writes it to all of them.  With lengths uniform
// between a quarter and the whole of seq_len that leaves 0.63 of the rows of every product and
// norm.  (Padding in front of a sequence's last token is kept: its position is one of the rows.)
#include "ls_device.h"
#include "ls_launch.h"

#include <algorithm>

namespace lsh {

namespace {
constexpr int kPackMaxBatch = 1024;
constexpr int kItemHeadShift = 16, kItemBlocksShift = 28;  // as in qkv_attn_kernels.hip
}  // namespace

// One workgroup: a wavefront per sequence finds the last token (COUNT: counts its tokens, what a
// GPT model takes for the length of a text), then starts by a prefix sum, and
// the work items of the fused QKV + attention kernel in the order that kernel wants (see
// qkv_attn_plan_kernel; longest sequence first for the attention over more than 128 keys).  Bound by two or three trips to memory.
template <bool COUNT>
__global__ void __launch_bounds__(1024)
enc_pack_plan_kernel(const int* __restrict__ tokens, int padding_id, int* __restrict__ seq,
                     int* __restrict__ items, int batch, int S, int head_num,
                     unsigned long long* host_rows, unsigned ticket, int* real_len, float* ppl) {
  __shared__ int len[kPackMaxBatch], order[kPackMaxBatch];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int b = wave; b < batch; b += 16) {
    int last = 0;
    const int* row = tokens + (long)b * S;
#pragma unroll 4
    for (int i = lane; i < S; i += 64) {
      const bool token = row[i] != padding_id;
      last = COUNT ? last + token : token ? i + 1 : last;
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const int o = __shfl_xor(last, m, 64);
      last = COUNT ? last + o : max(last, o);
    }
    if (lane == 0) len[b] = last;
    if (COUNT && lane == 0) {
      real_len[b] = last;
      ppl[b] = 0.f;
    }
  }
  __syncthreads();
  if (wave == 0) {
    int base = 0;
    bool padded = false;
    for (int b0 = 0; b0 < batch; b0 += 64) {
      const int b = b0 + lane, n = b < batch ? len[b] : 0;
      padded |= __ballot(b < batch && n < S) != 0;
      int sum = n;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const int t = __shfl_up(sum, m, 64);
        if (lane >= m) sum += t;
      }
      if (b < batch) {
        seq[2 * b] = base + sum - n;
        seq[2 * b + 1] = n;
      }
      base += __shfl(sum, 63, 64);
    }
    if (lane == 0) {
      padded &= !COUNT;
      seq[2 * batch] = padded ? base : -1;
      if (host_rows != nullptr)
        __hip_atomic_store(host_rows, (unsigned long long)ticket << 32 | (unsigned)(base + (padded ? 1 : 0)),
                           __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  if (items == nullptr) return;
  for (int b = tid; b < batch; b += 1024) {
    int rank = 0;
    for (int o = 0; o < batch; ++o) rank += len[o] > len[b] || (len[o] == len[b] && o < b);
    order[rank] = b;
  }
  __syncthreads();
  const int n = batch * head_num;
  for (int w = tid; w < n; w += 1024) {
    int seq_rank, head;
    if ((batch & 7) == 0 && S <= 128) {
      const int xcd = w & 7, j = w >> 3, per_xcd = n >> 3;
      const int q = j < 32 ? j : per_xcd - 1 - (j - 32);
      seq_rank = xcd + 8 * (q / head_num);
      head = q % head_num;
    } else {
      seq_rank = w / head_num;
      head = w % head_num;
    }
    const int b = order[seq_rank];
    items[w] = b | (head << kItemHeadShift) | (min((len[b] + 31) >> 5, 7) << kItemBlocksShift);
  }
}

bool enc_pack_supported(int batch, int seq_len, int head_num) {
  return batch >= 1 && batch <= kPackMaxBatch && seq_len >= 1 && seq_len <= 1024 && head_num >= 1 &&
         head_num < (1 << (kItemBlocksShift - kItemHeadShift));
}

int enc_pack_plan(const int* tokens, int padding_id, const EncPack& pack, int batch, int seq_len,
                  int head_num, unsigned long long* host_rows, unsigned ticket, hipStream_t s) {
  if (!tokens || !pack.seq || !pack.row_map || !enc_pack_supported(batch, seq_len, head_num))
    return lsh_fail(LSH_ERR_INVALID, "enc_pack_plan: bad arguments");
  enc_pack_plan_kernel<false><<<1, 1024, 0, s>>>(tokens, padding_id, pack.seq, pack.items, batch,
                                                 seq_len, head_num, host_rows, ticket, nullptr, nullptr);
  return lsh_check_launch("enc_pack_plan_kernel");
}

int text_pack_plan(const int* tokens, int padding_id, int* seq, int* real_len, float* ppl, int batch,
                   int seq_len, unsigned long long* host_rows, unsigned ticket, hipStream_t s) {
  if (!tokens || !seq || !real_len || !ppl || !enc_pack_supported(batch, seq_len, 1))
    return lsh_fail(LSH_ERR_INVALID, "text_pack_plan: bad arguments");
  enc_pack_plan_kernel<true><<<1, 1024, 0, s>>>(tokens, padding_id, seq, nullptr, batch, seq_len, 1,
                                                host_rows, ticket, real_len, ppl);
  return lsh_check_launch("enc_pack_plan_kernel");
}

// grid (positions, sequences), a thread per 8 elements; the arithmetic of enc_emb_kernel
__global__ void __launch_bounds__(1024)
enc_emb_packed_kernel(const int8_t* __restrict__ token_emb, const __half* __restrict__ pos_emb,
                      const int* __restrict__ tokens, __half* __restrict__ output,
                      int* __restrict__ pad_mask, const int* __restrict__ seq,
                      int* __restrict__ row_map, int pad_id, int batch, int S, int hidden, float scale,
                      int vocab, int32_t* clear) {
  const int dim = threadIdx.x * 8, pos = blockIdx.x, b = blockIdx.y;
  const long at = (long)b * S + pos;
  if (clear != nullptr && dim < hidden) {
    int4* p = reinterpret_cast<int4*>(clear + at * hidden + dim);
    p[0] = p[1] = make_int4(0, 0, 0, 0);
  }
  int token = tokens[at];
  const int start = seq[2 * b], len = seq[2 * b + 1], pad_row = seq[2 * batch];
  const bool pad = token == pad_id;
  const int row = pos < len ? start + pos : pad_row;
  if (threadIdx.x == 0) {
    pad_mask[at] = pad ? 1 : 0;
    row_map[at] = row;
  }
  // of the positions behind the ends, the last one of the first such sequence writes their row
  bool store = pos < len;
  if (!store && pos == S - 1) {
    store = true;
    for (int o = 0; o < b; ++o) store &= seq[2 * o + 1] == S;
  }
  if (!store || dim >= hidden) return;
  half8_t o;
  if (pad) {
#pragma unroll
    for (int k = 0; k < 8; ++k) o.v[k] = __float2half_rn(0.f);
  } else {
    if (vocab > 0) token = min(max(token, 0), vocab - 1);
    const uint2 w = *reinterpret_cast<const uint2*>(token_emb + (long)token * hidden + dim);
    const half8_t p = *reinterpret_cast<const half8_t*>(pos_emb + (long)pos * hidden + dim);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      o.v[k] = __float2half_rn((float)unpack_i8(k < 4 ? w.x : w.y, k & 3) * scale + __half2float(p.v[k]));
  }
  *reinterpret_cast<half8_t*>(output + (long)row * hidden + dim) = o;
}

int enc_emb_packed(const int8_t* token_emb, const __half* pos_emb, const int* tokens, __half* output,
                   int* pad_mask, int padding_id, const EncPack& pack, int batch, int seq_len,
                   int hidden, hipStream_t s, float dequant_scale, bool scaled, int vocab_size,
                   int32_t* clear) {
  if (!token_emb || !pos_emb || !tokens || !output || !pad_mask || !pack.seq || !pack.row_map ||
      batch <= 0 || seq_len <= 0 || hidden <= 0 || hidden % 8 != 0 || hidden > 8192)
    return lsh_fail(LSH_ERR_INVALID, "enc_emb_packed: bad arguments");
  float scale = dequant_scale;
  if (scaled) scale *= sqrtf((float)hidden);
  const int threads = (hidden / 8 + 63) / 64 * 64;
  enc_emb_packed_kernel<<<dim3(seq_len, batch), threads, 0, s>>>(token_emb, pos_emb, tokens, output,
                                                                 pad_mask, pack.seq, pack.row_map,
                                                                 padding_id, batch, seq_len, hidden,
                                                                 scale, vocab_size, clear);
  return lsh_check_launch("enc_emb_packed_kernel");
}

}  // namespace lsh
