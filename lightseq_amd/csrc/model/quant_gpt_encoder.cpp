#include "quant_gpt_encoder.h"

#include "../ls_device.h"

#include <algorithm>

namespace lightseq {
namespace hip {

using namespace lsh;

QuantGptEncoder::QuantGptEncoder(int max_batch_size, const int* p_d_token_id, float* p_d_ppl,
                                 int* p_d_sample_id, const QuantGptWeight& tw, hipStream_t stream)
    : _p_d_token_id(p_d_token_id),
      _p_d_ppl(p_d_ppl),
      _p_d_sample_id(p_d_sample_id),
      _max_batch_size(max_batch_size),
      _tw(tw),
      _stream(stream),
      _src_emb_clip_max(tw._src_emb_clip_max),
      _output_ln_clip_max(tw._output_ln_clip_max),
      _logits_clip_max(tw._logits_clip_max),
      _enc_clip_max(tw._enc_clip_max),
      _atten_scaler(__half2float(__float2half_rn(sqrtf(1.f / (float)std::max(tw._dim_per_head, 1))))),
      _max_batch_dim((long)max_batch_size * tw._max_step * tw._hidden_size) {}

QuantGptEncoder::~QuantGptEncoder() {
  if (_h_unfinished) (void)hipHostFree(_h_unfinished);
}

std::string QuantGptEncoder::check() {
  if (_tw._inner_size & 1) return "violate inner_size % 2 = 0";
  if (_tw._dim_per_head & 1) return "violate dim_per_head % 2 = 0";
  if ((int)_tw.layers.size() != _tw._n_enc_layer)
    return "violate p_d_enc_wei.size() = weight_per_enc_layer * n_enc_layer";
  if ((int)_enc_clip_max.size() != 12 * _tw._n_enc_layer) return "wrong clip_max table size";
  const std::string& m = _tw._sampling_method;
  if (m != "topk" && m != "topp" && m != "ppl")
    return std::string("unsupported sampling_method: ") + m;
  if (m == "topk" && _tw._topk != 1 && _tw._topk != 2 && _tw._topk != 4 && _tw._topk != 8 &&
      _tw._topk != 16 && _tw._topk != 32)
    return "topk argument should be in [1,2,4,8,16,32], the model file has topk = " +
           std::to_string(_tw._topk);
  if (m == "topp" && (!(_tw._topp > 0.f) || _tw._topp > 1.f))
    return "topp must lie in (0, 1], the model file has topp = " + std::to_string(_tw._topp);
  if (_tw._src_vocab_size > (1 << 20)) return "violate vocab_size <= 2^20 (sampling kernels)";
  if (_tw._hidden_size % 16 != 0 || _tw._inner_size % 16 != 0)
    return "violate hidden_size % 16 = 0 and inner_size % 16 = 0 (int8 MFMA GEMM)";
  if (_tw._dim_per_head != 32 && _tw._dim_per_head != 64 && _tw._dim_per_head != 128)
    return "violate dim_per_head in {32, 64, 128} (fused attention kernel)";
  if (_tw._max_step > 4096) return "violate max_step <= 4096";
  if (_tw._eos_id < 0 || _tw._eos_id >= _tw._src_vocab_size)
    return "eos_id outside the vocabulary";
  return "";
}

void QuantGptEncoder::init_buffer() {
  const int H = _tw._hidden_size, I = _tw._inner_size, L = _tw._n_enc_layer;
  const int V = _tw._src_vocab_size;
  const size_t tokens = (size_t)_max_batch_size * _tw._max_step;
  _real_seq_len.alloc(_max_batch_size);
  _pack_seq.alloc(2 * (size_t)_max_batch_size + 1);
  _pack_map.alloc(tokens);
  _ids.alloc(tokens);
  _last_ids.alloc(_max_batch_size);
  _unfinished.alloc(1);
  _sample_state.alloc(2 * (size_t)_max_batch_size);  // 16 bytes per sequence
  set_seed(0);
  CHECK_GPU_ERROR(hipHostMalloc(reinterpret_cast<void**>(&_h_unfinished), sizeof(int)));
  *_h_unfinished = 0;
  _ops.blocked = LayerProducts::can_block(H, I, _tw._dim_per_head);
  _logits_stride = _ops.blocked ? (V + 63) & ~63 : V;
  _query[0].alloc((size_t)_max_batch_dim);
  _query[1].alloc((size_t)_max_batch_size * H);
  _qkv_buf.alloc((size_t)(3 * _max_batch_dim));
  const size_t wide = _ops.rows(tokens) * (size_t)std::max(I, 3 * H);
  _buf_a.alloc(wide);
  _buf_b.alloc(wide);
  _buf_q.alloc(wide);
  for (auto& h : _hid_last) h.alloc(_ops.rows(_max_batch_size) * H);
  // perplexity needs the logits of every position, sampling only of the last one
  _logits.alloc((_tw._sampling_method == "ppl" ? tokens : (size_t)_max_batch_size) * _logits_stride);
  // room for the accumulator planes of the split-K second FFN product
  _int32_ffn_out_buf.alloc(std::max(tokens * H * 4, (size_t)64 * H * 8));
  _out_sums.alloc((size_t)_max_batch_size * H);
  _self_k_cache.alloc((size_t)L * _max_batch_dim);
  _self_v_cache.alloc((size_t)L * _max_batch_dim);
  CHECK_GPU_ERROR(hipMemsetAsync(_self_k_cache.get(), 0, _self_k_cache.size(), _stream));
  CHECK_GPU_ERROR(hipMemsetAsync(_self_v_cache.get(), 0, _self_v_cache.size(), _stream));

  // stored [H, vocab]; a [vocab, H] copy serves the row lookup and, where products run on
  // row-major operands, the logits; a blocked one padded to whole tiles serves them otherwise
  _int8_emb = upload_kernel(_tw.token_embedding, H, V, true, _stream);
  if (_ops.blocked) _emb_blk = block_weight_padded(_int8_emb, V, H, _stream);
  _pos_emb = upload_half(_tw.position_embedding, _stream);
  _out_ln_scale = upload_half(_tw.norm_scale, _stream);
  _out_ln_bias = upload_half(_tw.norm_bias, _stream);
  _layers.clear();
  _layers.resize(L);
  for (int l = 0; l < L; ++l) {
    const QuantBertLayerWeight& w = _tw.layers[l];
    Layer& d = _layers[l];
    d.ln1_scale = upload_half(w.multihead_norm_scale, _stream);
    d.ln1_bias = upload_half(w.multihead_norm_bias, _stream);
    d.b_qkv = upload_half(w.multihead_project_bias_qkv, _stream);
    d.b_out = upload_half(w.multihead_project_bias_output, _stream);
    d.ln2_scale = upload_half(w.ffn_norm_scale, _stream);
    d.ln2_bias = upload_half(w.ffn_norm_bias, _stream);
    d.b_ffn1 = upload_half(w.ffn_first_bias, _stream);
    d.b_ffn2 = upload_half(w.ffn_second_bias, _stream);
    d.w_qkv = _ops.weight(w.multihead_project_kernel_qkv, H, 3 * H, _stream);
    d.w_out = _ops.weight(w.multihead_project_kernel_output, H, H, _stream);
    d.w_ffn1 = _ops.weight(w.ffn_first_kernel, H, I, _stream);
    {
      const float* c = &_enc_clip_max[l * 12];
      d.ffn1_act_lut.alloc((size_t)I * 256);
      LSH_CALL(build_act_lut(d.ffn1_act_lut.get(), d.b_ffn1.get(), I, c[10] / _quant_range,
                             _quant_range / c[7], c[7], kActGelu, _stream));
    }
    d.w_ffn2 = _ops.weight(w.ffn_second_kernel, I, H, _stream);
  }
  CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
}

// FFN block and the LayerNorm that follows it (:646-776).  `in` holds the int8
// LayerNorm output and receives the next one; `tmp` is scratch of the same size.  ln_in: the first
// product makes its rows by this layer norm; ln_out: receives the one that follows, which then
// the next layer's first product makes.
// Step taps (debug): name -> what is copied, of the tapped layer at the tapped cached step.
//   ln1_q, self_q, ctx_q, out_q, ln2_q, next_ln_q: int8 [batch, hidden];  act_q: int8 [batch, inner]
//   ffn2_acc: int32 [batch, hidden];  k_cache, v_cache: the layer's int8 caches [batch, heads,
//   max_step, d] after the append;  res_in, res_attn, res_out: the fp16 residual stream [batch,
//   hidden] at the start of the layer, after the first and after the last layer norm
#define TAP(name, ptr, bytes) step_taps.copy(_layer_id, _tap_step, name, ptr, bytes, _stream)
#define TAP_CODES(name, ptr, rows, cols) \
  step_taps.copy_codes(_layer_id, _tap_step, name, ptr, rows, cols, _ops.blocked, _stream)

void QuantGptEncoder::ffn_add_norm(int rows, int8_t* in, int8_t* tmp, bool blocked_out,
                                   const LnStep* ln_in, LnStep* ln_out, int32_t* ffn_sums) {
  const int H = _tw._hidden_size, I = _tw._inner_size;
  const Layer& w = _layers[_layer_id];
  const float* c = &_enc_clip_max[_layer_id * 12];
  const float Q = _quant_range;
  _ops.lut(in, w.w_ffn1.get(), tmp, w.ffn1_act_lut.get(), rows, I, H, c[2] * c[6] / (c[10] * Q),
           _stream, ln_in);
  TAP_CODES("act_q", tmp, rows, I);
  // a tapped accumulator is one plane (the planes of a split product sum to it exactly)
  const bool tap_acc = step_taps.wants(_layer_id, _tap_step, "ffn2_acc");
  const int32_t* acc;
  const int nparts = _ops.i32_sums(tmp, w.w_ffn2.get(), _int32_ffn_out_buf.get(), ffn_sums, &acc, rows, H, I,
                                   tap_acc ? 1 : rows <= 64 ? 8 : 4, _stream);
  TAP("ffn2_acc", acc, (size_t)rows * H * sizeof(int32_t));
  const float dequant_scale = c[3] * c[7] / (Q * Q);
  const __half *scale_ptr, *bias_ptr, *res_bias_ptr;
  float clip_max;
  if (_layer_id == _tw._n_enc_layer - 1) {
    scale_ptr = _out_ln_scale.get();
    bias_ptr = _out_ln_bias.get();
    res_bias_ptr = nullptr;
    clip_max = _output_ln_clip_max;
  } else {
    const Layer& nx = _layers[_layer_id + 1];
    scale_ptr = nx.ln1_scale.get();
    bias_ptr = nx.ln1_bias.get();
    res_bias_ptr = nx.b_out.get();
    clip_max = _enc_clip_max[(_layer_id + 1) * 12 + 4];
  }
  if (ln_out && _layer_id != _tw._n_enc_layer - 1) {
    *ln_out = LnStep{acc, nparts, (long)rows * H, _query[_res].get(),
                     _query[_res ^ 1].get(), scale_ptr, bias_ptr, res_bias_ptr, nullptr, dequant_scale,
                     Q / clip_max, 0};
    _res ^= 1;
    return;
  }
  LSH_CALL((residual_bias_ln_i8O<__half, int32_t>(
      acc, scale_ptr, bias_ptr, res_bias_ptr, in, _query[_res].get(), rows, H,
      dequant_scale, Q / clip_max, _stream, false, nullptr, nparts, (long)rows * H, blocked_out)));
  TAP_CODES("next_ln_q", in, rows, H);
  TAP("res_out", _query[_res].get(), (size_t)rows * H * sizeof(__half));
}

// A perplexity has no use for the rows of padded positions: where the whole pass can do without
// them, it computes those of text_pack_plan (0.62 of them with lengths uniform between a quarter
// and the whole of the longest).  A generation's steps read the caches of all positions.
bool QuantGptEncoder::packed_route() const {
  return _ops.blocked && gpt_prefill_i8_enabled() && _tw._hidden_size % 128 == 0 &&
         gpt_prefill_i8_supported(_batch_seq_len, _tw._head_num, _tw._dim_per_head) &&
         enc_pack_supported(_batch_size, _batch_seq_len, 1);  // (at most 2^20 positions)
}

// the rows of the plan: counted here, or as the plan counted them (the device embeds and
// normalises the first layer's rows meanwhile)
int QuantGptEncoder::count_rows(const int* host_token_ids) const {
  if (!host_token_ids) return _rows_notice.wait(_stream);
  int rows = 0;
  for (int i = 0; i < _batch_size * _batch_seq_len; ++i) rows += host_token_ids[i] != _tw._padding_id;
  return rows;
}

// all prompt positions at once (:253-291 / :299-341); leaves the int8 LayerNorm output of
// the last layer in _buf_a, row-major where the caller picks positions from it.  packed: the rows
// are those of the plan, and _batch_token_num is their number afterwards.
void QuantGptEncoder::prompt_pass(const int* ids, bool row_major_out, bool packed,
                                  const int* host_token_ids) {
  const int H = _tw._hidden_size;
  int M = _batch_token_num;
  const int* seq = packed ? _pack_seq.get() : nullptr;
  const float Q = _quant_range;
  _res = 0;
  _tap_step = -2;
  if (packed) {
    const StepNotice n = host_token_ids ? StepNotice{} : _rows_notice.next(nullptr);
    LSH_CALL(text_pack_plan(ids, _tw._padding_id, _pack_seq.get(), _real_seq_len.get(), _p_d_ppl,
                            _batch_size, _batch_seq_len, n.slot, n.tag, _stream));
  } else {
    CHECK_GPU_ERROR(hipMemsetAsync(_real_seq_len.get(), 0, sizeof(int) * _batch_size, _stream));
  }
  LSH_CALL(gpt_embedding_i8I<__half>(_batch_size, _batch_seq_len, H, _stream, _int8_emb.get(),
                                     _pos_emb.get(), ids, _query[_res].get(), _real_seq_len.get(),
                                     _tw._padding_id, 0, _src_emb_clip_max / Q,
                                     _tw._src_vocab_size, _tw._max_step, nullptr, seq, packed ? _pack_map.get() : nullptr));
  // until the number of rows is known, launches cover the most there can be
  if (packed && host_token_ids) M = _batch_token_num = count_rows(host_token_ids);
  if (M == 0) return;  // nothing but padding
  int8_t *a = _buf_a.get(), *b = _buf_b.get();
  __half* qc = _qkv_buf.get();
  __half* kc = qc + _max_batch_dim;
  __half* vd = kc + _max_batch_dim;
  const bool on_codes =
      gpt_prefill_i8_enabled() && H % 128 == 0 &&
      gpt_prefill_i8_supported(_batch_seq_len, _tw._head_num, _tw._dim_per_head);
  for (_layer_id = 0; _layer_id < _tw._n_enc_layer; _layer_id++) {
    const Layer& w = _layers[_layer_id];
    const float* c = &_enc_clip_max[_layer_id * 12];
    if (_layer_id == 0)
      LSH_CALL(norm_layer_resual_i8O<__half>(M, H, _stream, _query[_res].get(), a, w.ln1_scale.get(),
                                             w.ln1_bias.get(), w.b_out.get(), Q / c[4], false,
                                             _ops.blocked));
    if (packed && !host_token_ids && _layer_id == 0) {
      M = _batch_token_num = count_rows(nullptr);
      if (M == 0) return;
    }
    const float qkv_alpha = c[0] * c[4] / (c[8] * Q);
    int8_t* k_cache = _self_k_cache.get() + (size_t)_layer_id * _max_batch_dim;
    int8_t* v_cache = _self_v_cache.get() + (size_t)_layer_id * _max_batch_dim;
    if (on_codes) {
      // int8 end to end: q codes and the caches are all the arrange stage writes, and the
      // attention reads them
      int8_t* q8 = reinterpret_cast<int8_t*>(qc);
      if (_ops.blocked && _batch_size * _batch_seq_len < (1 << 22)) {
        LSH_CALL(gemm_blk_prompt_qkv(a, w.w_qkv.get(), w.b_qkv.get(), q8, k_cache, v_cache, M, H,
                                     _batch_size, _batch_seq_len, _tw._head_num, _tw._max_step,
                                     packed ? _pack_map.get() : nullptr, qkv_alpha, c[8] / Q, Q / c[11],
                                     _stream));
      } else {
        _ops.i8o(a, w.w_qkv.get(), b, M, 3 * H, H, qkv_alpha, _stream);
        LSH_CALL(gpt_arrange_qkv_prefill_i8(M, H, _stream, b, w.b_qkv.get(), q8, k_cache, v_cache,
                                            _batch_seq_len, _tw._dim_per_head, _tw._head_num,
                                            _tw._max_step, c[8] / Q, Q / c[11]));
      }
      LSH_CALL(gpt_prefill_attention_i8(q8, k_cache, v_cache, _real_seq_len.get(), a, Q / c[5],
                                        c[11] / Q, Q / c[11], _batch_size, _batch_seq_len,
                                        _tw._head_num, _tw._dim_per_head, _tw._max_step, _stream,
                                        _ops.blocked, seq));
    } else {
      _ops.i8o(a, w.w_qkv.get(), b, M, 3 * H, H, qkv_alpha, _stream);
      LSH_CALL(gpt_arrange_qkv_prefill_f16(M, H, _stream, b, w.b_qkv.get(), qc, kc, vd, k_cache,
                                           v_cache, _batch_seq_len, _tw._dim_per_head,
                                           _tw._head_num, _tw._max_step, c[8] / Q, Q / c[11]));
      LSH_CALL(gpt_prefill_attention_f16(qc, kc, vd, _real_seq_len.get(), nullptr,
                                         _ops.blocked ? b : a, Q / c[5], c[11] / Q, _batch_size,
                                         _batch_seq_len, _tw._head_num, _tw._dim_per_head, _stream));
      if (_ops.blocked) LSH_CALL(block_rows(b, a, M, H, false, _stream));
    }
    _ops.i8o(a, w.w_out.get(), b, M, H, H, c[1] * c[5] / (c[9] * Q), _stream);
    LSH_CALL((residual_bias_ln_i8O<__half, int8_t>(b, w.ln2_scale.get(), w.ln2_bias.get(),
                                                   w.b_ffn2.get(), a, _query[_res].get(), M, H,
                                                   c[9] / Q, Q / c[6], _stream, false, nullptr, 1,
                                                   0, _ops.blocked)));
    ffn_add_norm(M, a, b, _ops.blocked && !(row_major_out && _layer_id == _tw._n_enc_layer - 1),
                 nullptr, nullptr);
  }
}

// One cached step for the tokens in _last_ids at position _batch_seq_len - 1 (:363-377): the
// embedding, then the layers from..to - 1; after the last layer _step.a holds its int8
// LayerNorm output [batch, hidden].
void QuantGptEncoder::step_begin(StepNotice notice) {
  LnFewRowsScope few_rows;  // every step of every batch size: layer norms by the row kernel
  const int H = _tw._hidden_size, B = _batch_size;
  const float Q = _quant_range;
  _step.a = _buf_a.get();
  _step.b = _buf_b.get();
  _tap_step = _steps_run;
  // the opt-in launch of the QKV product and the attention reads row-major operands
  _step.qkv_attn = !_out_run && !step_taps.any() && decself_qkv_attention_enabled() && _tw._dim_per_head == 64 &&
                   decself_qkv_attention_supported(B, H, _tw._head_num, _tw._max_step);
  _step.ln1_blocked = _ops.blocked && !_step.qkv_attn;
  // few rows: the layer norms between two layers and between the two halves of a layer are made
  // by the products that read them
  _step.ln_in_product = !step_taps.any() && !_step.qkv_attn && _ops.ln_in_product(B, H);
  _step.out_in_attention =
      _out_run && decself_attention_out_supported(B, _tw._head_num, _tw._dim_per_head, _batch_seq_len);
  _out_sums.begin_step(_batch_seq_len * _tw._n_enc_layer);
  _res = 0;
  if (emb_ln_fused()) {
    const Layer& w0 = _layers[0];
    LSH_CALL(gpt_emb_step_norm_layer_i8O<__half>(
        _int8_emb.get(), _pos_emb.get(), _last_ids.get(), _query[_res].get(), _step.a,
        w0.ln1_scale.get(), w0.ln1_bias.get(), w0.b_out.get(), _real_seq_len.get(),
        _unfinished.get(), B, H, _tw._src_vocab_size, _tw._padding_id, _batch_seq_len - 1,
        _tw._max_step, _src_emb_clip_max / Q, Q / _enc_clip_max[4], false, _stream,
        _step.ln1_blocked, notice));
  } else {
    LSH_CALL(gpt_embedding_i8I<__half>(B, 1, H, _stream, _int8_emb.get(), _pos_emb.get(),
                                       _last_ids.get(), _query[_res].get(), _real_seq_len.get(),
                                       _tw._padding_id, _batch_seq_len - 1, _src_emb_clip_max / Q,
                                       _tw._src_vocab_size, _tw._max_step, _unfinished.get()));
  }
}

// the step's embedding and the first layer norm are one launch where the row kernel covers the
// width (the same bytes); with taps set the two launches run
bool QuantGptEncoder::emb_ln_fused() const {
  return !step_taps.any() && _tw._hidden_size % 4 == 0 && _tw._hidden_size <= 1024 &&
         _tw._n_enc_layer > 0;
}

// Decided once a run: a step that left the sums' turn out would leave the next one's buffer uncleared.
// (A run whose caches outgrow the launch goes on without it: it never comes back.)
bool QuantGptEncoder::out_run() const {
  if (!_ops.blocked || step_taps.any() || decself_qkv_attention_enabled() ||
      !decself_attention_out_supported(_batch_size, _tw._head_num, _tw._dim_per_head, _batch_seq_len + 1))
    return false;
  for (int l = 0; l < _tw._n_enc_layer; ++l) {
    const float* c = &_enc_clip_max[l * 12];
    if (c[1] * c[5] / (c[9] * _quant_range) == 0.f) return false;  // no code but zero: LnStep's "none"
  }
  return true;
}

void QuantGptEncoder::step_layers(int from, int to) {
  LnFewRowsScope few_rows;
  const int H = _tw._hidden_size, B = _batch_size;
  const float Q = _quant_range;
  int8_t *&a = _step.a, *&b = _step.b;
  const bool qkv_attn = _step.qkv_attn, ln1_blocked = _step.ln1_blocked,
             ln_in_product = _step.ln_in_product, out = _step.out_in_attention;
  LnStep ln{}, &ln_next = _step.ln_next;
  const size_t bh = (size_t)B * H;
  for (_layer_id = from; _layer_id < to; _layer_id++) {
    Layer& w = _layers[_layer_id];
    const float* c = &_enc_clip_max[_layer_id * 12];
    int8_t* k_cache = _self_k_cache.get() + (size_t)_layer_id * _max_batch_dim;
    int8_t* v_cache = _self_v_cache.get() + (size_t)_layer_id * _max_batch_dim;
    if (_layer_id == 0 && !emb_ln_fused())
      LSH_CALL(norm_layer_resual_i8O<__half>(B, H, _stream, _query[_res].get(), a, w.ln1_scale.get(),
                                             w.ln1_bias.get(), w.b_out.get(), Q / c[4], false, ln1_blocked));
    TAP_CODES("ln1_q", a, B, H);
    TAP("res_in", _query[_res].get(), bh * sizeof(__half));
    // With taps set the two launches run, so that q and the caches are copied before the
    // attention as the tap names promise.
    if (qkv_attn) {
      if (_ops.blocked && !w.w_qkv_rows.get()) w.w_qkv_rows = unblock_weight(w.w_qkv, 3 * H, H, _stream);
      LSH_CALL(decself_qkv_attention_i8(
          a, (_ops.blocked ? w.w_qkv_rows : w.w_qkv).get(), w.b_qkv.get(), _buf_q.get(), k_cache,
          v_cache, b, B, H, _tw._head_num, _tw._max_step, _batch_seq_len - 1,
          c[0] * c[4] / (c[8] * Q), c[8] / Q, Q / c[11], _atten_scaler, c[11] / Q, Q / c[5], _stream,
          _ops.blocked));
    } else {
      // QKV product; its epilogue is ker_arrange_decself_qkv_i8I_i8O: q -> _buf_q, k / v appended
      // to the caches at the token's position
      _ops.decself_qkv(a, w.w_qkv.get(), w.b_qkv.get(), _buf_q.get(), k_cache, v_cache, B, H,
                       _tw._head_num, _tw._max_step, _batch_seq_len - 1, c[0] * c[4] / (c[8] * Q),
                       c[8] / Q, Q / c[11], _stream,
                       ln_in_product && _layer_id > 0 ? &ln_next : nullptr);
      TAP("self_q", _buf_q.get(), bh);
      TAP("k_cache", k_cache, bh * _tw._max_step);
      TAP("v_cache", v_cache, bh * _tw._max_step);
      if (!out)
        LSH_CALL(decself_attention_i8(_buf_q.get(), k_cache, v_cache, b, B * _tw._head_num,
                                      _batch_seq_len, _tw._max_step, _tw._head_num,
                                      _tw._dim_per_head, _atten_scaler, c[11] / Q, Q / c[5], _stream,
                                      _ops.blocked));
    }
    const float out_alpha = c[1] * c[5] / (c[9] * Q);
    const int32_t* sums = _out_sums.sums();
    if (out) {
      // the attention and the out-projection in one launch; the layer norm requantises its sums
      LSH_CALL(decself_attention_out_i8(_buf_q.get(), k_cache, v_cache, w.w_out.get(), _out_sums.sums(),
                                        _out_sums.next_sums(), _out_sums.ffn_sums(), B, _batch_seq_len, _tw._max_step, _tw._head_num,
                                        _atten_scaler, c[11] / Q, Q / c[5], _stream));
      _out_sums.launched();
    } else {
      TAP_CODES("ctx_q", b, B, H);
      _ops.i8o(b, w.w_out.get(), a, B, H, H, out_alpha, _stream);
      TAP("out_q", a, bh);
    }
    if (ln_in_product) {
      ln = LnStep{a, 0, 0, _query[_res].get(), _query[_res ^ 1].get(), w.ln2_scale.get(),
                  w.ln2_bias.get(), w.b_ffn2.get(), nullptr, c[9] / Q, Q / c[6], 0};
      if (out) ln.acc = sums, ln.planes = 1, ln.requant = out_alpha;
      _res ^= 1;
      ffn_add_norm(B, a, b, true, &ln, &ln_next, out ? _out_sums.ffn_sums() : nullptr);
      continue;
    }
    if (out)
      LSH_CALL((residual_bias_ln_i8O<__half, int32_t>(sums, w.ln2_scale.get(), w.ln2_bias.get(),
                                                      w.b_ffn2.get(), b, _query[_res].get(), B, H,
                                                      c[9] / Q, Q / c[6], _stream, false, nullptr, 1,
                                                      0, _ops.blocked, out_alpha)));
    else
      LSH_CALL((residual_bias_ln_i8O<__half, int8_t>(a, w.ln2_scale.get(), w.ln2_bias.get(),
                                                     w.b_ffn2.get(), b, _query[_res].get(), B, H,
                                                     c[9] / Q, Q / c[6], _stream, false, nullptr, 1,
                                                     0, _ops.blocked)));
    TAP_CODES("ln2_q", b, B, H);
    TAP("res_attn", _query[_res].get(), bh * sizeof(__half));
    ffn_add_norm(B, b, a, _layer_id == _tw._n_enc_layer - 1 ? _ops.blocked : ln1_blocked, nullptr,
                 nullptr);
    std::swap(a, b);  // `a` names the buffer holding the layer's int8 LayerNorm output
  }
  if (to == _tw._n_enc_layer) _tap_step = -2;
}

#undef TAP
#undef TAP_CODES

// int8 logits of `rows` hidden rows, _logits_stride codes from one row to the next (:399-404)
void QuantGptEncoder::logits_product(const int8_t* hidden, int rows) {
  _ops.i8o(hidden, (_ops.blocked ? _emb_blk : _int8_emb).get(), _logits.get(), rows, _logits_stride,
           _tw._hidden_size,
           _output_ln_clip_max * _src_emb_clip_max / (_logits_clip_max * _quant_range), _stream);
}

// logits of the last position + greedy choice, enqueued only (:399-487)
void QuantGptEncoder::enqueue_sampling(const int8_t* hidden, bool clear_flag) {
  const int V = _tw._src_vocab_size, B = _batch_size;
  logits_product(hidden, B);
  if (_rec_logits && _steps_run < _rec_max_steps)
    CHECK_GPU_ERROR(hipMemcpy2DAsync(_rec_logits + (size_t)_steps_run * B * V, V, _logits.get(),
                                     _logits_stride, V, B, hipMemcpyDeviceToDevice, _stream));
  // (after a cached step the flag was cleared by the step's embedding launch)
  if (clear_flag) LSH_CALL(fill_i32(_unfinished.get(), 0, 1, _stream));
  const bool topp = _tw._sampling_method == "topp";
  if (!topp && _tw._topk == 1) {
    LSH_CALL(gpt_greedy_step(_logits.get(), _ids.get(), _last_ids.get(), V, _tw._max_step,
                             _batch_seq_len, B, _unfinished.get(), _tw._eos_id, _stream,
                             _logits_stride));
  } else {
    // ker_topk_sample_i8I<k> / ker_topp_sample_i8I (:405-430, :448-473)
    LSH_CALL(gpt_sample_step(_logits.get(), _ids.get(), _last_ids.get(), V, _tw._max_step,
                             _batch_seq_len, B, _unfinished.get(), _tw._eos_id,
                             topp ? 0 : _tw._topk, _tw._topp, _logits_clip_max / _quant_range,
                             _sample_state.get(), _stream, _logits_stride));
  }
}

// Restart the generator states of the random-sampling steps: sequence i draws from (seed, i).
void QuantGptEncoder::set_seed(unsigned long long seed) {
  LSH_CALL(sample_state_setup(_sample_state.get(), _max_batch_size, seed, _stream));
}

// host side of a sampled token: the counters
void QuantGptEncoder::count_token() {
  ++_steps_run;
  _batch_seq_len++;
  _batch_token_num += _batch_size;
}

// the unfinished flag of the step just enqueued (one word back from the device)
int QuantGptEncoder::read_unfinished() {
  CHECK_GPU_ERROR(hipMemcpyAsync(_h_unfinished, _unfinished.get(), sizeof(int),
                                 hipMemcpyDeviceToHost, _stream));
  CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
  return *_h_unfinished;
}

int QuantGptEncoder::run_one_sample(int batch_size, int batch_seq_len) {
  if (batch_size > _max_batch_size)
    throw std::runtime_error("batch size of input greater than max_batch_size");
  if (batch_seq_len > _tw._max_step)
    throw std::runtime_error("seq len of input greater than max_step");
  if (batch_size <= 0 || batch_seq_len <= 0) throw std::runtime_error("empty input");
  if (_tw._sampling_method == "ppl")
    throw std::runtime_error("this model file is configured for perplexity, not sampling");
  _batch_size = batch_size;
  _batch_seq_len = batch_seq_len;
  _batch_token_num = batch_size * batch_seq_len;
  _batch_max_seq_len = std::min(_tw._max_step, batch_seq_len + _tw._extra_decode_length);
  _steps_run = 0;
  const int H = _tw._hidden_size;
  _out_run = out_run();

  _phases.mark(0, _stream);
  // ids [batch, max_step] <- prompt
  CHECK_GPU_ERROR(hipMemcpy2DAsync(_ids.get(), sizeof(int) * _tw._max_step, _p_d_token_id,
                                   sizeof(int) * batch_seq_len, sizeof(int) * batch_seq_len,
                                   batch_size, hipMemcpyDeviceToDevice, _stream));
  prompt_pass(_p_d_token_id, true);
  // hidden states of the last prompt position of every sequence
  CHECK_GPU_ERROR(hipMemcpy2DAsync(_hid_last[0].get(), H,
                                   _buf_a.get() + (size_t)(batch_seq_len - 1) * H,
                                   (size_t)batch_seq_len * H, H, batch_size,
                                   hipMemcpyDeviceToDevice, _stream));
  if (_ops.blocked)
    LSH_CALL(block_rows(_hid_last[0].get(), _hid_last[1].get(), batch_size, H, false, _stream));
  int loop_steps = 0;
  if (_batch_seq_len < _tw._max_step) {
    // (:347-353) after the prompt pass the run ends when nothing is unfinished
    enqueue_sampling(_hid_last[_ops.blocked].get(), true);
    count_token();
    const int L = _tw._n_enc_layer;
    if (_out_run) _out_sums.begin_run((size_t)batch_size * H, _stream);
    if (!_is_benchmark && !_use_graphs && !_rec_logits && emb_ln_fused()) {
      _phases.mark(1, _stream);
      while (_batch_seq_len < _batch_max_seq_len) {
        step_begin(_notice.next(_unfinished.get()));
        const int ahead = layers_ahead(loop_steps + 1, L);
        step_layers(0, ahead);
        if (_notice.wait(_stream) == 0) break;
        ++loop_steps;
        step_layers(ahead, L);
        enqueue_sampling(_step.a, false);
        count_token();
      }
    } else {
      const bool go_on = !(read_unfinished() == 0 || _batch_seq_len >= _batch_max_seq_len);
      _phases.mark(1, _stream);
      while (go_on && _batch_seq_len < _batch_max_seq_len) {
        ++loop_steps;
        // the launches of a step depend on the batch size, the position and the run's route only
        const uint64_t key = ((uint64_t)_batch_size << 32) | ((uint64_t)_out_run << 31) | (uint32_t)_batch_seq_len;
        _graphs.run(key, _stream, _use_graphs && !_rec_logits && !step_taps.any(), [&] {
          step_begin(StepNotice{});
          step_layers(0, L);
          enqueue_sampling(_step.a, false);
        });
        count_token();
        // nothing stops a benchmark run but the length
        if (!_is_benchmark && read_unfinished() == 0) break;
      }
    }
  } else {
    _phases.mark(1, _stream);
  }
  _phases.mark(2, _stream);
  _phases.set_loop_steps(loop_steps);
  CHECK_GPU_ERROR(hipMemcpy2DAsync(_p_d_sample_id, sizeof(int) * _batch_seq_len, _ids.get(),
                                   sizeof(int) * _tw._max_step, sizeof(int) * _batch_seq_len,
                                   batch_size, hipMemcpyDeviceToDevice, _stream));
  CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
  return _batch_seq_len;
}

void QuantGptEncoder::run_one_infer(int batch_size, int batch_seq_len, const int* host_token_ids) {
  if (batch_size > _max_batch_size)
    throw std::runtime_error("batch size of input greater than max_batch_size");
  if (batch_seq_len > _tw._max_step)
    throw std::runtime_error("seq len of input greater than max_step");
  if (batch_size <= 0 || batch_seq_len <= 0) throw std::runtime_error("empty input");
  if (_tw._sampling_method != "ppl")
    throw std::runtime_error("this model file is configured for sampling, not perplexity");
  _batch_size = batch_size;
  _batch_seq_len = batch_seq_len;
  _batch_token_num = batch_size * batch_seq_len;
  const int V = _tw._src_vocab_size;
  const bool packed = packed_route();
  if (!packed) CHECK_GPU_ERROR(hipMemsetAsync(_p_d_ppl, 0, sizeof(float) * batch_size, _stream));
  prompt_pass(_p_d_token_id, false, packed, host_token_ids);
  if (_batch_token_num == 0) return;  // no text has a term; the results are zero
  /* compute_ppl (:781-797) */
  logits_product(_buf_a.get(), _batch_token_num);
  // the FFN2 accumulator buffer (tokens * hidden int32, idle by now) holds the per-position terms
  LSH_CALL(ppl_i8I(batch_size, batch_seq_len, _stream, _logits.get(), _p_d_token_id,
                   _real_seq_len.get(), _p_d_ppl, V, _logits_clip_max / _quant_range,
                   reinterpret_cast<float*>(_int32_ffn_out_buf.get()), _logits_stride,
                   packed ? _pack_seq.get() : nullptr));
}

}  // namespace hip
}  // namespace lightseq
