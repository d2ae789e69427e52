#include "quant_decoder.h"

#include "../ls_device.h"

#include <algorithm>

namespace lightseq {
namespace hip {

using namespace lsh;

static const float kMinLogProbability = -2000.f;  // inference/kernels/transformerKernels.h:12

QuantDecoder::QuantDecoder(int max_batch_size, const int* p_d_padding_mask,
                           const __half* p_d_encoder_output, int* p_d_result,
                           QuantTransformerWeight& tw, hipStream_t stream, bool output_topk)
    : _p_d_padding_mask(p_d_padding_mask),
      _p_d_encoder_output(p_d_encoder_output),
      _p_d_result(p_d_result),
      _output_topk(output_topk),
      _max_batch_size(max_batch_size),
      _tw(tw),
      _stream(stream),
      _trg_emb_clip_max(tw._trg_emb_clip_max),
      _output_ln_clip_max(tw._output_ln_clip_max),
      _logits_clip_max(tw._logits_clip_max),
      _dec_clip_max(tw._dec_clip_max),
      _layer_size_encdec_k((long)max_batch_size * tw._max_step * tw._hidden_size),
      _layer_size_self_k((long)max_batch_size * tw._max_step * tw._hidden_size * tw._beam_size),
      _h_alive_seq_probs((size_t)max_batch_size * std::max(tw._beam_size, 1),
                         kMinLogProbability / 2),
      _h_length_norm((size_t)std::max(tw._max_step, 1), 1.f) {
  // only the first beam of a sentence is alive before the first step (:64-66)
  for (size_t i = 0; i < _h_alive_seq_probs.size(); i += std::max(tw._beam_size, 1))
    _h_alive_seq_probs[i] = 0.f;
  if (tw._length_penalty >= 0)
    for (size_t i = 0; i < _h_length_norm.size(); i++)
      _h_length_norm[i] = length_norm((int)i + 1, tw._length_penalty);
}

QuantDecoder::~QuantDecoder() {
  if (_h_num_finished) (void)hipHostFree(_h_num_finished);
}

std::string QuantDecoder::check() {
  if (_tw._inner_size & 1) return "violate inner_size % 2 = 0";
  if (_tw._dim_per_head & 1) return "violate dim_per_head % 2 = 0";
  if (_tw._multilg_type != 0) return "multilingual models are not supported";
  if ((int)_tw.dec_layers.size() != _tw._n_dec_layer)
    return "violate p_d_dec_wei.size() = weight_per_dec_layer * n_dec_layer";
  if ((int)_dec_clip_max.size() != 19 * _tw._n_dec_layer) return "wrong clip_max table size";
  bool btmp = false;
  for (int i = 1; i < 64; i *= 2)
    if (i == _tw._beam_size) btmp = true;
  if (!btmp) return "wrong beam_size, should be 1, 2, 4, 8, 16 or 32";
  const std::string& m = _tw._sampling_method;
  if (m != "beam_search" && m != "topk" && m != "topp" && m != "topk_greedy")
    return std::string("unsupported sampling_method: ") + m;
  // (inference/model/quant_decoder.cc.cu:392-397)
  if (m == "topk" || m == "topp") _output_topk = false;
  if (m == "topk_greedy") _output_topk = true;
  if (m == "topk" && _tw._topk != 1 && _tw._topk != 2 && _tw._topk != 4 && _tw._topk != 8 &&
      _tw._topk != 16 && _tw._topk != 32)
    return "topk argument should be in [1,2,4,8,16,32]";
  if (m == "topp" && (!(_tw._topp > 0.f) || _tw._topp > 1.f)) return "topp outside (0, 1]";
  if (_tw._diverse_lambda != 0.f) return "diverse beam search is not available in this build";
  if (_tw._max_step > 1024) return "max_step should not greater than 1024";
  if (_tw._hidden_size % 16 != 0 || _tw._inner_size % 16 != 0)
    return "violate hidden_size % 16 = 0 and inner_size % 16 = 0 (int8 MFMA GEMM)";
  if (_tw._end_id < 0 || _tw._end_id >= _tw._trg_vocab_size || _tw._start_id < 0 ||
      _tw._start_id >= _tw._trg_vocab_size)
    return "start_id / end_id outside the target vocabulary";
  return "";
}

void QuantDecoder::init_buffer() {
  const int H = _tw._hidden_size, I = _tw._inner_size, L = _tw._n_dec_layer;
  const int V = _tw._trg_vocab_size, beam = _tw._beam_size;
  const size_t rows = (size_t)_max_batch_size * beam;
  const size_t tokens = (size_t)_max_batch_size * _tw._max_step;

  _encdec_k.alloc((size_t)L * _layer_size_encdec_k);
  _encdec_v.alloc((size_t)L * _layer_size_encdec_k);
  for (auto& q : _cur_step_query) q.alloc(rows * H);
  _query_buf1.alloc(rows * H);
  _ops.blocked = LayerProducts::can_block(H, I, _tw._dim_per_head);
  _encoder_out_buf.alloc(_ops.blocked ? _ops.rows(tokens) * H : tokens * (size_t)L * 2 * H);
  _logits_stride = _ops.blocked ? (V + 63) & ~63 : V;
  const size_t wide = _ops.rows(rows) * (size_t)std::max(I, 3 * H);
  _buf_a.alloc(wide);
  _buf_b.alloc(wide);
  _buf_q.alloc(wide);
  _logits.alloc(rows * (size_t)_logits_stride);
  // up to 8 accumulator planes of the split-K second FFN product
  _int32_ffn_out_buf.alloc(rows * H * 8);
  _out_sums.alloc((size_t)rows * H);
  for (int i = 0; i < 2; ++i) {
    _self_k_cache[i].alloc((size_t)L * _layer_size_self_k);
    _self_v_cache[i].alloc((size_t)L * _layer_size_self_k);
    CHECK_GPU_ERROR(hipMemsetAsync(_self_k_cache[i].get(), 0, _self_k_cache[i].size(), _stream));
    CHECK_GPU_ERROR(hipMemsetAsync(_self_v_cache[i].get(), 0, _self_v_cache[i].size(), _stream));
  }
  std::vector<int> start_id_vec(rows * _tw._max_step, _tw._start_id);
  for (int i = 0; i < 2; ++i) {
    _alive_seq[i].alloc(start_id_vec.size());
    _alive_seq[i].upload(start_id_vec.data(), start_id_vec.size(), _stream);
  }
  _beam_stride = (_tw._max_step + 3) & ~3;
  for (auto& b : _beam_from) b.alloc((size_t)rows * _beam_stride);
  _alive_seq_probs.alloc(rows);
  _alive_seq_score_own.alloc(rows);
  CHECK_GPU_ERROR(hipMemsetAsync(_alive_seq_score_own.get(), 0, rows * sizeof(float), _stream));
  if (!_p_d_alive_seq_score) _p_d_alive_seq_score = _alive_seq_score_own.get();
  _top_score.alloc(rows * beam);
  _top_idx.alloc(rows * beam);
  // the per-row top-k dealt to several workgroups per row, where the vocabulary allows
  if (const size_t words = beam_search_step_workspace_words(_max_batch_size, beam, _tw._trg_vocab_size))
    _topk_part_ws.alloc(words);
  _parent.alloc(rows);
  _num_finished.alloc(1);
  _sample_unfinished.alloc(1);
  _sample_state.alloc(rows * 2);
  set_seed(0);
  CHECK_GPU_ERROR(hipHostMalloc(reinterpret_cast<void**>(&_h_num_finished), sizeof(int)));
  *_h_num_finished = 0;
  CHECK_GPU_ERROR(hipStreamSynchronize(_stream));  // start_id_vec dies below

  // ---- embedding block ----
  // stored [H, vocab]; a [vocab, H] copy serves the row lookup and, where products run on
  // row-major operands, the logits; a blocked one padded to whole tiles serves them otherwise
  _int8_trg_emb = upload_kernel(_tw.trg_token_embedding, H, V, true, _stream);
  if (_ops.blocked) _emb_blk = block_weight_padded(_int8_trg_emb, V, H, _stream);
  _pos_emb = upload_half(_tw.trg_position_embedding, _stream);
  _out_ln_scale = upload_half(_tw.trg_norm_scale, _stream);
  _out_ln_bias = upload_half(_tw.trg_norm_bias, _stream);
  _kv_bias = upload_half(_tw.encode_output_project_bias_kv, _stream);
  _logit_bias = upload_half(_tw.shared_bias, _stream);
  {
    // The K/V projection stays an fp16 GEMM (:497-501).  File layout [H, n_layer*2*H],
    // dequantised in flat chunks of 2*H*H with one clip each
    // (inference/proto/quant_transformer_weight.cc:144-160), then transposed to the
    // K-contiguous [n_layer*2*H, H] form of the GEMM here.
    const size_t kv_dim = (size_t)L * 2 * H, chunk = (size_t)2 * H * H;
    const std::vector<uint8_t>& src = _tw.encode_output_project_kernel_kv;
    std::vector<__half> t(kv_dim * H);
    for (size_t k = 0; k < (size_t)H; ++k)
      for (size_t n = 0; n < kv_dim; ++n) {
        const size_t flat = k * kv_dim + n;
        const float clip = _tw._encode_output_project_kernel_kv_clip_max[flat / chunk];
        // inference/tools/util.cc.cu:346-348
        const float v = ((float)src[flat] - _quant_range) * clip / _quant_range;
        t[n * H + k] = __float2half_rn(v);
      }
    _kv_kernel.alloc(t.size());
    _kv_kernel.upload(t.data(), t.size(), _stream);
    if (_ops.blocked) {  // (kv_dim is a multiple of 16: whole blocks)
      DeviceBuffer<__half> b(t.size());
      LSH_CALL(block_rows(_kv_kernel.get(), b.get(), (int)kv_dim, 2 * H, false, _stream));
      CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
      _kv_kernel = std::move(b);
    }
    CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
  }

  // ---- layers ----
  _layers.clear();
  _layers.resize(L);
  for (int l = 0; l < L; ++l) {
    const QuantDecoderLayerWeight& w = _tw.dec_layers[l];
    Layer& d = _layers[l];
    d.self_ln_scale = upload_half(w.self_norm_scale, _stream);
    d.self_ln_bias = upload_half(w.self_norm_bias, _stream);
    d.b_self_qkv = upload_half(w.self_project_bias_qkv, _stream);
    d.b_self_out = upload_half(w.self_project_bias_output, _stream);
    d.encdec_ln_scale = upload_half(w.encdec_norm_scale, _stream);
    d.encdec_ln_bias = upload_half(w.encdec_norm_bias, _stream);
    d.b_encdec_q = upload_half(w.encdec_project_bias_q, _stream);
    d.b_encdec_out = upload_half(w.encdec_project_bias_output, _stream);
    d.ffn_ln_scale = upload_half(w.ffn_norm_scale, _stream);
    d.ffn_ln_bias = upload_half(w.ffn_norm_bias, _stream);
    d.b_ffn1 = upload_half(w.ffn_first_bias, _stream);
    d.b_ffn2 = upload_half(w.ffn_second_bias, _stream);
    d.w_self_qkv = _ops.weight(w.self_project_kernel_qkv, H, 3 * H, _stream);
    d.w_self_out = _ops.weight(w.self_project_kernel_output, H, H, _stream);
    d.w_encdec_q = _ops.weight(w.encdec_project_kernel_q, H, H, _stream);
    d.w_encdec_out = _ops.weight(w.encdec_project_kernel_output, H, H, _stream);
    d.w_ffn1 = _ops.weight(w.ffn_first_kernel, H, I, _stream);
    {
      const float* c = &_dec_clip_max[l * 19];
      d.ffn1_act_lut.alloc((size_t)I * 256);
      LSH_CALL(build_act_lut(d.ffn1_act_lut.get(), d.b_ffn1.get(), I, c[16] / _quant_range,
                             _quant_range / c[11], c[11],
                             _tw._use_gelu ? kActGelu : kActReluNarrow, _stream));
    }
    d.w_ffn2 = _ops.weight(w.ffn_second_kernel, I, H, _stream);
    if (!_tw._use_gelu) {
      // ReLU offset trick (:332-354): column sums of the fp16-rounded dequantised FFN2
      // kernel times clip/2
      const size_t n = w.ffn_second_kernel.size();
      DeviceBuffer<uint8_t> raw(n);
      raw.upload(w.ffn_second_kernel.data(), n, _stream);
      DeviceBuffer<__half> deq(n);
      LSH_CALL(stored_u8_dequant<__half>(raw.get(), deq.get(), (long)n, _dec_clip_max[l * 19 + 5],
                                         _stream));
      d.ffn2_colsum.alloc(H);
      LSH_CALL(scaled_colsum<__half>(deq.get(), d.ffn2_colsum.get(), I, H,
                                     _dec_clip_max[l * 19 + 11] / 2, _stream));
      CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
    }
  }
}

void QuantDecoder::set_seed(unsigned long long seed) {
  LSH_CALL(sample_state_setup(_sample_state.get(), (int)(_sample_state.size() / 2), seed, _stream));
}

// "topk_greedy" opens with one beam-search step, which gives every beam of a sentence another
// first token (inference/model/quant_decoder.cc.cu:1101-1106)
bool QuantDecoder::step_runs_beam_search() const {
  return !_is_sampling || (_tw._sampling_method == "topk_greedy" && _cur_step == 0);
}

void QuantDecoder::run_one_infer(int batch_size, int batch_seq_len) {
  if (batch_size > _max_batch_size)
    throw std::runtime_error("batch size of input greater than max_batch_size");
  if (batch_seq_len > _tw._max_step)
    throw std::runtime_error("seq len of input greater than max_step");
  if (batch_size <= 0 || batch_seq_len <= 0) throw std::runtime_error("empty input");

  /* ---step1. init--- */
  _batch_size = batch_size;
  _batch_seq_len = batch_seq_len;
  _batch_token_num = batch_size * batch_seq_len;
  _step_token_num = batch_size * _tw._beam_size;
  _batch_max_decode_length =
      std::min(_tw._max_step, batch_seq_len + _tw._extra_decode_length) - 1;
  // (:429-434)
  _is_sampling = _tw._sampling_method == "topk" || _tw._sampling_method == "topp" ||
                 _tw._sampling_method == "topk_greedy";
  if (_is_sampling) {
    _batch_max_decode_length = _tw._max_step;
    // nothing writes the scores of a sampled sequence; the reference hands its buffer to the
    // result writer as allocated, here every call starts it from zeros
    CHECK_GPU_ERROR(hipMemsetAsync(_alive_seq_score_own.get(), 0, sizeof(float) * _step_token_num,
                                   _stream));
  }
  _steps_run = 0;
  // every call starts from the same halves of the double-buffered sequences and caches (column
  // 0 of both sequence buffers holds the start token; everything else is rewritten as the
  // steps go), so that a step's launches are the same from call to call
  _alive_cur = 0;
  _cache_cur = 0;
  const int d = _tw._dim_per_head;
  _by_beam = !_is_sampling && (d == 32 || d == 64 || d == 128) && _step_token_num <= 65535 && !step_taps.any() &&
             !_rec_logits && !_rec_alive && !decself_qkv_attention_enabled();
  _out_run = out_run();
  if (_out_run) _out_sums.begin_run((size_t)_step_token_num * _tw._hidden_size, _stream);

  _phases.mark(0, _stream);
  project_encoder_output();
  CHECK_GPU_ERROR(hipMemcpyAsync(_alive_seq_probs.get(), _h_alive_seq_probs.data(),
                                 sizeof(float) * _step_token_num, hipMemcpyHostToDevice,
                                 _stream));

  /* ---step2. autoregressive decoding--- */
  _phases.mark(1, _stream);
  const int limit = _batch_max_decode_length - 1;
  if (!_is_benchmark && !_use_graphs && !_rec_logits && !_rec_alive && !step_taps.any() &&
      emb_ln_fused()) {
    const int L = _tw._n_dec_layer;
    for (_cur_step = 0; _cur_step < limit; _cur_step++) {
      if (_cur_step == 0) {
        step_begin(StepNotice{});
        step_layers(0, L);
      }
      step_end();
      const bool search = step_runs_beam_search();
      step_done(search);
      if (_cur_step + 1 == limit) {
        if (finished(search, read_finished(search))) break;
        continue;
      }
      ++_cur_step;
      step_begin(_notice.next(search ? _num_finished.get() : _sample_unfinished.get()));
      const int ahead = layers_ahead(_cur_step, L);
      step_layers(0, ahead);
      const bool stop = finished(search, _notice.wait(_stream));
      if (!stop) step_layers(ahead, L);
      --_cur_step;
      if (stop) break;
    }
  } else {
    for (_cur_step = 0; _cur_step < limit; _cur_step++) {
      const bool early_stop = run_step();
      if (early_stop) break;
    }
  }
  _phases.mark(2, _stream);
  _phases.set_loop_steps(_steps_run);

  /* ---step3. output the decoding result--- */
  // The steps keep the scores of finished beams in the decoder's own buffer: a step may be a
  // recorded graph, and the caller may hand over another output buffer between two calls.
  if (_p_d_alive_seq_score != _alive_seq_score_own.get())
    CHECK_GPU_ERROR(hipMemcpyAsync(_p_d_alive_seq_score, _alive_seq_score_own.get(),
                                   sizeof(float) * _step_token_num, hipMemcpyDeviceToDevice,
                                   _stream));
  int* alive = _alive_seq[_alive_cur].get();
  if (_output_topk || _is_sampling) {
    if (_cur_step == _batch_max_decode_length) _cur_step -= 1;
    LSH_CALL(write_topk_result(alive, _p_d_alive_seq_score, _p_d_result, _tw._trg_vocab_size,
                               _tw._max_step, _tw._beam_size, _tw._end_id, _step_token_num,
                               _cur_step + 1, _stream));
    return;
  }
  if (_tw._length_penalty >= 0.f || _cur_step == _batch_max_decode_length) {
    LSH_CALL(write_trg_tokenid_pos_penalty(alive, _p_d_alive_seq_score, _p_d_result,
                                           _tw._max_step, _tw._beam_size, _batch_size,
                                           _cur_step + 1, _stream));
  } else {
    LSH_CALL(write_trg_tokenid_neg_penalty(alive, _p_d_alive_seq_score, _p_d_result,
                                           _tw._max_step, _tw._beam_size, _tw._trg_vocab_size,
                                           _tw._end_id, _batch_size, _cur_step + 1, _stream));
  }
}

void QuantDecoder::project_encoder_output() {
  const int H = _tw._hidden_size, L = _tw._n_dec_layer;
  const int kv_dim = H * 2 * L;
  if (_ops.blocked) {
    // one product whose epilogue adds the bias and leaves keys and values where the layers read
    // them (16 x 64 tokens, 6 layers of 1024: 145 + 17 us as product and rearrangement, 45 now)
    LSH_CALL(block_rows(_p_d_encoder_output, _encoder_out_buf.get(), _batch_token_num, 2 * H, false, _stream));
    LSH_CALL(gemm_blk_kv_f16(_encoder_out_buf.get(), _kv_kernel.get(), _batch_token_num, L, H, H,
                             _kv_bias.get(), _batch_seq_len, _tw._head_num, _encdec_k.get(),
                             _encdec_v.get(), _layer_size_encdec_k, _stream));
    return;
  }
  LSH_CALL(gemm_f16_nt(_p_d_encoder_output, _kv_kernel.get(), _encoder_out_buf.get(),
                       _batch_token_num, kv_dim, H, _stream));
  // _encoder_out_buf: [batch_size, batch_seq_len, layer_num, 2, hidden_size]
  LSH_CALL(arrange_encdec_kv<__half>(_batch_token_num, L, H, _stream, _encoder_out_buf.get(),
                                     _kv_bias.get(), _encdec_k.get(), _encdec_v.get(),
                                     _layer_size_encdec_k, _batch_seq_len, _tw._dim_per_head,
                                     _tw._head_num));
}

bool QuantDecoder::run_step() {
  const bool search = step_runs_beam_search();
  // The launches of a step depend on the shapes of the call, its routes, the step index and which of the
  // two sequence / cache buffers is current: one graph per such key.  A sampling step clears
  // its flag with a memset and runs eagerly.
  const uint64_t key = ((uint64_t)_batch_size << 40) | ((uint64_t)_batch_seq_len << 24) |
                       ((uint64_t)_cur_step << 8) | (uint64_t)(_out_run << 3 | _by_beam << 2 | _alive_cur << 1 | _cache_cur);
  _graphs.run(key, _stream,
              _use_graphs && !_is_sampling && !_rec_logits && !_rec_alive && !step_taps.any(),
              [&] {
                step_begin(StepNotice{});
                step_layers(0, _tw._n_dec_layer);
                step_end();
              });
  step_done(search);
  return !_is_benchmark && finished(search, read_finished(search));
}

// host side of an enqueued step (a step that samples keeps its sequences in their buffer and does
// not reorder the caches; :979-984, 1126-1131)
void QuantDecoder::step_done(bool search) {
  ++_steps_run;
  if (!search) return;
  _alive_cur ^= 1;
  if (_cur_step > 0 && !_by_beam) _cache_cur ^= 1;
}

// the one device-to-host word of a step: all beams finished -> stop early
int QuantDecoder::read_finished(bool search) {
  CHECK_GPU_ERROR(hipMemcpyAsync(_h_num_finished,
                                 search ? _num_finished.get() : _sample_unfinished.get(), sizeof(int),
                                 hipMemcpyDeviceToHost, _stream));
  CHECK_GPU_ERROR(hipStreamSynchronize(_stream));
  return *_h_num_finished;
}
bool QuantDecoder::finished(bool search, int word) const {
  return search ? word == _step_token_num : word != 1;
}

// What a step puts on the stream: embedding (step_begin), the layers from..to - 1 (step_layers),
// the logits, the search and the cache reorder (step_end) -- kernels and device-to-device copies
// only, so that it can be captured.
void QuantDecoder::step_begin(StepNotice notice) {
  LnFewRowsScope few_rows;  // every step of every batch size: layer norms by the row kernel
  // The opt-in launch reads row-major operands.  With taps set the two launches run, so that q
  // and the caches are copied before the attention as the tap names promise; the bytes are the
  // same either way.
  _qkv_attn = !_by_beam && !_out_run && !step_taps.any() && decself_qkv_attention_enabled() && _tw._dim_per_head == 64 &&
              decself_qkv_attention_supported(_step_token_num, _tw._hidden_size, _tw._head_num,
                                              _tw._max_step);
  // few rows: the layer norms inside the stack are made by the products that read them; that in
  // front of the cross attention by its launch, whatever the number of rows
  _ln_in_product = !step_taps.any() && !_qkv_attn && _ops.ln_in_product(_step_token_num, _tw._hidden_size);
  _ln_in_encdec = !step_taps.any() && _ops.blocked && _tw._hidden_size % 256 == 0;
  _out_step = _out_run && decself_attention_out_supported(_step_token_num, _tw._head_num, _tw._dim_per_head,
                                                          _cur_step + 1);
  _out_sums.begin_step(_cur_step * _tw._n_dec_layer * (encdec_out() ? 2 : 1));
  _res = 0;
  embedding(notice);
}

void QuantDecoder::step_layers(int from, int to) {
  LnFewRowsScope few_rows;
  for (_layer_id = from; _layer_id < to; _layer_id++) {
    self_attention();
    encdec_attention();
    ffn_add_norm();
  }
}

void QuantDecoder::step_end() {
  /* --- Project hidden states to vocab logits (:527-532) --- */
  _ops.i8o(_buf_a.get(), (_ops.blocked ? _emb_blk : _int8_trg_emb).get(), _logits.get(),
           _step_token_num, _logits_stride, _tw._hidden_size,
           _output_ln_clip_max * _trg_emb_clip_max / (_logits_clip_max * _quant_range), _stream);
  if (_rec_logits && _cur_step < _rec_max_steps)
    CHECK_GPU_ERROR(hipMemcpy2DAsync(
        _rec_logits + (size_t)_cur_step * _step_token_num * _tw._trg_vocab_size,
        _tw._trg_vocab_size, _logits.get(), _logits_stride, _tw._trg_vocab_size, _step_token_num,
        hipMemcpyDeviceToDevice, _stream));
  if (step_runs_beam_search())
    beam_search();
  else
    sample_tokens();
}

// Step taps (debug): name -> what is copied, of layer step_taps' layer at its step.
//   self_ln_q, self_q, self_ctx_q, self_out_q, encdec_ln_q, encdec_ctx_q, encdec_out_q, ffn_ln_q,
//   next_ln_q: int8 [rows, hidden];  ffn1_act_q: int8 [rows, inner];  ffn2_acc: int32 [rows, hidden]
//   self_k_cache, self_v_cache: the layer's int8 caches [rows, heads, max_step, d] after the append
//   encdec_q: fp16 [batch, heads, beam, d];  encdec_k, encdec_v: fp16 [batch, heads, src_len, d]
//   res_in, res_self, res_encdec, res_out: the fp16 residual stream [rows, hidden] at the start of
//   the layer, after the first, the second and the last layer norm
#define TAP(name, ptr, bytes) step_taps.copy(_layer_id, _cur_step, name, ptr, bytes, _stream)
#define TAP_CODES(name, ptr, cols) \
  step_taps.copy_codes(_layer_id, _cur_step, name, ptr, _step_token_num, cols, _ops.blocked, _stream)

// hidden sizes the fused embedding + first layer norm covers
bool QuantDecoder::emb_ln_fused() const {
  return _tw._hidden_size % 4 == 0 && _tw._hidden_size <= 1024;
}

void QuantDecoder::embedding(StepNotice notice) {
  if (_layers.empty()) return;
  const int H = _tw._hidden_size, M = _step_token_num;
  const Layer& w = _layers[0];
  const float quant_scale = _quant_range / _dec_clip_max[6];
  const bool blocked = _ops.blocked && !_qkv_attn;
  if (emb_ln_fused()) {
    // the step's embedding and the first layer norm in one launch (the bytes of the pair)
    LSH_CALL(dec_emb_norm_layer_i8O<__half>(
        _int8_trg_emb.get(), _pos_emb.get(), _alive_seq[_alive_cur].get(),
        _cur_step_query[_res].get(), _buf_a.get(), w.self_ln_scale.get(), w.self_ln_bias.get(),
        w.b_self_out.get(), M, H, _tw._trg_vocab_size, _cur_step, _tw._max_step,
        _trg_emb_clip_max / _quant_range, true, quant_scale, _tw._is_post_ln, _stream, blocked, notice));
    return;
  }
  LSH_CALL(dec_emb_i8I<__half>(_int8_trg_emb.get(), _pos_emb.get(), _alive_seq[_alive_cur].get(),
                               _cur_step_query[_res].get(), _batch_size, _tw._beam_size, H,
                               _tw._trg_vocab_size, _cur_step, _tw._max_step, _stream,
                               _trg_emb_clip_max / _quant_range, true, true));
  LSH_CALL(norm_layer_resual_i8O<__half>(M, H, _stream, _cur_step_query[_res].get(), _buf_a.get(),
                                         w.self_ln_scale.get(), w.self_ln_bias.get(),
                                         w.b_self_out.get(), quant_scale, _tw._is_post_ln, blocked));
}

void QuantDecoder::self_attention() {
  const int H = _tw._hidden_size, M = _step_token_num;
  Layer& w = _layers[_layer_id];
  const float* c = &_dec_clip_max[_layer_id * 19];
  const float Q = _quant_range;
  int8_t* k_cache = _self_k_cache[_cache_cur].get() + (size_t)_layer_id * _layer_size_self_k;
  int8_t* v_cache = _self_v_cache[_cache_cur].get() + (size_t)_layer_id * _layer_size_self_k;

  const size_t mh = (size_t)M * H;
  TAP_CODES("self_ln_q", _buf_a.get(), H);
  TAP("res_in", _cur_step_query[_res].get(), mh * sizeof(__half));
  const float attn_scale =
      __half2float(__float2half_rn(sqrtf(1.f / (float)_tw._dim_per_head)));
  if (_qkv_attn) {
    if (_ops.blocked && !w.w_self_qkv_rows.get())
      w.w_self_qkv_rows = unblock_weight(w.w_self_qkv, 3 * H, H, _stream);
    LSH_CALL(decself_qkv_attention_i8(
        _buf_a.get(), (_ops.blocked ? w.w_self_qkv_rows : w.w_self_qkv).get(), w.b_self_qkv.get(),
        _buf_q.get(), k_cache, v_cache, _buf_b.get(), M, H, _tw._head_num, _tw._max_step, _cur_step,
        c[0] * c[6] / (c[12] * Q), c[12] / Q, Q / c[18], attn_scale, c[18] / Q, Q / c[7], _stream,
        _ops.blocked));
  } else {
    // QKV product; its epilogue is ker_arrange_decself_qkv_i8I_i8O: q -> _buf_q, k / v -> slot
    // _cur_step of the caches (all three with the cache clip)
    if (_tw._dim_per_head % 16 == 0) {
      _ops.decself_qkv(_buf_a.get(), w.w_self_qkv.get(), w.b_self_qkv.get(), _buf_q.get(), k_cache,
                       v_cache, M, H, _tw._head_num, _tw._max_step, _cur_step,
                       c[0] * c[6] / (c[12] * Q), c[12] / Q, Q / c[18], _stream,
                       _ln_in_product && _layer_id > 0 ? &_ln : nullptr);
    } else {
      LSH_CALL(gemm_i8_i8o(_buf_a.get(), w.w_self_qkv.get(), _buf_b.get(), M, 3 * H, H,
                           c[0] * c[6] / (c[12] * Q), _stream));
      LSH_CALL(arrange_decself_qkv_i8I_i8O<__half>(
          M, H, _stream, _buf_b.get(), w.b_self_qkv.get(), _buf_q.get(), k_cache, v_cache,
          _tw._head_num, _tw._dim_per_head, _tw._max_step, _cur_step, c[12] / Q, Q / c[18]));
    }
    TAP("self_q", _buf_q.get(), mh);
    TAP("self_k_cache", k_cache, mh * _tw._max_step);
    TAP("self_v_cache", v_cache, mh * _tw._max_step);
    // int8 q.K -> softmax -> new value, one kernel
    const CacheBeams beams{_beam_from[_alive_cur].get(), _beam_stride};
    if (_out_step)  // ... with the out-projection behind it; the layer norm requantises its sums
      LSH_CALL(decself_attention_out_i8(_buf_q.get(), k_cache, v_cache, w.w_self_out.get(), _out_sums.sums(),
                                        _out_sums.next_sums(), _out_sums.ffn_sums(), M, _cur_step + 1, _tw._max_step, _tw._head_num,
                                        attn_scale, c[18] / Q, Q / c[7], _stream, _by_beam ? &beams : nullptr));
    else
      LSH_CALL(decself_attention_i8(_buf_q.get(), k_cache, v_cache, _buf_b.get(), M * _tw._head_num,
                                  _cur_step + 1, _tw._max_step, _tw._head_num, _tw._dim_per_head,
                                  attn_scale, c[18] / Q, Q / c[7], _stream, _ops.blocked,
                                  _by_beam ? &beams : nullptr));
  }
  const float out_alpha = c[1] * c[7] / (c[13] * Q);
  const int32_t* sums = _out_sums.sums();
  if (_out_step) {
    _out_sums.launched();
  } else {
    TAP_CODES("self_ctx_q", _buf_b.get(), H);
    _ops.i8o(_buf_b.get(), w.w_self_out.get(), _buf_a.get(), M, H, H, out_alpha, _stream);
    TAP("self_out_q", _buf_a.get(), mh);
  }
  if (encdec_q_fused() ? _ln_in_encdec : _ln_in_product && _tw._dim_per_head % 16 == 0) {
    _ln = LnStep{_buf_a.get(), 0, 0, _cur_step_query[_res].get(), _cur_step_query[_res ^ 1].get(),
                 w.encdec_ln_scale.get(), w.encdec_ln_bias.get(), w.b_encdec_out.get(), nullptr,
                 c[13] / Q, Q / c[8], _tw._is_post_ln};
    if (_out_step) _ln.acc = sums, _ln.planes = 1, _ln.requant = out_alpha;
    _res ^= 1;
    return;
  }
  if (_out_step)
    LSH_CALL((residual_bias_ln_i8O<__half, int32_t>(
        sums, w.encdec_ln_scale.get(), w.encdec_ln_bias.get(), w.b_encdec_out.get(), _buf_b.get(),
        _cur_step_query[_res].get(), M, H, c[13] / Q, Q / c[8], _stream, _tw._is_post_ln, nullptr, 1, 0,
        _ops.blocked, out_alpha)));
  else
    LSH_CALL((residual_bias_ln_i8O<__half, int8_t>(
        _buf_a.get(), w.encdec_ln_scale.get(), w.encdec_ln_bias.get(), w.b_encdec_out.get(),
        _buf_b.get(), _cur_step_query[_res].get(), M, H, c[13] / Q, Q / c[8], _stream, _tw._is_post_ln,
        nullptr, 1, 0, _ops.blocked)));
  TAP_CODES("encdec_ln_q", _buf_b.get(), H);
  TAP("res_self", _cur_step_query[_res].get(), mh * sizeof(__half));
}

// Short sources, heads of 64: the query product and the cross attention are one launch (the same
// bytes).  With taps set they are two.
bool QuantDecoder::encdec_q_fused() const {
  return !step_taps.any() && _tw._dim_per_head == 64 &&
         encdec_q_attention_supported(_tw._beam_size, _tw._head_num, _tw._hidden_size, _batch_seq_len);
}

// The cross attention's out-projection goes with the self attention's: the launch of short sources,
// with the layer norm in it (so a run's steps have one launch with sums a layer, or two).
bool QuantDecoder::encdec_out() const {
  return _out_run && encdec_q_fused() &&
         encdec_q_attention_out_supported(_batch_size, _tw._head_num, _tw._hidden_size);
}

// Decided once a run: a step that left the sums' turn out would leave the next one's buffer uncleared.
// (A run whose caches outgrow the launch goes on without it: it never comes back.)
bool QuantDecoder::out_run() const {
  if (!_ops.blocked || _layers.empty() || step_taps.any() || decself_qkv_attention_enabled() ||
      !decself_attention_out_supported(_step_token_num, _tw._head_num, _tw._dim_per_head, 1))
    return false;
  // the launch of a short source with the layer norm in it reads sums only with its own out-projection
  if (encdec_q_fused() && _tw._hidden_size % 256 == 0 &&
      !encdec_q_attention_out_supported(_batch_size, _tw._head_num, _tw._hidden_size))
    return false;
  for (int l = 0; l < _tw._n_dec_layer; ++l) {
    const float* c = &_dec_clip_max[l * 19];
    if (c[1] * c[7] / (c[13] * _quant_range) == 0.f || c[3] * c[9] / (c[15] * _quant_range) == 0.f)
      return false;  // no code but zero: LnStep's "none"
  }
  return true;
}

void QuantDecoder::encdec_attention() {
  const int H = _tw._hidden_size, M = _step_token_num;
  const Layer& w = _layers[_layer_id];
  const float* c = &_dec_clip_max[_layer_id * 19];
  const float Q = _quant_range;

  const size_t mh = (size_t)M * H;
  if (encdec_q_fused()) {
    // the context goes to the second part of _buf_a because other workgroups still read the
    // rows (_buf_b, or the first part)
    int8_t* ctx_q = _buf_a.get() + _ops.rows(M) * H;
    const bool out = _out_step && encdec_out();
    const OutSums sums{w.w_encdec_out.get(), _out_sums.sums(), _out_sums.next_sums()};
    LSH_CALL(encdec_q_attention_f16(
        _buf_b.get(), w.w_encdec_q.get(), w.b_encdec_q.get(),
        _encdec_k.get() + (size_t)_layer_id * _layer_size_encdec_k,
        _encdec_v.get() + (size_t)_layer_id * _layer_size_encdec_k, _p_d_padding_mask, ctx_q,
        Q / c[9], _batch_size, _tw._beam_size, _tw._head_num, _batch_seq_len, H,
        c[2] * c[8] / (c[14] * Q), c[14] / Q, _stream, _ops.blocked, _ln_in_encdec ? &_ln : nullptr,
        out ? &sums : nullptr));
    if (out)
      _out_sums.launched();
    else
      _ops.i8o(ctx_q, w.w_encdec_out.get(), _buf_a.get(), M, H, H, c[3] * c[9] / (c[15] * Q), _stream);
    encdec_norm(out ? sums.acc : nullptr);
    return;
  }
  // q product; its epilogue is ker_arrange_encdec_q_i8I (fp16 q [batch, heads, beam, d])
  if (_tw._dim_per_head % 16 == 0) {
    _ops.encdec_q(_buf_b.get(), w.w_encdec_q.get(), w.b_encdec_q.get(), _query_buf1.get(), M, H,
                  _tw._beam_size, _tw._head_num, c[2] * c[8] / (c[14] * Q), c[14] / Q, _stream,
                  _ln_in_product ? &_ln : nullptr);
  } else {
    LSH_CALL(gemm_i8_i8o(_buf_b.get(), w.w_encdec_q.get(), _buf_a.get(), M, H, H,
                         c[2] * c[8] / (c[14] * Q), _stream));
    LSH_CALL(arrange_encdec_q_i8I<__half>(M, H, _stream, _buf_a.get(), w.b_encdec_q.get(),
                                          _query_buf1.get(), _tw._beam_size, _tw._dim_per_head,
                                          _tw._head_num, c[14] / Q));
  }
  TAP("encdec_q", _query_buf1.get(), mh * sizeof(__half));
  TAP("encdec_k", _encdec_k.get() + (size_t)_layer_id * _layer_size_encdec_k,
      (size_t)_batch_token_num * H * sizeof(__half));
  TAP("encdec_v", _encdec_v.get() + (size_t)_layer_id * _layer_size_encdec_k,
      (size_t)_batch_token_num * H * sizeof(__half));
  // scores -> masked softmax -> context -> merge heads + quantise, one kernel
  LSH_CALL(encdec_attention_f16(
      _query_buf1.get(), _encdec_k.get() + (size_t)_layer_id * _layer_size_encdec_k,
      _encdec_v.get() + (size_t)_layer_id * _layer_size_encdec_k, _p_d_padding_mask, nullptr,
      _buf_b.get(), Q / c[9], _batch_size, _tw._beam_size, _tw._head_num, _batch_seq_len,
      _tw._dim_per_head, _stream, _ops.blocked));
  TAP_CODES("encdec_ctx_q", _buf_b.get(), H);
  _ops.i8o(_buf_b.get(), w.w_encdec_out.get(), _buf_a.get(), M, H, H, c[3] * c[9] / (c[15] * Q),
           _stream);
  encdec_norm(nullptr);
}

// the layer norm behind the cross attention; sums: of the out-projection, codes in _buf_a otherwise
void QuantDecoder::encdec_norm(const int32_t* sums) {
  const int H = _tw._hidden_size, M = _step_token_num;
  const Layer& w = _layers[_layer_id];
  const float* c = &_dec_clip_max[_layer_id * 19];
  const float Q = _quant_range;
  const float out_alpha = c[3] * c[9] / (c[15] * Q);
  if (!sums) TAP("encdec_out_q", _buf_a.get(), (size_t)M * H);
  if (_ln_in_product) {
    _ln = LnStep{_buf_a.get(), 0, 0, _cur_step_query[_res].get(), _cur_step_query[_res ^ 1].get(),
                 w.ffn_ln_scale.get(), w.ffn_ln_bias.get(), w.b_ffn2.get(), nullptr, c[15] / Q,
                 Q / c[10], _tw._is_post_ln};
    if (sums) _ln.acc = sums, _ln.planes = 1, _ln.requant = out_alpha;
    _res ^= 1;
    return;
  }
  if (sums)
    LSH_CALL((residual_bias_ln_i8O<__half, int32_t>(
        sums, w.ffn_ln_scale.get(), w.ffn_ln_bias.get(), w.b_ffn2.get(), _buf_b.get(),
        _cur_step_query[_res].get(), M, H, c[15] / Q, Q / c[10], _stream, _tw._is_post_ln, nullptr, 1, 0,
        _ops.blocked, out_alpha)));
  else
    LSH_CALL((residual_bias_ln_i8O<__half, int8_t>(
        _buf_a.get(), w.ffn_ln_scale.get(), w.ffn_ln_bias.get(), w.b_ffn2.get(), _buf_b.get(),
        _cur_step_query[_res].get(), M, H, c[15] / Q, Q / c[10], _stream, _tw._is_post_ln, nullptr, 1, 0,
        _ops.blocked)));
  TAP_CODES("ffn_ln_q", _buf_b.get(), H);
  TAP("res_encdec", _cur_step_query[_res].get(), (size_t)M * H * sizeof(__half));
}

void QuantDecoder::ffn_add_norm() {
  const int H = _tw._hidden_size, I = _tw._inner_size, M = _step_token_num;
  const Layer& w = _layers[_layer_id];
  const float* c = &_dec_clip_max[_layer_id * 19];
  const float Q = _quant_range;

  // FFN1 GEMM with the bias + activation + requantisation in its epilogue
  // (with the layer norm inside the product _buf_a is its input)
  int8_t* act = (_ln_in_product ? _buf_b : _buf_a).get();
  _ops.lut(_buf_b.get(), w.w_ffn1.get(), act, w.ffn1_act_lut.get(), M, I, H,
           c[4] * c[10] / (c[16] * Q), _stream, _ln_in_product ? &_ln : nullptr);
  TAP_CODES("ffn1_act_q", act, I);
  // a tapped accumulator is one plane (the planes of a split product sum to it exactly)
  const bool tap_acc = step_taps.wants(_layer_id, _cur_step, "ffn2_acc");
  const int32_t* acc;
  const int nparts = _ops.i32_sums(act, w.w_ffn2.get(), _int32_ffn_out_buf.get(),
                                   _out_step && _ln_in_product ? _out_sums.ffn_sums() : nullptr, &acc, M, H, I, tap_acc ? 1 : 8,
                                   _stream);
  TAP("ffn2_acc", acc, (size_t)M * H * sizeof(int32_t));

  const float dequant_scale =
      _tw._use_gelu ? c[5] * c[11] / (Q * Q) : c[5] * c[11] / (2 * Q * Q);
  const __half *scale_ptr, *bias_ptr, *res_bias_ptr;
  float clip_max;
  if (_layer_id == _tw._n_dec_layer - 1) {
    scale_ptr = _out_ln_scale.get();
    bias_ptr = _out_ln_bias.get();
    res_bias_ptr = nullptr;
    clip_max = _output_ln_clip_max;
  } else {
    const Layer& nx = _layers[_layer_id + 1];
    scale_ptr = nx.self_ln_scale.get();
    bias_ptr = nx.self_ln_bias.get();
    res_bias_ptr = nx.b_self_out.get();
    clip_max = _dec_clip_max[(_layer_id + 1) * 19 + 6];
  }
  if (_ln_in_product && _layer_id != _tw._n_dec_layer - 1) {
    _ln = LnStep{acc, nparts, (long)M * H, _cur_step_query[_res].get(),
                 _cur_step_query[_res ^ 1].get(), scale_ptr, bias_ptr, res_bias_ptr,
                 w.ffn2_colsum.get(), dequant_scale, Q / clip_max, _tw._is_post_ln};
    _res ^= 1;
    return;
  }
  LSH_CALL((residual_bias_ln_i8O<__half, int32_t>(
      acc, scale_ptr, bias_ptr, res_bias_ptr, _buf_a.get(),
      _cur_step_query[_res].get(), M, H, dequant_scale, Q / clip_max, _stream, _tw._is_post_ln,
      w.ffn2_colsum.get(), nparts, (long)M * H,
      _ops.blocked && (!_qkv_attn || _layer_id == _tw._n_dec_layer - 1))));
  TAP_CODES("next_ln_q", _buf_a.get(), H);
  TAP("res_out", _cur_step_query[_res].get(), (size_t)M * H * sizeof(__half));
}

#undef TAP
#undef TAP_CODES

// QuantDecoder::sample and ::topk_greedy_search after its first step
// (inference/model/quant_decoder.cc.cu:952-984, 1108-1131): one token per row, in place
void QuantDecoder::sample_tokens() {
  int* alive = _alive_seq[_alive_cur].get();
  CHECK_GPU_ERROR(hipMemsetAsync(_sample_unfinished.get(), 0, sizeof(int), _stream));
  const float dq = _logits_clip_max / _quant_range;
  if (_tw._sampling_method == "topp") {
    LSH_CALL(dec_topp_sample_i8I<__half>(_step_token_num, _cur_step + 1, _tw._max_step, 1, _stream,
                                         _logits.get(), _logit_bias.get(), alive,
                                         _tw._trg_vocab_size, _tw._topp, _sample_unfinished.get(),
                                         _sample_state.get(), _tw._end_id, dq, _logits_stride));
  } else {
    const int k = _tw._sampling_method == "topk" ? _tw._topk : 1;
    LSH_CALL(dec_topk_sample_i8I<__half>(_step_token_num, _cur_step + 1, _tw._max_step, 1, _stream,
                                         _logits.get(), _logit_bias.get(), alive,
                                         _tw._trg_vocab_size, k, _sample_unfinished.get(),
                                         _sample_state.get(), _tw._end_id, dq, _logits_stride));
  }
  if (_rec_alive && _cur_step < _rec_max_steps)
    CHECK_GPU_ERROR(hipMemcpyAsync(
        _rec_alive + (size_t)_cur_step * _step_token_num * _tw._max_step, alive,
        (size_t)_step_token_num * _tw._max_step * sizeof(int), hipMemcpyDeviceToDevice, _stream));
}

void QuantDecoder::beam_search() {
  int* alive = _alive_seq[_alive_cur].get();
  int* alive_new = _alive_seq[_alive_cur ^ 1].get();
  LSH_CALL(beam_search_step_i8I<__half>(
      _logits.get(), _logit_bias.get(), _alive_seq_probs.get(), _alive_seq_score_own.get(), alive,
      alive_new, _top_score.get(), _top_idx.get(), _parent.get(), _num_finished.get(),
      _logits_clip_max / _quant_range, _tw._trg_vocab_size, _tw._max_step,
      _h_length_norm[_cur_step], _cur_step, _batch_size, _tw._beam_size, _tw._end_id, _stream,
      _topk_part_ws.get(), _topk_part_ws.size(), _logits_stride,
      _by_beam ? _beam_from[_alive_cur].get() : nullptr, _by_beam ? _beam_from[_alive_cur ^ 1].get() : nullptr,
      _beam_stride));
  if (_rec_alive && _cur_step < _rec_max_steps)
    CHECK_GPU_ERROR(hipMemcpyAsync(
        _rec_alive + (size_t)_cur_step * _step_token_num * _tw._max_step, alive_new,
        (size_t)_step_token_num * _tw._max_step * sizeof(int), hipMemcpyDeviceToDevice, _stream));

  /* ---refresh cache: k, v for decoder self attention--- (also on a step that turns out to be
   * the last one: the early-stop test reads the finished count after the step) */
  if (_cur_step > 0 && !_by_beam) {
    LSH_CALL(refresh_cache_by_parent_i8(
        _tw._n_dec_layer, _step_token_num, _stream, _parent.get(),
        _self_k_cache[_cache_cur].get(), _self_v_cache[_cache_cur].get(),
        _self_k_cache[_cache_cur ^ 1].get(), _self_v_cache[_cache_cur ^ 1].get(),
        _layer_size_self_k, _tw._beam_size, _tw._dim_per_head, _tw._head_num, _cur_step,
        _tw._max_step));
  }
}

}  // namespace hip
}  // namespace lightseq
