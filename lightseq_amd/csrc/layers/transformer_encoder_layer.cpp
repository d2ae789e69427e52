// Forward pass of the quantised encoder layer
// (lightseq/csrc/layers/transformer_encoder_layer.cpp:66-293) in seven launches (eight with a
// closing layer norm): the preparations, four products with the operators between them as
// epilogues, the attention core, the layer norm between the halves.
#include "transformer_encoder_layer.h"

#include <algorithm>

#include "context.h"

namespace lightseq {
namespace hip {

using namespace lsh;

template <typename T>
TransformerEncoderLayer<T>::TransformerEncoderLayer(
    int layer_id, int max_batch_tokens, int max_seq_len, int hidden_size, int num_heads,
    int intermediate_size, float attn_prob_dropout_ratio, float activation_dropout_ratio,
    float hidden_output_dropout_ratio, bool pre_or_postLayerNorm, std::string activation_fn,
    bool mask_future_tokens)
    : _layer_id(layer_id),
      _max_batch_tokens(max_batch_tokens),
      _max_seq_len(max_seq_len),
      _hidden_size(hidden_size),
      _heads(num_heads),
      _intermediate_size(intermediate_size),
      _is_pre_ln(pre_or_postLayerNorm),
      _activation_fn(activation_fn),
      _mask_future_tokens(mask_future_tokens),
      _kh((hidden_size + 63) & ~63),
      _ki((intermediate_size + 63) & ~63) {
  (void)attn_prob_dropout_ratio;  // ratios only matter in training mode, which Forward rejects
  (void)activation_dropout_ratio;
  (void)hidden_output_dropout_ratio;
  if (max_batch_tokens <= 0 || max_seq_len <= 0 || hidden_size <= 0 || num_heads <= 0 ||
      intermediate_size <= 0)
    throw std::runtime_error("TransformerEncoderLayer: sizes must be positive");
  if (hidden_size % num_heads != 0)
    throw std::runtime_error("TransformerEncoderLayer: hidden_size % num_heads != 0");
  const int hd = hidden_size / num_heads;
  if (hd != 32 && hd != 64 && hd != 128)
    throw std::runtime_error("TransformerEncoderLayer: head dim must be 32, 64 or 128");
  if (hidden_size % 16 != 0 || intermediate_size % 16 != 0)
    throw std::runtime_error(
        "TransformerEncoderLayer: hidden and intermediate size must be multiples of 16");
  if (activation_fn != "relu" && activation_fn != "gelu")
    throw std::runtime_error("not supported activation: " + activation_fn);

  const size_t tok = (size_t)max_batch_tokens, hs = (size_t)hidden_size,
               ims = (size_t)intermediate_size;
  const size_t rows = (tok + 15) & ~(size_t)15;
  _qkv.alloc(3 * tok * hs);
  _ffn_inp.alloc(tok * hs);
  _mask.alloc(tok);
  alloc_blocked(_qin, rows, hs, _kh);
  alloc_blocked(_act, rows, ims, _ki);
  _wqkv.alloc((3 * hs + 15) / 16 * 16 * _kh);
  _wout.alloc((hs + 15) / 16 * 16 * _kh);
  _winter.alloc((ims + 15) / 16 * 16 * _kh);
  _woutput.alloc((hs + 15) / 16 * 16 * _ki);
}

template <typename T>
size_t TransformerEncoderLayer<T>::param_count() const {
  const size_t hs = _hidden_size, ims = _intermediate_size;
  return hs * hs * 3 + hs * 3 + hs * hs + hs + hs + hs + hs * ims + ims + hs * ims + hs + hs +
         hs + 12;
}

template <typename T>
void TransformerEncoderLayer<T>::assign_weight_ptr(const T* weights_ptr) {
  if (!weights_ptr) throw std::runtime_error("assign_weight_ptr: null parameter blob");
  const size_t hs = _hidden_size, ims = _intermediate_size;
  const T* wptr = weights_ptr;
  _attn_qkvw_ptr = wptr; wptr += hs * hs * 3;
  _attn_qkvb_ptr = wptr; wptr += hs * 3;
  _attn_ow_ptr = wptr;   wptr += hs * hs;
  _attn_ob_ptr = wptr;   wptr += hs;
  _attn_nw_ptr = wptr;   wptr += hs;
  _attn_nb_ptr = wptr;   wptr += hs;
  _inter_w_ptr = wptr;   wptr += hs * ims;
  _inter_b_ptr = wptr;   wptr += ims;
  _output_w_ptr = wptr;  wptr += hs * ims;
  _output_b_ptr = wptr;  wptr += hs;
  _ffn_nw_ptr = wptr;    wptr += hs;
  _ffn_nb_ptr = wptr;    wptr += hs;
  _attn_qkv_cmax_ptr = wptr;       wptr += 3;
  _attn_out_cmax_ptr = wptr;       wptr += 3;
  _inter_cmax_ptr = wptr;          wptr += 3;
  _output_cmax_ptr = wptr;         wptr += 2;
  _attn_qkv_cache_cmax_ptr = wptr; wptr += 1;
}

template <typename T>
void TransformerEncoderLayer<T>::set_cur_batch_shape(int batch_size, int seq_len) {
  if (batch_size <= 0 || seq_len <= 0)
    throw std::runtime_error("set_cur_batch_shape: batch_size and seq_len must be positive");
  if ((long)batch_size * seq_len > _max_batch_tokens)
    throw std::runtime_error("Batch token numbers " + std::to_string((long)batch_size * seq_len) +
                             " exceeds the limit " + std::to_string(_max_batch_tokens) + ".");
  if (seq_len > _max_seq_len)
    throw std::runtime_error("Sequence length " + std::to_string(seq_len) +
                             " exceeds the limit " + std::to_string(_max_seq_len) + ".");
  _batch_size = batch_size;
  _seq_len = seq_len;
  _batch_tokens = batch_size * seq_len;
}

template <typename T>
void TransformerEncoderLayer<T>::SetTrainingMode(bool training) { _training = training; }

template <typename T>
void TransformerEncoderLayer<T>::SetQuantMode(bool enable_quant) { _enable_quant = enable_quant; }

// transformer_encoder_layer.cpp:277-293
template <typename T>
void TransformerEncoderLayer<T>::Forward(const T* input_ptr, const void* input_mask_ptr, int mask_kind,
                                         T* out_ptr) {
  if (!input_ptr || !out_ptr) throw std::runtime_error("Forward: null input or output");
  if (!_attn_qkvw_ptr) throw std::runtime_error("Forward: no parameter blob assigned");
  if (_batch_tokens == 0) throw std::runtime_error("Forward: set_cur_batch_shape not called");
  if (_training)
    throw std::runtime_error("Forward: training mode (dropout, saved activations) is not provided");
  if (!_enable_quant)
    throw std::runtime_error("Forward: only the quantised path of the layer is provided");
  _stream = Context::Instance().get_stream();
  const int tok = _batch_tokens, hs = _hidden_size, ims = _intermediate_size, hd = hs / _heads;
  const bool relu = _activation_fn == "relu";

  // what the first product reads, and what rides in later launches ahead of its reader
  LayerPrep prep, with_attn, with_norm;
  const bool riders = layer_attention_takes_riders(_seq_len, _seq_len, (long)_batch_size * _heads, hd);
  LayerPrep& later = riders ? with_attn : prep;
  LSH_CALL(prep.codes(_attn_qkvw_ptr, _wqkv.get(), _attn_qkv_cmax_ptr + 1, 3 * hs, hs, _kh));
  LSH_CALL(later.codes(_attn_ow_ptr, _wout.get(), _attn_out_cmax_ptr + 1, hs, hs, _kh));
  LSH_CALL(later.codes(_inter_w_ptr, _winter.get(), _inter_cmax_ptr + 1, ims, hs, _kh));
  LSH_CALL(with_norm.halfs(_output_w_ptr, _woutput.get(), _output_cmax_ptr + 1, hs, ims, _ki, 1, ims, 0));
  if (_is_pre_ln)
    LSH_CALL(prep.norm(input_ptr, _qin.get(), _attn_nw_ptr, _attn_nb_ptr, _attn_qkv_cmax_ptr, tok, hs, _kh));
  else
    LSH_CALL(prep.codes(input_ptr, _qin.get(), _attn_qkv_cmax_ptr, tok, hs, _kh));
  const T* mask = static_cast<const T*>(input_mask_ptr);
  if (mask && mask_kind != kMaskNone) {
    LSH_CALL(prep.mask(input_mask_ptr, mask_kind, _mask.get(), tok));
    mask = _mask.get();
  }
  LSH_CALL(prep.launch(_stream));

  // attention (:66-185)
  const size_t batch_dim = (size_t)tok * hs;
  T* const heads[3] = {_qkv.get(), _qkv.get() + batch_dim, _qkv.get() + 2 * batch_dim};
  const int len[3] = {_seq_len, _seq_len, _seq_len}, at[3] = {0, 0, 0};
  LSH_CALL(layer_gemm_heads(_qin.get(), _wqkv.get(), tok, 3, hs, _kh, _attn_qkvb_ptr, _attn_qkv_cmax_ptr,
                            _mask_future_tokens ? _attn_qkv_cache_cmax_ptr : nullptr, _seq_len, _heads,
                            heads, len, at, _stream));
  LSH_CALL(layer_attention_codes(heads[0], heads[1], heads[2], mask, _qin.get(), _attn_out_cmax_ptr, _kh,
                                 _batch_size, _seq_len, _seq_len, _heads, hd, _mask_future_tokens, _stream,
                                 riders ? &with_attn : nullptr));
  LSH_CALL(layer_gemm_residual(_qin.get(), _wout.get(), tok, hs, _kh, _attn_ob_ptr, _attn_out_cmax_ptr,
                               input_ptr, _ffn_inp.get(), _stream));

  // feed forward (:188-250); dropout.h:118-122: ReLU output goes through the unsigned quantiser.
  // The norm between the halves closes the first (post) or opens the second (pre).
  LSH_CALL(layer_norm_codes(_ffn_inp.get(), _is_pre_ln ? nullptr : _ffn_inp.get(), _qin.get(),
                            _is_pre_ln ? _ffn_nw_ptr : _attn_nw_ptr, _is_pre_ln ? _ffn_nb_ptr : _attn_nb_ptr,
                            _inter_cmax_ptr, tok, hs, _kh, _stream, &with_norm));
  LSH_CALL(layer_gemm_act(_qin.get(), _winter.get(), tok, ims, _kh, _inter_b_ptr, _inter_cmax_ptr,
                          _output_cmax_ptr, relu, _act.get(), _ki, _stream));
  LSH_CALL(layer_gemm_ffn2(_act.get(), _woutput.get(), tok, hs, _ki, _output_b_ptr, _ffn_inp.get(), out_ptr,
                           _stream));
  if (!_is_pre_ln)
    LSH_CALL(layer_norm_codes(out_ptr, out_ptr, nullptr, _ffn_nw_ptr, _ffn_nb_ptr, nullptr, tok, hs, _kh,
                              _stream));
}

template class TransformerEncoderLayer<__half>;

}  // namespace hip
}  // namespace lightseq
