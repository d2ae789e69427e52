// Forward pass of the quantised decoder layer
// (lightseq/csrc/layers/transformer_decoder_layer.cpp:91-547): one launch of preparations, six
// products with the operators between them as epilogues, the two attention cores, the layer
// norms between the blocks; layer 0 makes the cross-attention keys and values of the stack first.
#include "transformer_decoder_layer.h"

#include <algorithm>

#include "context.h"

namespace lightseq {
namespace hip {

using namespace lsh;

template <typename T>
int TransformerDecoderLayer<T>::_shared_nlayer = 0;
template <typename T>
DeviceBuffer<T> TransformerDecoderLayer<T>::_shared_encdec_kv;
template <typename T>
DeviceBuffer<T> TransformerDecoderLayer<T>::_shared_enc_out;
template <typename T>
DeviceBuffer<T> TransformerDecoderLayer<T>::_shared_kv_weight;
template <typename T>
T* TransformerDecoderLayer<T>::_shared_infer_encdec_kv_ptr = nullptr;

template <typename T>
TransformerDecoderLayer<T>::TransformerDecoderLayer(
    int layer_id, int max_batch_tokens, int max_seq_len, int hidden_size, int num_heads,
    int intermediate_size, float attn_prob_dropout_ratio, float activation_dropout_ratio,
    float hidden_output_dropout_ratio, bool pre_or_postLayerNorm, std::string activation_fn)
    : _layer_id(layer_id),
      _max_batch_tokens(max_batch_tokens),
      _max_seq_len(max_seq_len),
      _hidden_size(hidden_size),
      _heads(num_heads),
      _intermediate_size(intermediate_size),
      _is_pre_ln(pre_or_postLayerNorm),
      _activation_fn(activation_fn),
      _kh((hidden_size + 63) & ~63),
      _ki((intermediate_size + 63) & ~63) {
  (void)attn_prob_dropout_ratio;  // ratios only matter in training mode, which Forward rejects
  (void)activation_dropout_ratio;
  (void)hidden_output_dropout_ratio;
  if (layer_id < 0) throw std::runtime_error("TransformerDecoderLayer: negative layer id");
  if (max_batch_tokens <= 0 || max_seq_len <= 0 || hidden_size <= 0 || num_heads <= 0 ||
      intermediate_size <= 0)
    throw std::runtime_error("TransformerDecoderLayer: sizes must be positive");
  if (hidden_size % num_heads != 0)
    throw std::runtime_error("TransformerDecoderLayer: hidden_size % num_heads != 0");
  const int hd = hidden_size / num_heads;
  if (hd != 32 && hd != 64 && hd != 128)
    throw std::runtime_error("TransformerDecoderLayer: head dim must be 32, 64 or 128");
  if (hidden_size % 16 != 0 || intermediate_size % 16 != 0)
    throw std::runtime_error(
        "TransformerDecoderLayer: hidden and intermediate size must be multiples of 16");
  if (activation_fn != "relu" && activation_fn != "gelu")
    throw std::runtime_error("not supported activation: " + activation_fn);

  const size_t tok = (size_t)max_batch_tokens, hs = (size_t)hidden_size,
               ims = (size_t)intermediate_size;
  const size_t rows = (tok + 15) & ~(size_t)15;
  _qkv.alloc(3 * tok * hs);
  _encdec_inp.alloc(tok * hs);
  _ffn_inp.alloc(tok * hs);
  _mask.alloc(tok);
  alloc_blocked(_qin, rows, hs, _kh);
  alloc_blocked(_act, rows, ims, _ki);
  const size_t square = (hs + 15) / 16 * 16 * _kh;
  _wqkv.alloc((3 * hs + 15) / 16 * 16 * _kh);
  _wself_out.alloc(square);
  _wq.alloc(square);
  _wcross_out.alloc(square);
  _winter.alloc((ims + 15) / 16 * 16 * _kh);
  _woutput.alloc((hs + 15) / 16 * 16 * _ki);
  ++_shared_nlayer;  // transformer_decoder_layer.cpp:64
}

template <typename T>
TransformerDecoderLayer<T>::~TransformerDecoderLayer() {
  // The reference never takes a layer down; here the count follows the live layers, so that
  // one process can build a second stack after destroying the first.
  if (--_shared_nlayer == 0) {
    _shared_encdec_kv = DeviceBuffer<T>();
    _shared_enc_out = DeviceBuffer<T>();
    _shared_kv_weight = DeviceBuffer<T>();
    _shared_infer_encdec_kv_ptr = nullptr;
  }
}

template <typename T>
size_t TransformerDecoderLayer<T>::param_count() const {
  const size_t hs = _hidden_size, ims = _intermediate_size;
  size_t n = hs * hs * 3 + hs * 3 + hs * hs + 3 * hs     // self attention
             + hs * hs + hs + hs * hs + 3 * hs           // cross attention
             + hs * ims + ims + hs * ims + 3 * hs        // ffn
             + 3 * 6 + 5 + 1;                            // clip values
  if (_layer_id == 0) n += (size_t)_shared_nlayer * (hs * hs * 2 + hs * 2);
  return n;
}

template <typename T>
void TransformerDecoderLayer<T>::assign_weight_ptr(const T* weights_ptr) {
  if (!weights_ptr) throw std::runtime_error("assign_weight_ptr: null parameter blob");
  const size_t hs = _hidden_size, ims = _intermediate_size;
  const T* wptr = weights_ptr;
  _attn_qkvw_ptr = wptr; wptr += hs * hs * 3;
  _attn_qkvb_ptr = wptr; wptr += hs * 3;
  _attn_ow_ptr = wptr;   wptr += hs * hs;
  _attn_ob_ptr = wptr;   wptr += hs;
  _attn_nw_ptr = wptr;   wptr += hs;
  _attn_nb_ptr = wptr;   wptr += hs;
  _encdec_attn_qw_ptr = wptr; wptr += hs * hs;
  _encdec_attn_qb_ptr = wptr; wptr += hs;
  _encdec_attn_ow_ptr = wptr; wptr += hs * hs;
  _encdec_attn_ob_ptr = wptr; wptr += hs;
  _encdec_attn_nw_ptr = wptr; wptr += hs;
  _encdec_attn_nb_ptr = wptr; wptr += hs;
  _inter_w_ptr = wptr;   wptr += hs * ims;
  _inter_b_ptr = wptr;   wptr += ims;
  _output_w_ptr = wptr;  wptr += hs * ims;
  _output_b_ptr = wptr;  wptr += hs;
  _ffn_nw_ptr = wptr;    wptr += hs;
  _ffn_nb_ptr = wptr;    wptr += hs;
  _attn_qkv_cmax_ptr = wptr;       wptr += 3;
  _attn_out_cmax_ptr = wptr;       wptr += 3;
  _encdec_qkv_cmax_ptr = wptr;     wptr += 3;
  _encdec_out_cmax_ptr = wptr;     wptr += 3;
  _inter_cmax_ptr = wptr;          wptr += 3;
  _output_cmax_ptr = wptr;         wptr += 3;
  _encdec_kv_cmax_ptr = wptr;      wptr += 5;
  _attn_qkv_cache_cmax_ptr = wptr; wptr += 1;
  if (_layer_id == 0) {
    _encdec_attn_kvw_ptr = wptr; wptr += (size_t)_shared_nlayer * hs * hs * 2;
    _encdec_attn_kvb_ptr = wptr; wptr += (size_t)_shared_nlayer * hs * 2;
  } else {
    _encdec_attn_kvw_ptr = nullptr;
    _encdec_attn_kvb_ptr = nullptr;
    _encdec_kv_cmax_ptr = nullptr;
  }
}

template <typename T>
void TransformerDecoderLayer<T>::set_cur_batch_shape(int batch_size, int trg_seq_len,
                                                     int src_seq_len, int step) {
  if (batch_size <= 0 || trg_seq_len <= 0 || src_seq_len <= 0)
    throw std::runtime_error("set_cur_batch_shape: batch_size and lengths must be positive");
  if ((long)batch_size * trg_seq_len > _max_batch_tokens)
    throw std::runtime_error("Batch token numbers " +
                             std::to_string((long)batch_size * trg_seq_len) +
                             " exceeds the limit " + std::to_string(_max_batch_tokens) + ".");
  if ((long)batch_size * src_seq_len > _max_batch_tokens)
    throw std::runtime_error("Source token numbers " +
                             std::to_string((long)batch_size * src_seq_len) +
                             " exceeds the limit " + std::to_string(_max_batch_tokens) + ".");
  if (src_seq_len > _max_seq_len || (step < 0 ? trg_seq_len : step + 1) > _max_seq_len)
    throw std::runtime_error("Sequence length exceeds the limit " +
                             std::to_string(_max_seq_len) + ".");
  _batch_size = batch_size;
  _trg_seq_len = trg_seq_len;  // the beam size in a decoding step
  _src_seq_len = src_seq_len;
  _batch_tokens = batch_size * trg_seq_len;
  _predict = step >= 0;
  _step = _predict ? step : -1;
}

template <typename T>
void TransformerDecoderLayer<T>::SetTrainingMode(bool training) { _training = training; }

template <typename T>
void TransformerDecoderLayer<T>::SetQuantMode(bool enable_quant) { _enable_quant = enable_quant; }

// transformer_decoder_layer.cpp:508-547
template <typename T>
void TransformerDecoderLayer<T>::Forward(const T* dec_input_ptr, const T* enc_output_ptr,
                                         long enc_stride_b, long enc_stride_s,
                                         const void* enc_mask_ptr, int mask_kind,
                                         T* dec_output_ptr, const std::vector<T*>& cache) {
  if (!dec_input_ptr || !dec_output_ptr) throw std::runtime_error("Forward: null input or output");
  if (!_attn_qkvw_ptr) throw std::runtime_error("Forward: no parameter blob assigned");
  if (_batch_tokens == 0) throw std::runtime_error("Forward: set_cur_batch_shape not called");
  if (_training)
    throw std::runtime_error("Forward: training mode (dropout, saved activations) is not provided");
  if (!_enable_quant)
    throw std::runtime_error("Forward: only the quantised path of the layer is provided");
  if (_predict) {
    if (cache.size() < (_layer_id == 0 ? 5u : 4u))
      throw std::runtime_error("Forward: a decoding step needs the cache pointers");
    if (!cache[0] || !cache[1] || (_step > 0 && (!cache[2] || !cache[3])) ||
        (_layer_id == 0 && !cache[4]))
      throw std::runtime_error("Forward: null cache pointer");
  }
  _stream = Context::Instance().get_stream();

  const int tok = _batch_tokens, hs = _hidden_size, ims = _intermediate_size, hd = hs / _heads;
  const bool relu = _activation_fn == "relu";
  const int src_tok = _batch_size * _src_seq_len;

  const int self_batch = _predict ? _batch_size * _trg_seq_len : _batch_size;
  const int from_len = _predict ? 1 : _trg_seq_len, to_len = _predict ? _step + 1 : _trg_seq_len;
  // what the first product reads, and what rides in later launches ahead of its reader
  LayerPrep prep, with_self, with_norm, with_cross, with_norm2;
  const bool self_riders = layer_attention_takes_riders(from_len, to_len, (long)self_batch * _heads, hd);
  const bool cross_riders = layer_attention_takes_riders(_trg_seq_len, _src_seq_len, (long)_batch_size * _heads, hd);
  LayerPrep& early = self_riders ? with_self : prep;
  LSH_CALL(prep.codes(_attn_qkvw_ptr, _wqkv.get(), _attn_qkv_cmax_ptr + 1, 3 * hs, hs, _kh));
  LSH_CALL(early.codes(_attn_ow_ptr, _wself_out.get(), _attn_out_cmax_ptr + 1, hs, hs, _kh));
  LSH_CALL(early.codes(_encdec_attn_qw_ptr, _wq.get(), _encdec_qkv_cmax_ptr + 1, hs, hs, _kh));
  LSH_CALL(with_norm.codes(_encdec_attn_ow_ptr, _wcross_out.get(), _encdec_out_cmax_ptr + 1, hs, hs, _kh));
  LSH_CALL((cross_riders ? with_cross : with_norm)
               .codes(_inter_w_ptr, _winter.get(), _inter_cmax_ptr + 1, ims, hs, _kh));
  LSH_CALL(with_norm2.halfs(_output_w_ptr, _woutput.get(), _output_cmax_ptr + 1, hs, ims, _ki, 1, ims, 0));
  if (_is_pre_ln)
    LSH_CALL(prep.norm(dec_input_ptr, _qin.get(), _attn_nw_ptr, _attn_nb_ptr, _attn_qkv_cmax_ptr, tok, hs, _kh));
  else
    LSH_CALL(prep.codes(dec_input_ptr, _qin.get(), _attn_qkv_cmax_ptr, tok, hs, _kh));
  const T* mask = static_cast<const T*>(enc_mask_ptr);
  if (mask && mask_kind != kMaskNone) {
    LSH_CALL(prep.mask(enc_mask_ptr, mask_kind, _mask.get(), src_tok));
    mask = _mask.get();
  }
  if (_predict && _step > 0)  // :173-180: new cache = previous cache ++ this step's k / v
    for (int i = 0; i < 2; ++i)
      LSH_CALL(prep.grow(cache[2 + i], cache[i], self_batch * _heads, _step * hd, (long)(_step + 1) * hd));
  const int nl = _shared_nlayer;
  if (_layer_id == 0 && _predict) _shared_infer_encdec_kv_ptr = cache[4];
  if (makes_encdec_kv()) {
    // :236-262: fake-quantised weights, the encoder output as it is
    if (!enc_output_ptr) throw std::runtime_error("Forward: null encoder output");
    if (reinterpret_cast<uintptr_t>(enc_output_ptr) % 16 != 0 || (_batch_size > 1 && enc_stride_b % 8 != 0) ||
        (_src_seq_len > 1 && enc_stride_s % 8 != 0))
      throw std::runtime_error("Forward: the encoder output must be 16-byte aligned, its strides multiples of 8");
    if (!_encdec_attn_kvw_ptr)
      throw std::runtime_error("Forward: layer 0 holds no cross-attention k/v weights");
    const size_t enc_elems = (((size_t)_max_batch_tokens + 15) & ~(size_t)15) * _kh;
    if (_shared_enc_out.size() != enc_elems) _shared_enc_out.alloc(enc_elems);
    const size_t kv_elems = (size_t)nl * 2 * _max_batch_tokens * hs;
    if (!_predict && _shared_encdec_kv.size() != kv_elems) _shared_encdec_kv.alloc(kv_elems);
    const size_t w_elems = ((size_t)nl * 2 * hs + 15) / 16 * 16 * _kh;
    if (_shared_kv_weight.size() != w_elems) _shared_kv_weight.alloc(w_elems);
    LSH_CALL(prep.halfs(_encdec_attn_kvw_ptr, _shared_kv_weight.get(), _encdec_kv_cmax_ptr + 1, nl * 2 * hs,
                        hs, _kh, 1, hs, 0));
    LSH_CALL(prep.halfs(enc_output_ptr, _shared_enc_out.get(), nullptr, src_tok, hs, _kh, _src_seq_len,
                        enc_stride_b, enc_stride_s));
  }
  LSH_CALL(prep.launch(_stream));

  const size_t src_dim = (size_t)src_tok * hs;
  T* kv = _predict ? _shared_infer_encdec_kv_ptr : _shared_encdec_kv.get();
  if (makes_encdec_kv())
    LSH_CALL(gemm_blk_kv_f16(_shared_enc_out.get(), _shared_kv_weight.get(), src_tok, nl, hs, _kh,
                             _encdec_attn_kvb_ptr, _src_seq_len, _heads, kv, kv + src_dim,
                             (long)(2 * src_dim), _stream));
  if (!kv) throw std::runtime_error("Forward: layer 0 has not produced the cross-attention k/v");

  // self attention (:91-233); k and v leave the product as the cache will hold them: fake-quantised
  // (:134-138)
  const size_t batch_dim = (size_t)tok * hs;
  T* q = _qkv.get();
  T* const self[3] = {q, _predict ? cache[0] : q + batch_dim, _predict ? cache[1] : q + 2 * batch_dim};
  const int self_at = _predict ? _step : 0;
  const int len[3] = {from_len, to_len, to_len}, at[3] = {0, self_at, self_at};
  LSH_CALL(layer_gemm_heads(_qin.get(), _wqkv.get(), tok, 3, hs, _kh, _attn_qkvb_ptr, _attn_qkv_cmax_ptr,
                            _attn_qkv_cache_cmax_ptr, from_len, _heads, self, len, at, _stream));
  LSH_CALL(layer_attention_codes(self[0], self[1], self[2], nullptr, _qin.get(), _attn_out_cmax_ptr, _kh,
                                 self_batch, from_len, to_len, _heads, hd, !_predict, _stream,
                                 self_riders ? &with_self : nullptr));
  LSH_CALL(layer_gemm_residual(_qin.get(), _wself_out.get(), tok, hs, _kh, _attn_ob_ptr, _attn_out_cmax_ptr,
                               dec_input_ptr, _encdec_inp.get(), _stream));

  // cross attention (:278-412); a norm between two blocks closes the first (post) or opens the
  // second (pre)
  T* x = _encdec_inp.get();
  LSH_CALL(layer_norm_codes(x, _is_pre_ln ? nullptr : x, _qin.get(),
                            _is_pre_ln ? _encdec_attn_nw_ptr : _attn_nw_ptr,
                            _is_pre_ln ? _encdec_attn_nb_ptr : _attn_nb_ptr, _encdec_qkv_cmax_ptr, tok, hs,
                            _kh, _stream, &with_norm));
  T* const cross[1] = {q};
  LSH_CALL(layer_gemm_heads(_qin.get(), _wq.get(), tok, 1, hs, _kh, _encdec_attn_qb_ptr,
                            _encdec_qkv_cmax_ptr, nullptr, _trg_seq_len, _heads, cross, &_trg_seq_len, at,
                            _stream));
  const T* k = kv + (size_t)_layer_id * 2 * src_dim;
  LSH_CALL(layer_attention_codes(q, k, k + src_dim, mask, _qin.get(), _encdec_out_cmax_ptr, _kh, _batch_size,
                                 _trg_seq_len, _src_seq_len, _heads, hd, false, _stream,
                                 cross_riders ? &with_cross : nullptr));
  LSH_CALL(layer_gemm_residual(_qin.get(), _wcross_out.get(), tok, hs, _kh, _encdec_attn_ob_ptr,
                               _encdec_out_cmax_ptr, x, _ffn_inp.get(), _stream));

  // feed forward (:415-483); dropout.h:118-122: ReLU output goes through the unsigned quantiser
  x = _ffn_inp.get();
  LSH_CALL(layer_norm_codes(x, _is_pre_ln ? nullptr : x, _qin.get(),
                            _is_pre_ln ? _ffn_nw_ptr : _encdec_attn_nw_ptr,
                            _is_pre_ln ? _ffn_nb_ptr : _encdec_attn_nb_ptr, _inter_cmax_ptr, tok, hs, _kh,
                            _stream, &with_norm2));
  LSH_CALL(layer_gemm_act(_qin.get(), _winter.get(), tok, ims, _kh, _inter_b_ptr, _inter_cmax_ptr,
                          _output_cmax_ptr, relu, _act.get(), _ki, _stream));
  LSH_CALL(layer_gemm_ffn2(_act.get(), _woutput.get(), tok, hs, _ki, _output_b_ptr, x, dec_output_ptr,
                           _stream));
  if (!_is_pre_ln)
    LSH_CALL(layer_norm_codes(dec_output_ptr, dec_output_ptr, nullptr, _ffn_nw_ptr, _ffn_nb_ptr, nullptr,
                              tok, hs, _kh, _stream));
}

template class TransformerDecoderLayer<__half>;

}  // namespace hip
}  // namespace lightseq
