#include "quant_bert.h"

#include <algorithm>

namespace lightseq {
namespace hip {

QuantBert::QuantBert(const std::string weight_path, const int max_batch_size)
    : LSModel({"token_ids"}, {"encoder_output"}), _max_batch_size(max_batch_size) {
  if (max_batch_size <= 0) throw std::runtime_error("max_batch_size must be positive");
  CHECK_GPU_ERROR(hipSetDevice(0));
  stream_.create();
  side_stream_.create();
  h_lens_.alloc(max_batch_size);

  std::string res = tw_.initializing(weight_path);
  if (!res.empty()) throw std::runtime_error(res);

  const size_t tokens = (size_t)_max_batch_size * tw_._max_step;
  d_input_.alloc(tokens);
  d_padding_mask_.alloc(tokens);
  d_encoder_output_.alloc(tokens * tw_._hidden_size);

  encoder_ = std::make_shared<QuantBertEncoder>(max_batch_size, d_input_.get(),
                                                d_padding_mask_.get(), d_encoder_output_.get(),
                                                tw_, stream_);
  res = encoder_->check();
  if (!res.empty()) throw std::runtime_error(res);
  encoder_->init_buffer();
  encoder_->make_padding_row();
  CHECK_GPU_ERROR(hipStreamSynchronize(stream_));
  describe_input(0, kInt32, {_max_batch_size, tw_._max_step}, &encoder_->_p_d_token_id);
  describe_output(0, kFloat16, {_max_batch_size, tw_._max_step, tw_._hidden_size},
                  &encoder_->_p_d_output);
}

QuantBert::~QuantBert() {
  encoder_.reset();  // before the buffers and the stream it uses (members, released after this)
}

void QuantBert::Infer() { infer(nullptr, false); }

// Whether the padding of a result goes to the host by a launch of its own, ahead of the stack: it costs
// a launch and a second stream to wait for, and slows what runs beside it; the link needs 18.5 us for
// a MB.  (7 x 75 x 768 with 0.55 MB of padding: 441 us so, 438 in one go.)
bool QuantBert::pads_first(int batch, int seq_len, bool host_f16) {
  if (batch > _max_batch_size || seq_len > tw_._max_step) return false;  // refused by the encoder
  long pads = 0;
  for (int b = 0; b < batch; ++b) {
    int n = 0;
    while (n < seq_len && host_ids_[(long)b * seq_len + seq_len - 1 - n] == tw_._padding_id) ++n;
    h_lens_.get()[b] = seq_len - n;
    pads += n;
  }
  return pads * tw_._hidden_size * (host_f16 ? 2 : 4) >= (1 << 20);
}

void QuantBert::infer(void* host_out, bool host_f16) {
  if (input_shapes_[0].size() != 2) throw std::runtime_error("token_ids must be 2-D");
  int batch_size = input_shapes_[0][0], seq_len = input_shapes_[0][1];
  const int H = tw_._hidden_size;
  const __half* padding = host_out && host_ids_ && pads_first(batch_size, seq_len, host_f16)
                              ? encoder_->padding_row(batch_size, seq_len) : nullptr;
  // the caller's memory is not left with a kernel writing it, however this ends
  struct Waits {
    hipStream_t s = nullptr;
    ~Waits() {
      if (s) (void)hipStreamSynchronize(s);
    }
  } side;
  if (padding) {
    side.s = side_stream_;
    LSH_CALL(lsh::host_padding(padding, h_lens_.get(), host_out, host_f16, batch_size, seq_len, H, side_stream_));
  }
  auto run = [&] {
    encoder_->run_one_infer(batch_size, seq_len, host_ids_);
    if (host_out) {
      const long n = (long)batch_size * seq_len * H;
      if (padding)
        LSH_CALL(lsh::host_tokens(encoder_->_p_d_output, encoder_->sequences(), host_out, host_f16, batch_size,
                                  seq_len, H, stream_));
      else if (host_f16) LSH_CALL(lsh::copy_words(encoder_->_p_d_output, host_out, n / 2, stream_));
      else LSH_CALL(lsh::widen_f16(encoder_->_p_d_output, static_cast<float*>(host_out), n, stream_));
    }
    CHECK_GPU_ERROR(hipStreamSynchronize(stream_));
  };
  run();
  if (encoder_->finish_infer()) {  // a route gave up and was switched off: once more without it
    run();
    encoder_->finish_infer();
  }
  encoder_->collect_profile();
  set_output_shape(0, {batch_size, seq_len, tw_._hidden_size});
}

// Where the GPU sees `bytes` bytes of the caller's memory.  A kernel writes there: memory that was not
// allocated as pinned would be a fault, so it is asked for first.
static void* device_view(void* p, size_t bytes) {
  hipPointerAttribute_t first{}, last{};
  const bool known = hipPointerGetAttributes(&first, p) == hipSuccess &&
                     hipPointerGetAttributes(&last, static_cast<char*>(p) + bytes - 1) == hipSuccess;
  if (!known) (void)hipGetLastError();
  if (!known || first.type == hipMemoryTypeUnregistered || !first.devicePointer ||
      static_cast<char*>(last.devicePointer) != static_cast<char*>(first.devicePointer) + bytes - 1)
    throw std::runtime_error("host_out is not pinned host memory of the size of the output");
  return first.devicePointer;
}

void QuantBert::InferHost(const int* ids, int batch, int seq_len, void* host_out, bool host_f16) {
  // more ids than the input holds: Infer() names the limit that was passed
  const size_t n = (size_t)std::max(batch, 0) * (size_t)std::max(seq_len, 0);
  if (ids && n > 0 && n <= d_input_.size()) {
    if (host_out) host_out = device_view(host_out, n * tw_._hidden_size * (host_f16 ? sizeof(__half) : sizeof(float)));
    h_ids_.upload(ids, n, d_input_.get(), d_input_.size(), stream_);
  }
  set_input_ptr(0, d_input_.get());
  set_input_shape(0, {batch, seq_len});
  HostIdsScope scope(host_ids_, ids);
  infer(host_out, host_f16);
}

LSMODEL_REGISTER(QuantBert)

}  // namespace hip
}  // namespace lightseq
