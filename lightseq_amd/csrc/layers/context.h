// Process-wide launch context of the layer API: the stream every layer launches on
// (the reference's Context singleton, lightseq/csrc/ops/includes/context.h:14-43, without
// its cuBLAS handles -- the GEMMs here are this library's own kernels).
#pragma once

#include <hip/hip_runtime.h>

#include "../model/model_util.h"

namespace lightseq {
namespace hip {

class Context {
 public:
  static Context& Instance() {
    static Context ctx;
    return ctx;
  }
  void set_stream(hipStream_t stream) { _stream = stream; }
  hipStream_t get_stream() const { return _stream; }

 private:
  Context() : _stream(nullptr) {}
  hipStream_t _stream;
};

// Room for a blocked matrix [rows, k] with rows of k_pad elements.  The columns beyond k are
// multiplied like the others and written by nobody: zeros.
template <typename T>
void alloc_blocked(DeviceBuffer<T>& buf, size_t rows, int k, int k_pad) {
  buf.alloc(rows * (size_t)k_pad);
  if (k_pad == k) return;
  CHECK_GPU_ERROR(hipMemset(buf.get(), 0, rows * (size_t)k_pad * sizeof(T)));
  CHECK_GPU_ERROR(hipDeviceSynchronize());
}

}  // namespace hip
}  // namespace lightseq
