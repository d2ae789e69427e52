// Small host-side helpers of the model layer: error check that throws (the
// reference's CHECK_GPU_ERROR, lightseq/inference/tools/util.h:69-79), a device
// buffer owner and host<->device copies.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <list>
#include <map>
#include <stdexcept>
#include <string>
#include <thread>
#include <unordered_map>
#include <unordered_set>
#include <vector>

#include "../ls_launch.h"

namespace lightseq {
namespace hip {

inline void check_gpu_error(hipError_t e, const char* file, int line) {
  if (e != hipSuccess)
    throw std::runtime_error(std::string("[HIP][ERROR] ") + file + "(" + std::to_string(line) +
                             "): " + hipGetErrorName(e) + " " + hipGetErrorString(e));
}
#define CHECK_GPU_ERROR(val) ::lightseq::hip::check_gpu_error((val), __FILE__, __LINE__)

// status of a library launcher -> exception carrying its message
inline void check_status(int rc) {
  if (rc != LSH_OK) throw std::runtime_error(lsh_last_error());
}
#define LSH_CALL(expr) ::lightseq::hip::check_status((expr))

// Owning device allocation.
template <typename T>
class DeviceBuffer {
 public:
  DeviceBuffer() {}
  explicit DeviceBuffer(size_t n) { alloc(n); }
  DeviceBuffer(const DeviceBuffer&) = delete;
  DeviceBuffer& operator=(const DeviceBuffer&) = delete;
  DeviceBuffer(DeviceBuffer&& o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr; o.n_ = 0; }
  DeviceBuffer& operator=(DeviceBuffer&& o) noexcept {
    if (this != &o) { release(); p_ = o.p_; n_ = o.n_; o.p_ = nullptr; o.n_ = 0; }
    return *this;
  }
  ~DeviceBuffer() { release(); }
  void alloc(size_t n) {
    release();
    if (n == 0) return;
    CHECK_GPU_ERROR(hipMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T)));
    n_ = n;
  }
  void upload(const T* host, size_t n, hipStream_t s) {
    if (n > n_) throw std::runtime_error("DeviceBuffer::upload: too large");
    CHECK_GPU_ERROR(hipMemcpyAsync(p_, host, n * sizeof(T), hipMemcpyHostToDevice, s));
  }
  T* get() const { return p_; }
  size_t size() const { return n_; }

 private:
  void release() {
    if (p_) (void)hipFree(p_);
    p_ = nullptr;
    n_ = 0;
  }
  T* p_ = nullptr;
  size_t n_ = 0;
};

// Token ids that arrive in host memory: a pinned buffer of the model's largest input, from which a
// kernel brings them to the GPU.  The buffer is free again once the model's stream has been
// synchronised, which every call does before it returns.
class HostIds {
 public:
  HostIds() = default;
  HostIds(const HostIds&) = delete;
  HostIds& operator=(const HostIds&) = delete;
  ~HostIds() {
    if (p_) (void)hipHostFree(p_);
  }
  // `ids` (n of them, n <= capacity) on their way to `dst`
  void upload(const int* ids, size_t n, int* dst, size_t capacity, hipStream_t s) {
    if (!p_) CHECK_GPU_ERROR(hipHostMalloc(reinterpret_cast<void**>(&p_), capacity * sizeof(int)));
    std::memcpy(p_, ids, n * sizeof(int));
    LSH_CALL(lsh::copy_words(p_, dst, (long)n, s));
  }

 private:
  int* p_ = nullptr;
};

// Pinned ints that kernels read.
class PinnedInts {
 public:
  PinnedInts() = default;
  PinnedInts(const PinnedInts&) = delete;
  PinnedInts& operator=(const PinnedInts&) = delete;
  ~PinnedInts() {
    if (p_) (void)hipHostFree(p_);
  }
  void alloc(size_t n) {
    if (!p_) CHECK_GPU_ERROR(hipHostMalloc(reinterpret_cast<void**>(&p_), n * sizeof(int)));
  }
  int* get() const { return p_; }

 private:
  int* p_ = nullptr;
};

// A pointer that is set for the length of a call.
class HostIdsScope {
 public:
  HostIdsScope(const int*& slot, const int* ids) : slot_(slot) { slot_ = ids; }
  ~HostIdsScope() { slot_ = nullptr; }
  HostIdsScope(const HostIdsScope&) = delete;
  HostIdsScope& operator=(const HostIdsScope&) = delete;

 private:
  const int*& slot_;
};

// A HIP stream of the default priority that is destroyed with its owner.
class StreamOwner {
 public:
  StreamOwner() = default;
  StreamOwner(const StreamOwner&) = delete;
  StreamOwner& operator=(const StreamOwner&) = delete;
  ~StreamOwner() {
    if (s_) (void)hipStreamDestroy(s_);
  }
  void create() {
    if (!s_) CHECK_GPU_ERROR(hipStreamCreate(&s_));
  }
  hipStream_t get() const { return s_; }
  operator hipStream_t() const { return s_; }

 private:
  hipStream_t s_ = nullptr;
};

// Three HIP events on the model's stream per Infer() of a generation model: entry, start of the
// step loop, end of the step loop.  times() is valid once the stream has been synchronised.
class PhaseEvents {
 public:
  PhaseEvents() = default;
  PhaseEvents(const PhaseEvents&) = delete;
  PhaseEvents& operator=(const PhaseEvents&) = delete;
  ~PhaseEvents() {
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
  }
  void mark(int i, hipStream_t s) {
    if (!ev_[i]) CHECK_GPU_ERROR(hipEventCreate(&ev_[i]));
    CHECK_GPU_ERROR(hipEventRecord(ev_[i], s));
    if (i == 0) loop_steps_ = 0;
    marked_ |= 1 << i;
  }
  void set_loop_steps(int n) { loop_steps_ = n; }
  // milliseconds before the step loop and inside it, steps the loop ran; false before a run
  bool times(float* prepare_ms, float* steps_ms, int* steps) const {
    if (marked_ != 7) return false;
    CHECK_GPU_ERROR(hipEventElapsedTime(prepare_ms, ev_[0], ev_[1]));
    CHECK_GPU_ERROR(hipEventElapsedTime(steps_ms, ev_[1], ev_[2]));
    *steps = loop_steps_;
    return true;
  }

 private:
  hipEvent_t ev_[3] = {nullptr, nullptr, nullptr};
  int marked_ = 0, loop_steps_ = 0;
};

// Debug taps of a generation step (parity bisection): device-to-device copies of named
// intermediates of decoder layer `layer` at step `step` into buffers the caller owns.  A name
// registered with a null pointer is forgotten.  A layer < 0 at the copy site means "any".
class StepTaps {
 public:
  void set(int layer, const std::string& name, void* dst) {
    _layer = layer;
    if (dst) _dst[name] = dst;
    else _dst.erase(name);
  }
  void set_step(int step) { _step = step; }
  bool any() const { return !_dst.empty(); }
  bool wants(int layer, int step, const char* name) const {
    return !_dst.empty() && step == _step && (layer < 0 || layer == _layer) && _dst.count(name);
  }
  // an int8 matrix, copied row-major whichever way the model holds it
  void copy_codes(int layer, int step, const char* name, const int8_t* src, int rows, int cols,
                  bool blocked, hipStream_t stream) const {
    if (!blocked) return copy(layer, step, name, src, (size_t)rows * cols, stream);
    if (wants(layer, step, name)) LSH_CALL(lsh::block_rows(src, _dst.at(name), rows, cols, true, stream));
  }
  void copy(int layer, int step, const char* name, const void* src, size_t bytes,
            hipStream_t stream) const {
    if (!wants(layer, step, name)) return;
    if (hipMemcpyAsync(_dst.at(name), src, bytes, hipMemcpyDeviceToDevice, stream) != hipSuccess)
      throw std::runtime_error(std::string("tap copy failed: ") + name);
  }

 private:
  int _layer = -1, _step = -1;
  std::map<std::string, void*> _dst;
};

// The host's side of StepNotice.  A generation loop has to know after every step whether it goes on;
// a copy of the word and a stream synchronisation leave the device idle for 25 - 35 us (the
// wait, then the first launches of the next step).  Instead the loop enqueues the next step's
// first layers, ahead of which a launch publishes the word, and waits for the word alone: the
// device works meanwhile.  A step enqueued too far writes nothing that a finished run reads.
class HostNotice {
 public:
  HostNotice() {}
  HostNotice(const HostNotice&) = delete;
  HostNotice& operator=(const HostNotice&) = delete;
  ~HostNotice() {
    if (slot_) (void)hipHostFree(slot_);
  }
  lsh::StepNotice next(const int* word) {
    if (!slot_) {
      CHECK_GPU_ERROR(hipHostMalloc(reinterpret_cast<void**>(&slot_), sizeof(*slot_)));
      *slot_ = 0;
    }
    return lsh::StepNotice{word, slot_, ++tag_};
  }
  // the word of the last next(): a bounded wait on the slot, then on the stream
  int wait(hipStream_t stream) const {
    unsigned long long v = 0;
    auto there = [&] {
      v = __atomic_load_n(slot_, __ATOMIC_ACQUIRE);
      return (unsigned)(v >> 32) == tag_;
    };
    for (int i = 0; i < 20000; ++i) {
      if (there()) return (int)(unsigned)v;
      __builtin_ia32_pause();
    }
    for (int i = 0; i < 200000; ++i) {
      if (there()) return (int)(unsigned)v;
      std::this_thread::yield();
    }
    CHECK_GPU_ERROR(hipStreamSynchronize(stream));
    if (!there()) throw std::runtime_error("generation step: no word from the device");
    return (int)(unsigned)v;
  }

 private:
  unsigned long long* slot_ = nullptr;  // pinned
  unsigned tag_ = 0;
};

// Layers of the next step that a loop enqueues before it waits for the word.  A launch costs the host
// 2.5 us and the device 3.3 or more, so what is enqueued covers the hiccups of the host, of 100 us
// and more in some runs and absent in others; but a run that ends there has computed it for
// nothing.  So it grows by a layer with every step run, up to the whole step: what a run throws
// away is at most one layer per step that it made, which is what waiting at every step cost.
// Milliseconds with none / this many / all layers from the first step on, hosts with hiccups:
// 16 x 64 tokens through 6 layers, beam 4, 32.5 / 31.0 / 31.0; GPT-2-medium, 128 tokens after 45,
// 68.3 / 61.3 / 61; 16 sequences after 512, 99 / 88.5 / 91; without: 13.7 / 13.2 / 13.2 (one sentence of
// 21), 56.2 / 57.5 / 57.6, 85.5 / 87.7 / 88.  A translation that ends after 2 steps takes 0.65 / 0.68 /
// 0.79, a text that ends after 3 tokens 1.66 / 1.69 / 2.07.
inline int layers_ahead(int steps_run, int layers) { return steps_run < layers ? steps_run : layers; }

// HIP graphs of a generation step.  A step is a fixed sequence of launches whose arguments
// depend only on the shapes of the call and on the position of the step, so the sequence
// enqueued for one key is the sequence for every later call with that key -- as long as the
// process-wide route switches stand as they stood at the capture (route_epoch(); a change drops
// every graph held) and the body bakes in no pointer that a caller can replace.
//   first time a key is seen   the step runs eagerly (kernel attributes get set, nothing is kept)
//   second time                the step is captured from the stream, instantiated and launched
//   later                      one hipGraphLaunch
// At most kMaxGraphs executables are kept, the least recently launched one is destroyed first.
// A key whose capture or instantiation fails runs eagerly from then on.
// The body may only enqueue kernels and device-to-device copies on the stream: no memset nodes
// (they replay wrongly on this platform), no synchronisation, no host reads.
class StepGraphs {
 public:
  StepGraphs() {}
  StepGraphs(const StepGraphs&) = delete;
  StepGraphs& operator=(const StepGraphs&) = delete;
  ~StepGraphs() { clear(); }
  void clear() {
    for (auto& kv : execs_) (void)hipGraphExecDestroy(kv.second.exec);
    execs_.clear();
    lru_.clear();
    seen_.clear();
    eager_only_.clear();
  }
  int captured() const { return captured_; }
  long replayed() const { return replayed_; }
  size_t held() const { return execs_.size(); }
  int last_graph_nodes() const { return last_nodes_; }  // launches of the step captured last
  static constexpr size_t kMaxGraphs = 512;

  template <typename Body>
  void run(uint64_t key, hipStream_t stream, bool enabled, Body&& body) {
    if (!enabled) {
      body();
      return;
    }
    const unsigned long epoch = lsh::route_epoch();
    if (epoch != epoch_) {
      clear();
      epoch_ = epoch;
    }
    auto it = execs_.find(key);
    if (it != execs_.end()) {
      lru_.splice(lru_.begin(), lru_, it->second.pos);
      CHECK_GPU_ERROR(hipGraphLaunch(it->second.exec, stream));
      ++replayed_;
      return;
    }
    if (eager_only_.count(key) || seen_.insert(key).second) {  // failed before / first encounter
      body();
      return;
    }
    hipGraphExec_t exec = capture(stream, body);
    if (!exec) {  // the platform refused: the step still has to run
      eager_only_.insert(key);
      body();
      return;
    }
    while (execs_.size() >= kMaxGraphs) {
      const uint64_t old = lru_.back();
      lru_.pop_back();
      auto o = execs_.find(old);
      (void)hipGraphExecDestroy(o->second.exec);
      execs_.erase(o);
    }
    lru_.push_front(key);
    execs_[key] = Held{exec, lru_.begin()};
    ++captured_;
    CHECK_GPU_ERROR(hipGraphLaunch(exec, stream));
    ++replayed_;
  }

 private:
  struct Held {
    hipGraphExec_t exec;
    std::list<uint64_t>::iterator pos;
  };
  // Records the body; null when the capture or the instantiation fails (nothing has run then).
  // An exception of the body itself (a launcher that rejects its arguments) propagates.
  template <typename Body>
  hipGraphExec_t capture(hipStream_t stream, Body&& body) {
    if (hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    hipGraph_t graph = nullptr;
    try {
      body();
    } catch (...) {
      (void)hipStreamEndCapture(stream, &graph);
      if (graph) (void)hipGraphDestroy(graph);
      throw;
    }
    if (hipStreamEndCapture(stream, &graph) != hipSuccess || !graph) {
      (void)hipGetLastError();
      if (graph) (void)hipGraphDestroy(graph);
      return nullptr;
    }
    size_t nodes = 0;
    if (hipGraphGetNodes(graph, nullptr, &nodes) == hipSuccess) last_nodes_ = (int)nodes;
    hipGraphExec_t exec = nullptr;
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    return exec;
  }
  std::unordered_map<uint64_t, Held> execs_;
  std::list<uint64_t> lru_;  // most recently launched first
  std::unordered_set<uint64_t> seen_, eager_only_;
  unsigned long epoch_ = 0;
  int captured_ = 0, last_nodes_ = 0;
  long replayed_ = 0;
};

inline std::vector<__half> to_half(const std::vector<float>& v) {
  std::vector<__half> out(v.size());
  for (size_t i = 0; i < v.size(); ++i) out[i] = __float2half_rn(v[i]);
  return out;
}

// float vector -> fp16 on the device
inline DeviceBuffer<__half> upload_half(const std::vector<float>& v, hipStream_t s) {
  std::vector<__half> h = to_half(v);
  DeviceBuffer<__half> d(h.size());
  d.upload(h.data(), h.size(), s);
  CHECK_GPU_ERROR(hipStreamSynchronize(s));  // `h` dies at return
  return d;
}

// stored uint8 [rows(in), cols(out)] -> int8 [cols, rows] (K-contiguous for the GEMM)
inline DeviceBuffer<int8_t> upload_kernel(const std::vector<uint8_t>& w, int rows, int cols,
                                          bool transpose, hipStream_t s) {
  DeviceBuffer<uint8_t> raw(w.size());
  raw.upload(w.data(), w.size(), s);
  DeviceBuffer<int8_t> q(w.size());
  LSH_CALL(lsh::stored_u8_to_i8(raw.get(), q.get(), rows, cols, transpose, s));
  CHECK_GPU_ERROR(hipStreamSynchronize(s));
  return q;
}

// row-major int8 [n, k] -> blocked; the row-major copy is released
inline DeviceBuffer<int8_t> block_weight(DeviceBuffer<int8_t>& w, int n, int k, hipStream_t s) {
  DeviceBuffer<int8_t> b((size_t)(n + 15) / 16 * 16 * k);
  LSH_CALL(lsh::block_rows(w.get(), b.get(), n, k, false, s));
  CHECK_GPU_ERROR(hipStreamSynchronize(s));
  w = DeviceBuffer<int8_t>();
  return b;
}
inline DeviceBuffer<int8_t> unblock_weight(const DeviceBuffer<int8_t>& b, int n, int k, hipStream_t s) {
  DeviceBuffer<int8_t> w((size_t)n * k);
  LSH_CALL(lsh::block_rows(b.get(), w.get(), n, k, true, s));
  CHECK_GPU_ERROR(hipStreamSynchronize(s));
  return w;
}

// [n, k] row-major -> a blocked copy whose rows are padded with zeros to a multiple of 64
inline DeviceBuffer<int8_t> block_weight_padded(const DeviceBuffer<int8_t>& w, int n, int k, hipStream_t s) {
  const size_t bytes = (size_t)((n + 63) & ~63) * k;
  DeviceBuffer<int8_t> b(bytes);
  CHECK_GPU_ERROR(hipMemsetAsync(b.get(), 0, bytes, s));
  LSH_CALL(lsh::block_rows(w.get(), b.get(), n, k, false, s));
  CHECK_GPU_ERROR(hipStreamSynchronize(s));
  return b;
}

// The int32 sums of the out-projections that attention launches add to: three buffers of [rows, hidden]
// that take turns.  A launch adds to the current one and clears that of the launch behind it; a run
// clears all three before its first step.  A step's first turn follows from its index alone, as a
// graph replay needs.
class OutSumsRing {
 public:
  void alloc(size_t most) { _buf.alloc(4 * most); }
  void begin_run(size_t n, hipStream_t s) {
    _n = n;
    LSH_CALL(lsh::fill_i32(_buf.get(), 0, (int)(3 * n), s));
  }
  void begin_step(int launches_before) { _turn = launches_before % 3; }
  int32_t* sums() const { return _buf.get() + (size_t)_turn * _n; }
  int32_t* next_sums() const { return _buf.get() + (size_t)((_turn + 1) % 3) * _n; }
  // the second feed-forward product's, which every launch of a self attention clears
  int32_t* ffn_sums() const { return _buf.get() + 3 * _n; }
  void launched() { _turn = (_turn + 1) % 3; }

 private:
  DeviceBuffer<int32_t> _buf;
  size_t _n = 0;
  int _turn = 0;
};

// The products of a layer stack whose int8 matrices are all blocked (hidden and inner size
// multiples of 64) or all row-major.
struct LayerProducts {
  bool blocked = false;
  static bool can_block(int hidden, int inner, int dim_per_head) {
    return hidden % 64 == 0 && inner % 64 == 0 && dim_per_head % 16 == 0;
  }
  // Where a step's layer norms are made by the products that read them (LnStep).
  bool ln_in_product(int rows, int hidden) const { return blocked && lsh::ln_step_supported(rows, hidden); }
  // rows an activation matrix needs room for
  size_t rows(size_t n) const { return (n + 15) & ~(size_t)15; }
  DeviceBuffer<int8_t> weight(const std::vector<uint8_t>& w, int k, int n, hipStream_t s) const {
    DeviceBuffer<int8_t> q = upload_kernel(w, k, n, true, s);
    return blocked ? block_weight(q, n, k, s) : std::move(q);
  }
  void i8o(const int8_t* x, const int8_t* w, int8_t* out, int m, int n, int k, float alpha,
           hipStream_t s) const {
    LSH_CALL(blocked ? lsh::gemm_blk_i8o(x, w, out, m, n, k, alpha, s)
                     : lsh::gemm_i8_i8o(x, w, out, m, n, k, alpha, s));
  }
  void lut(const int8_t* x, const int8_t* w, int8_t* out, const int8_t* table, int m, int n, int k,
           float alpha, hipStream_t s, const lsh::LnStep* ln = nullptr) const {
    LSH_CALL(blocked ? lsh::gemm_blk_lut(x, w, out, table, m, n, k, alpha, s, ln)
                     : lsh::gemm_i8_lut_i8o(x, w, out, table, m, n, k, alpha, s));
  }
  // the product as sums of `cleared` where splitting K pays (one plane in any case), else planes of `out`
  int i32_sums(const int8_t* x, const int8_t* w, int32_t* out, int32_t* cleared, const int32_t** acc, int m,
               int n, int k, int max_planes, hipStream_t s) const {
    const int ranges = blocked && cleared ? lsh::gemm_blk_preferred_ksplit(m, n, k) : 1;
    *acc = ranges > 1 ? cleared : out;
    if (ranges <= 1) return i32o(x, w, out, m, n, k, max_planes, s);
    LSH_CALL(lsh::gemm_blk_i32_add(x, w, cleared, m, n, k, ranges, s));
    return 1;
  }
  // int32 accumulators in up to max_planes planes of [m, n]; returns their number
  int i32o(const int8_t* x, const int8_t* w, int32_t* out, int m, int n, int k, int max_planes,
           hipStream_t s) const {
    if (blocked) {
      const int planes = std::min(max_planes, lsh::gemm_blk_preferred_ksplit(m, n, k));
      LSH_CALL(lsh::gemm_blk_i32o(x, w, out, m, n, k, planes, s));
      return planes;
    }
    int planes = 1;
    LSH_CALL(lsh::gemm_i8_i32o_splitk(x, w, out, m, n, k,
                                      std::min(max_planes, lsh::gemm_i8_preferred_ksplit(m, n, k)),
                                      &planes, s));
    return planes;
  }
  void decself_qkv(const int8_t* x, const int8_t* w, const __half* bias, int8_t* q, int8_t* k_cache,
                   int8_t* v_cache, int rows, int hidden, int head_num, int max_step, int step,
                   float alpha, float dequant_scale, float quant_scale, hipStream_t s,
                   const lsh::LnStep* ln = nullptr) const {
    LSH_CALL(blocked ? lsh::gemm_blk_decself_qkv(x, w, bias, q, k_cache, v_cache, rows, hidden, hidden,
                                                 head_num, max_step, step, alpha, dequant_scale,
                                                 quant_scale, s, ln)
                     : lsh::gemm_i8_decself_qkv_i8o(x, w, bias, q, k_cache, v_cache, rows, hidden,
                                                    hidden, head_num, max_step, step, alpha,
                                                    dequant_scale, quant_scale, s));
  }
  void encdec_q(const int8_t* x, const int8_t* w, const __half* bias, __half* q, int rows, int hidden,
                int beam_size, int head_num, float alpha, float dequant_scale, hipStream_t s,
                const lsh::LnStep* ln = nullptr) const {
    LSH_CALL(blocked ? lsh::gemm_blk_encdec_q(x, w, bias, q, rows, hidden, hidden, beam_size, head_num,
                                              alpha, dequant_scale, s, ln)
                     : lsh::gemm_i8_encdec_q_f16(x, w, bias, q, rows, hidden, hidden, beam_size,
                                                 head_num, alpha, dequant_scale, s));
  }
};

}  // namespace hip
}  // namespace lightseq
