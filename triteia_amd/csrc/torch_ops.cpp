// The ops' ordinary case from Python to the C ABI in one native call: argument checks, output and scratch from torch's
// caching allocator, the current stream, the launches.  (The same steps through ctypes and torch's Python API cost 15 - 20 us
// a call, more than most decode-size kernels take on the GPU; here 4 - 6 us.)
//
// Every function returns None for whatever is not the ordinary case -- another device, type, layout or shape, a pair
// of sizes that the library refuses -- before any kernel of the library has been launched; the Python op then takes its
// own path, which checks the arguments one by one and raises the reference's error texts.  A launch that fails raises.
// Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/Event.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#define TORCH_CUDA_CPP_API TORCH_HIP_CPP_API   // (as the torch of this build names it, but for this header)
#include <ATen/cuda/tunable/Tunable.h>

#include <unordered_map>

#include "../../include/triteia_hip.h"

namespace {

using at::Tensor;

// A call's arguments, taken apart while the interpreter lock is held: what follows runs without it and sees no Python object.
// Tensors are exactly torch.Tensor or Parameter; a subclass may give every operation another meaning, which the Python
// path honours.  So may a transform's wrapper around a tensor, a dispatch mode and a trace: what they follow are torch's
// operations, and a kernel launched from here would leave its result in them as a constant.
struct Args {
  static constexpr int kMax = 8;
  int n;
  const Tensor* tensors[kMax] = {};
  bool nones[kMax] = {};
  double number = 0;        // a last argument that is neither a tensor nor None
  bool numeric = false;
  Args(PyObject* const* values, Py_ssize_t count) : n(count <= kMax ? (int)count : 0) {
    const bool traced = at::tracer::impl::is_dispatch_enabled();
    for (int i = 0; i < n; i++) {
      if (!traced && THPVariable_CheckExact(values[i]) && !at::isTensorSubclassLike(THPVariable_Unpack(values[i])))
        tensors[i] = &THPVariable_Unpack(values[i]);
      nones[i] = values[i] == Py_None;
    }
    if (n == 0 || nones[n - 1] || THPVariable_Check(values[n - 1])) return;
    number = PyFloat_AsDouble(values[n - 1]);
    numeric = !PyErr_Occurred();
    PyErr_Clear();
  }
  bool tensor(int i) const { return i < n && tensors[i] != nullptr; }
  const Tensor& operator[](int i) const { return *tensors[i]; }
  bool none(int i) const { return i < n && nones[i]; }
};

bool on(const Tensor& t, const Tensor& ref, at::ScalarType type, int64_t dim) {
  return t.scalar_type() == type && t.dim() == dim && t.device() == ref.device() && t.layout() == at::kStrided;
}
bool dense_on(const Tensor& t, const Tensor& ref, at::ScalarType type, int64_t dim) { return on(t, ref, type, dim) && t.is_contiguous(); }

// the current stream of x's device, and that device current for what follows
struct Place {
  c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
  int dev;
  c10::hip::HIPStreamMasqueradingAsCUDA stream;
  explicit Place(const Tensor& x)
      : guard(x.device()), dev(x.device().index()), stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index())) {}
  void* handle() const { return stream.stream(); }
};

Tensor scratch_bytes(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)((bytes + 255) / 256 * 256)}, like.options().dtype(at::kByte));
}

// A library call that comes first: true if it was launched, false if it was refused.
bool launched(int code) {
  TORCH_CHECK(code != TRITEIA_HIP_ERR_RUNTIME, "triteia_hip error ", code, ": ", triteia_hip_last_error());
  return code == TRITEIA_HIP_OK;
}
// A call behind others, whose arguments have been checked ahead of the first: there is no way back.
void must_launch(int code) { TORCH_CHECK(code == TRITEIA_HIP_OK, "triteia_hip error ", code, ": ", triteia_hip_last_error()); }

// sizes that fit the library's ints, on a GPU
bool sizes_ok(std::initializer_list<int64_t> sizes) {
  for (int64_t s : sizes)
    if (s <= 0 || s > 0x7fffffff) return false;
  return true;
}

// stacked packed matrices: q [n, k/32, 2m], meta [n, m, k/16], s [n, 1, m]
bool packed_ok(const Tensor& q, const Tensor& meta, const Tensor& s, const Tensor& x, int64_t n, int64_t k, int64_t m) {
  return dense_on(q, x, at::kInt, 3) && dense_on(meta, x, at::kShort, 3) && dense_on(s, x, at::kHalf, 3) && m % 128 == 0 && k % 64 == 0 &&
         sizes_ok({n, k, m}) && q.size(0) == n && q.size(1) == k / 32 && q.size(2) == 2 * m && meta.size(0) == n && meta.size(1) == m &&
         meta.size(2) == k / 16 && s.size(0) == n && s.size(1) == 1 && s.size(2) == m;
}
// (what the routed product takes in one call, see triteia_hip_sbmm_2_4_routed_own)
constexpr int64_t kMaxRoutedDeltas = 8192;

// (under autocast the base product has autocast's type, whatever its inputs': another one than x's is refused by the Python path)
bool base_ok(const Args& a, int i, const Tensor& x, int64_t k, int64_t m) {
  return a.none(i) || (a.tensor(i) && on(a[i], x, x.scalar_type(), 2) && a[i].size(0) == m && a[i].size(1) == k &&
                       !(at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != x.scalar_type()));
}
// (a view that starts inside 16 bytes; a copy made by contiguous() does not)
bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// x [tokens, k] times the layer's dense weight, which base_ok has let pass: what the kernels add to.  A few hundred fp16 rows
// run on the library's own kernel, everything else -- more tokens, other types, rows that are not aligned, a product that
// autograd records, a process that has torch tune its products (torch.cuda.tunable) -- on torch's.
Tensor base_product(const Tensor& x, const Tensor& weight, const Place& at_) {
  const int64_t tokens = x.size(0), k = x.size(1), m = weight.size(0);
  const bool recorded = (at::GradMode::is_enabled() && (x.requires_grad() || weight.requires_grad())) || x._fw_grad(0).defined() || weight._fw_grad(0).defined();
  if (x.scalar_type() == at::kHalf && !recorded && sizes_ok({tokens, k, m}) && triteia_hip_dense_ok(tokens, m, k) &&
      !at::cuda::tunable::getTuningContext()->IsTunableOpEnabled() && x.is_contiguous() &&
      weight.stride(1) == 1 && weight.stride(0) >= k && weight.stride(0) % 8 == 0 && aligned(x) && aligned(weight) && !x.is_neg() && !weight.is_neg()) {
    Tensor y = at::empty({tokens, m}, x.options());
    const size_t bytes = triteia_hip_dense_scratch_bytes(tokens, m, k);
    const Tensor scratch = bytes ? scratch_bytes(bytes, x) : Tensor();
    must_launch(triteia_hip_dense(x.data_ptr(), k, weight.data_ptr(), weight.stride(0), y.data_ptr(), tokens, m, k, bytes ? scratch.data_ptr() : nullptr,
                                  bytes, at_.dev, at_.handle()));
    return y;
  }
  Tensor y = at::matmul(x, weight.t());
  TORCH_CHECK(y.scalar_type() == x.scalar_type() && y.is_contiguous(), "the base product is ", y.scalar_type(), ", expected a contiguous ",
              x.scalar_type());
  return y;
}

// matmul(qweight, x, meta, s): ops.matmul_4bit_2_4
Tensor matmul(const Args& a) {
  if (a.n != 4 || !a.tensor(0) || !a.tensor(1) || !a.tensor(2) || !a.tensor(3)) return {};
  const Tensor &q = a[0], &x = a[1], &meta = a[2], &s = a[3];
  if (!x.is_cuda() || x.dim() < 1 || x.scalar_type() != at::kHalf || s.dim() != 2) return {};
  const int64_t k = x.size(-1), m = s.size(1), rows = k > 0 ? x.numel() / k : 0;
  if (!sizes_ok({k, m, rows}) || m % 128 != 0 || k % 64 != 0 || s.size(0) != 1 || !dense_on(q, x, at::kInt, 2) || !dense_on(meta, x, at::kShort, 2) ||
      !dense_on(s, x, at::kHalf, 2) || q.size(0) != k / 32 || q.size(1) != 2 * m || meta.size(0) != m || meta.size(1) != k / 16)
    return {};
  const Place at_(x);
  const Tensor xc = x.is_contiguous() ? x : x.contiguous();
  c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = m;
  Tensor y = at::empty(shape, x.options());
  const size_t split = triteia_hip_bmm_scratch_bytes(m, 1, rows, k);
  const Tensor scratch = split ? scratch_bytes(split, x) : Tensor();
  return launched(triteia_hip_bmm_2_4_tokens_scratch(xc.data_ptr(), q.data_ptr(), meta.data_ptr(), y.data_ptr(), s.data_ptr(), m, 1, rows, k,
                                                     split ? scratch.data_ptr() : nullptr, split, at_.dev, at_.handle()))
             ? y
             : Tensor();
}

// bmm(qweights, xs, metas, ss): ops.bmm_4bit_2_4
Tensor bmm(const Args& a) {
  if (a.n != 4 || !a.tensor(0) || !a.tensor(1) || !a.tensor(2) || !a.tensor(3)) return {};
  const Tensor &q = a[0], &x = a[1], &meta = a[2], &s = a[3];
  if (!x.is_cuda() || x.dim() != 3 || x.scalar_type() != at::kHalf || s.dim() != 3) return {};
  const int64_t n = x.size(0), tokens = x.size(1), k = x.size(2), m = s.size(2);
  if (!sizes_ok({tokens}) || !packed_ok(q, meta, s, x, n, k, m)) return {};
  const Place at_(x);
  const Tensor xc = x.is_contiguous() ? x : x.contiguous();
  Tensor y = at::empty({n, tokens, m}, x.options());
  const size_t split = triteia_hip_bmm_scratch_bytes(m, n, tokens, k);
  const Tensor scratch = split ? scratch_bytes(split, x) : Tensor();
  return launched(triteia_hip_bmm_2_4_tokens_scratch(xc.data_ptr(), q.data_ptr(), meta.data_ptr(), y.data_ptr(), s.data_ptr(), m, n, tokens, k,
                                                     split ? scratch.data_ptr() : nullptr, split, at_.dev, at_.handle()))
             ? y
             : Tensor();
}

// The routed product of x [tokens, k], added to y (accumulate = 1) or stored with zeros in the rows without a delta
// (2: y need not be initialised).  The library's answer.
int routed(const Tensor& x, const Tensor& q, const Tensor& meta, const Tensor& s, const Tensor& indices, Tensor& y, int offset,
            int accumulate, const Place& at_) {
  const int64_t tokens = x.size(0), k = x.size(1), m = y.size(1), n = q.size(0);
  Tensor ws;
  size_t bytes = 0;
  if (!triteia_hip_routed_in_kernel(tokens, n, m, k)) {     // (a batch that is routed inside the kernel needs no plan)
    bytes = triteia_hip_sbmm_routed_workspace_bytes(tokens, n);
    ws = scratch_bytes(bytes, x);
  }
  return triteia_hip_sbmm_2_4_routed_own(x.data_ptr(), q.data_ptr(), meta.data_ptr(), y.data_ptr(), s.data_ptr(), indices.data_ptr(), offset, n,
                                         m, tokens, k, bytes ? ws.data_ptr() : nullptr, bytes, accumulate, at_.dev, at_.handle());
}

// sbmm(qweights, xs, metas, ss, indices, base or None): ops.sbmm_4bit_2_4_native
Tensor sbmm(const Args& a) {
  if (a.n != 6) return {};
  for (int i = 0; i < 5; i++)
    if (!a.tensor(i)) return {};
  const Tensor &q = a[0], &x = a[1], &meta = a[2], &s = a[3], &indices = a[4];
  if (!x.is_cuda() || x.dim() != 2 || x.scalar_type() != at::kHalf || s.dim() != 3) return {};
  const int64_t tokens = x.size(0), k = x.size(1), m = s.size(2);
  if (!sizes_ok({tokens}) || q.size(0) > kMaxRoutedDeltas || !packed_ok(q, meta, s, x, q.size(0), k, m) || !base_ok(a, 5, x, k, m)) return {};
  if (indices.device() != x.device() || indices.dim() != 1 || indices.size(0) != tokens || !indices.is_contiguous() ||
      !at::isIntegralType(indices.scalar_type(), false))
    return {};
  const Place at_(x);
  const Tensor xc = x.is_contiguous() ? x : x.contiguous();
  const Tensor idx = indices.scalar_type() == at::kInt ? indices : indices.to(at::kInt);
  Tensor y;
  if (a.none(5)) {
    y = at::empty({tokens, m}, x.options());
    return launched(routed(xc, q, meta, s, idx, y, 0, 2, at_)) ? y : Tensor();
  }
  y = base_product(xc, a[5], at_);
  must_launch(routed(xc, q, meta, s, idx, y, 0, 1, at_));
  return y;
}

// (the expand's grid has a row of workgroups per 256 columns)
constexpr int64_t kMaxLoraColumns = 65535 * 256;
bool lora_ok(const Tensor& A, const Tensor& B, const Tensor& x, const Tensor& indices) {
  return x.is_cuda() && x.dim() == 2 && (x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16) &&
         dense_on(A, x, x.scalar_type(), 3) && dense_on(B, x, x.scalar_type(), 3) && indices.device() == x.device() && indices.dim() == 1 &&
         indices.is_contiguous() && (indices.scalar_type() == at::kInt || indices.scalar_type() == at::kLong) &&
         sizes_ok({x.size(0), x.size(1), A.size(0), A.size(2), B.size(2)}) && indices.size(0) == x.size(0) && A.size(1) == x.size(1) &&
         B.size(0) == A.size(0) && B.size(1) == A.size(2) && B.size(2) % 8 == 0 && B.size(2) <= kMaxLoraColumns && aligned(A) &&
         aligned(B) && (!x.is_contiguous() || aligned(x));
}
size_t lora_bytes(const Tensor& A, const Tensor& x) { return triteia_hip_lora_scratch_bytes(x.size(0), A.size(0), A.size(1), A.size(2)); }
int lora_shrink(const Tensor& x, const Tensor& A, const Tensor& indices, const Tensor& scratch, bool accumulate, int dev, void* stream) {
  return triteia_hip_lora_shrink(x.data_ptr(), x.size(1), A.data_ptr(), indices.data_ptr(), indices.scalar_type() == at::kLong, x.size(0), A.size(0),
                                 A.size(1), A.size(2), accumulate, scratch.data_ptr(), scratch.numel(), x.scalar_type() == at::kBFloat16, dev,
                                 stream);
}
int lora_expand(const Tensor& y, const Tensor& A, const Tensor& B, const Tensor& scratch, double scale, bool accumulate, int dev, void* stream) {
  return triteia_hip_lora_expand(y.data_ptr(), y.size(1), B.data_ptr(), scratch.data_ptr(), y.size(0), B.size(0), A.size(1), B.size(1), y.size(1),
                                 (float)scale, accumulate, y.scalar_type() == at::kBFloat16, dev, stream);
}

// (one launch, where triteia_hip_lora_ok says that it pays)
bool lora_at_once(const Tensor& A, const Tensor& B, const Tensor& x) {
  return triteia_hip_lora_ok(x.size(0), A.size(0), A.size(1), A.size(2), B.size(2));
}
int lora_fused(const Tensor& y, const Tensor& x, const Tensor& A, const Tensor& B, const Tensor& indices, double scale, bool accumulate, int dev, void* stream) {
  return triteia_hip_lora(y.data_ptr(), y.size(1), x.data_ptr(), x.size(1), A.data_ptr(), B.data_ptr(), indices.data_ptr(),
                          indices.scalar_type() == at::kLong, x.size(0), A.size(0), A.size(1), A.size(2), B.size(2), (float)scale, accumulate,
                          x.scalar_type() == at::kBFloat16, dev, stream);
}

// lora(weights_A, weights_B, x, indices, base or None, scale): ops.lora_bgmv / lora_sgmv / lora_sgmv_routed
Tensor lora(const Args& a) {
  if (a.n != 6 || !a.tensor(0) || !a.tensor(1) || !a.tensor(2) || !a.tensor(3)) return {};
  const Tensor &A = a[0], &B = a[1], &x = a[2], &indices = a[3];
  if (!a.numeric || !lora_ok(A, B, x, indices) || !base_ok(a, 4, x, x.size(1), B.size(2))) return {};
  const size_t bytes = lora_bytes(A, x);
  if (bytes == 0) return {};
  const Place at_(x);
  const Tensor xc = x.is_contiguous() ? x : x.contiguous();
  const bool base = !a.none(4);
  if (lora_at_once(A, B, x)) {
    Tensor y = base ? base_product(xc, a[4], at_) : at::empty({x.size(0), B.size(2)}, x.options());
    must_launch(lora_fused(y, xc, A, B, indices, a.number, base, at_.dev, at_.handle()));
    return y;
  }
  const Tensor scratch = scratch_bytes(bytes, x);
  if (!launched(lora_shrink(xc, A, indices, scratch, base, at_.dev, at_.handle()))) return {};
  // (without a base weight every row is written by the expand: tokens without an adapter get zeros)
  Tensor y = base ? base_product(xc, a[4], at_) : at::empty({x.size(0), B.size(2)}, x.options());
  must_launch(lora_expand(y, A, B, scratch, a.number, base, at_.dev, at_.handle()));
  return y;
}

// A second stream beside the call's own (default priority, one per thread and device, made at first use).  The call's
// stream waits for its work also where a later step throws: the buffers then go back to that stream's pool.
class Beside {
 public:
  explicit Beside(const Place& at_) : own_(at_.stream.unwrap()), side_(stream(at_.dev).unwrap()), handle_(stream(at_.dev).stream()) { follow(); }
  ~Beside() {
    if (!joined_) {
      try {
        wait(side_, own_);
      } catch (...) {           // (the exception on its way out is the one to report)
      }
    }
  }
  Beside(const Beside&) = delete;
  Beside& operator=(const Beside&) = delete;
  void follow() { wait(own_, side_); }      // what comes next on the second stream sees what the call's stream has so far
  void join() {
    wait(side_, own_);
    joined_ = true;
  }
  void* handle() const { return handle_; }

 private:
  static void wait(const c10::Stream& first, const c10::Stream& second) {
    c10::Event event(first.device_type());
    event.record(first);
    event.block(second);
  }
  static c10::hip::HIPStreamMasqueradingAsCUDA stream(c10::DeviceIndex dev) {
    static thread_local std::unordered_map<int, c10::hip::HIPStreamMasqueradingAsCUDA> streams;
    auto it = streams.find(dev);
    if (it == streams.end()) it = streams.emplace(dev, c10::hip::getStreamFromPoolMasqueradingAsCUDA(false, dev)).first;
    return it->second;
  }
  c10::Stream own_, side_;
  void* handle_;
  bool joined_ = false;
};

// Whether ldmm runs its LoRA pair on a second stream, the shrink beside the base product and the expand beside the deltas
// (their rows of the output differ).  The fork and the joins hold a call up by about 60 us, which prompts hide and smaller
// batches do not.  One stream -> two, a call among others, 4 - 32 deltas, 4 or 32 adapters of rank 16 or 64:
//   4096 x 4096 with 2048 / 4096 tokens 126-175 -> 120-160 / 180-261 -> 172-247 us; 4096 x 11008 with 2048 / 4096
//   247-386 -> 227-378 / 546-718 -> 515-704; 11008 x 4096 with 4096 400-587 -> 368-558; in 198 such shapes 5 % less on average,
//   8 of them more than 2 % longer.
// Below either bound: 4096 x 4096 with 768 tokens 66-114 -> 76-115, 1024 x 1024 with 4096 59-72 -> 99-129, 8192 x 13824 with
// 1024 307-534 -> 302-541.  In a captured graph the fork costs more than it hides at every size (11008 x 4096, 32 + 32
// models, 1024 / 4096 tokens of rank 16: 275 -> 300 / 546 -> 576).
bool lora_hides(int64_t tokens, int64_t k, int64_t m) { return tokens >= 2048 && tokens * k >= (int64_t(1) << 35) / m; }
bool captured() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// ldmm(indices, x, LwA, LwB, DeltaW, metas, ss, base or None): ops.ldmm.
Tensor ldmm(const Args& a) {
  if (a.n != 8) return {};
  for (int i = 0; i < 7; i++)
    if (!a.tensor(i)) return {};
  const Tensor &indices = a[0], &x = a[1], &A = a[2], &B = a[3], &q = a[4], &meta = a[5], &s = a[6];
  if (x.scalar_type() != at::kHalf || !lora_ok(A, B, x, indices) || s.dim() != 3) return {};
  const int64_t k = x.size(1), m = B.size(2);
  const size_t bytes = lora_bytes(A, x);
  if (bytes == 0 || q.size(0) > kMaxRoutedDeltas || !packed_ok(q, meta, s, x, q.size(0), k, m) || !base_ok(a, 7, x, k, m)) return {};
  const Place at_(x);
  const Tensor xc = x.is_contiguous() ? x : x.contiguous();
  const Tensor idx = indices.scalar_type() == at::kInt ? indices : indices.to(at::kInt);
  const bool base = !a.none(7);
  const bool large = base && lora_hides(x.size(0), k, m);      // (the pair on either one stream or two: the same bits in a graph)
  if (!large && lora_at_once(A, B, x)) {
    // (without a base weight the LoRA launch stores the adapters' rows and zeros in all others, the deltas' among them)
    Tensor y = base ? base_product(xc, a[7], at_) : at::empty({x.size(0), m}, x.options());
    must_launch(lora_fused(y, xc, A, B, indices, 1.0, base, at_.dev, at_.handle()));
    must_launch(routed(xc, q, meta, s, idx, y, A.size(0), 1, at_));
    return y;
  }
  const Tensor scratch = scratch_bytes(bytes, x);
  if (large && !captured()) {
    Tensor y;                  // (like the other buffers ahead of the stream: freed only after it has been joined)
    Beside side(at_);
    if (!launched(lora_shrink(xc, A, indices, scratch, true, at_.dev, side.handle()))) return {};
    y = base_product(xc, a[7], at_);
    side.follow();
    must_launch(lora_expand(y, A, B, scratch, 1.0, true, at_.dev, side.handle()));
    must_launch(routed(xc, q, meta, s, idx, y, A.size(0), 1, at_));
    side.join();
    return y;
  }
  if (!launched(lora_shrink(xc, A, indices, scratch, base, at_.dev, at_.handle()))) return {};
  // (without a base weight the expand stores the adapters' rows and zeros in all others, the deltas' among them)
  Tensor y = base ? base_product(xc, a[7], at_) : at::empty({x.size(0), m}, x.options());
  must_launch(lora_expand(y, A, B, scratch, 1.0, base, at_.dev, at_.handle()));
  must_launch(routed(xc, q, meta, s, idx, y, A.size(0), 1, at_));
  return y;
}

PyObject* wrap(Tensor&& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(t));
}

// Other Python threads run while an op allocates, calls torch and launches (the caller holds references to its arguments).
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// torch's own translation of exceptions: an allocation that fails raises torch.OutOfMemoryError, as from Python
template <Tensor (*F)(const Args&)>
PyObject* call(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args a(v, n);
  Tensor y;
  {
    const WithoutGil released;
    y = F(a);
  }
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The packed tensors of a [k, m] weight and a scale per column: (qweight, meta, meta_raw).
bool packed(const Tensor& w, const Tensor& s, Tensor (&out)[3]) {
  const int64_t k = w.size(0), m = w.size(1);
  if (!sizes_ok({k, m}) || k % 32 != 0 || m % 64 != 0 || s.numel() != m ||
      (reinterpret_cast<uintptr_t>(w.data_ptr()) | reinterpret_cast<uintptr_t>(s.data_ptr())) % 4 != 0)
    return false;
  const Place at_(w);
  out[0] = at::empty({k / 32, 2 * m}, w.options().dtype(at::kInt));
  out[1] = at::empty({m, k / 16}, w.options().dtype(at::kShort));
  out[2] = at::empty({m, k / 16}, w.options().dtype(at::kShort));
  return launched(triteia_hip_pack_2_4(w.data_ptr(), s.data_ptr(), out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), k, m, at_.dev,
                                       at_.handle()));
}
// pack(weight, scales): the three of ops.utils.sparsity.prune_pack_2_4, or None
PyObject* pack(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args a(v, n);
  Tensor out[3];
  bool done = a.n == 2 && a.tensor(0) && a.tensor(1) && a[0].is_cuda() && dense_on(a[0], a[0], at::kHalf, 2) && dense_on(a[1], a[0], at::kHalf, 2);
  if (done) {
    const WithoutGil released;
    done = packed(a[0], a[1], out);
  }
  if (!done) Py_RETURN_NONE;
  return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(out[0])), THPVariable_Wrap(std::move(out[1])), THPVariable_Wrap(std::move(out[2])));
  END_HANDLE_TH_ERRORS
}
// sparse(weight, scale): the five of ops.utils.generator.fp16_to_sparse for tensors that are on the current GPU already, or None.  In one
// call: the moves, views and checks in Python cost as much as the packing of a small weight (768 x 2176 9.1 -> 7.4 us a call).
PyObject* sparse(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args a(v, n);
  Tensor out[3], scales;
  bool done = a.n == 2 && a.tensor(0) && a.tensor(1) && !at::impl::torch_function_mode_enabled() && a[0].is_cuda() &&
              a[0].device().index() == c10::hip::current_device() && dense_on(a[0], a[0], at::kHalf, 2) &&
              dense_on(a[1], a[0], at::kHalf, a[1].dim()) && !a[1].requires_grad();
  if (done) {
    const WithoutGil released;
    done = packed(a[0], a[1], out);
    if (done) scales = a[1].reshape({1, a[0].size(1)});
  }
  if (!done) Py_RETURN_NONE;
  Py_INCREF(v[0]);
  return Py_BuildValue("(NNNNN)", v[0], THPVariable_Wrap(std::move(out[0])), THPVariable_Wrap(std::move(scales)), THPVariable_Wrap(std::move(out[1])),
                       THPVariable_Wrap(std::move(out[2])));
  END_HANDLE_TH_ERRORS
}

#define METHOD(NAME_, FN_) {NAME_, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(FN_)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD("matmul", (call<matmul>)), METHOD("bmm", (call<bmm>)), METHOD("sbmm", (call<sbmm>)), METHOD("lora", (call<lora>)), METHOD("ldmm", (call<ldmm>)),
                         METHOD("pack", pack), METHOD("sparse", sparse), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "triteia_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_triteia_torch(void) { return PyModule_Create(&module); }
