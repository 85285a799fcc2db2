// Host side of the small per-token operators: operand checks, output tensors, the launch through the C ABI and the
// autograd node of a loss, in one native call each.
//
// A call of such an operator takes the GPU 5 to 20 us and took the host 18 to 30 us in Python, and a Python backward
// some 40 us more than a native one: the engine's device thread has to get the interpreter lock from the thread that
// waits for it.  Per call: policy_loss 18 -> 9 us, group_advantage 28 -> 13, reverse_scan 24 -> 7; whole passes
// (advantage, loss, backward), with the sums that the launch sends to the host itself: GRPO + PPO on 128 x 1024 165 -> 94 us,
// sampler correction + GSPO on 65536 tokens 254 -> 166, correction + PPO on 8.4 M 402 -> 352, GAE + value loss on 2.1 M 176 -> 115.
//
// Nothing here computes: the arithmetic is behind axon_amd.h.  The functions take what the Python wrappers of the same
// names (axon_amd/_ops.py) have normalised, and run without the interpreter lock, as a call through ctypes does.
#include <ATen/ATen.h>
#include <hip/hip_runtime_api.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/axon_amd.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

PyObject* g_error = nullptr;  // axon_amd._lib.AxonAmdError
struct AxonError : torch::PyTorchError {  // the autograd engine hands it on as what it is
  using PyTorchError::PyTorchError;
  PyObject* python_type() override { return g_error; }
};

void check(int rc, const char* what) {
  if (rc != 0) throw AxonError(std::string(what) + ": " + axon_amd_error_string(rc) + " (code " + std::to_string(rc) + ")");
}

// The HIP path only.  (The Python wrappers look at the first operand of every other function.)
void require_device(const Tensor& t, const char* what) {
  if (!t.is_cuda())
    throw AxonError(std::string(what) + ": tensor is on " + t.device().str() +
                    "; the axon_amd path runs on MI355X only and has no CPU fallback");
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }

// The kernels move four values per access: a view that starts off a 16-byte boundary is copied.
Tensor on_16_bytes(Tensor t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone(); }

// fp32, contiguous, aligned, outside the graph; the usual operand passes through untouched.
Tensor f32(const Tensor& x) {
  Tensor t = x.requires_grad() ? x.detach() : x;
  if (t.scalar_type() != at::kFloat || !t.is_contiguous()) t = t.to(at::kFloat).contiguous();
  return on_16_bytes(std::move(t));
}
Tensor f32(const OptTensor& x) { return x ? f32(*x) : Tensor(); }

// A response mask: fp32 and int64 are read natively.
std::pair<Tensor, int> mask_arg(const Tensor& x) {
  Tensor t = x.requires_grad() ? x.detach() : x;
  if (!t.is_contiguous()) t = t.contiguous();
  if (t.scalar_type() == at::kLong) return {on_16_bytes(std::move(t)), 1};
  if (t.scalar_type() != at::kFloat) t = t.to(at::kFloat);
  return {on_16_bytes(std::move(t)), 0};
}

// The kernels index every operand with the same token (or row) index.
void same_len(const char* what, const char* name, int64_t n, const Tensor& t) {
  if (t.numel() != n)
    throw py::value_error(std::string(what) + ": " + name + " has " + std::to_string(t.numel()) + " elements, expected " +
                          std::to_string(n));
}
void same_len(const char* what, const char* name, int64_t n, const OptTensor& t) {
  if (t) same_len(what, name, n, *t);
}

at::TensorOptions opts(const Tensor& like, at::ScalarType dtype = at::kFloat) {
  return at::TensorOptions().dtype(dtype).device(like.device());
}

// See _ops._acc8.
Tensor acc8(int64_t n_slots, const Tensor& like, const OptTensor& acc) {
  Tensor a = acc ? *acc : at::empty({8}, opts(like));
  if (n_slots == 0) return a.zero_();
  return capturing() ? a.fill_(std::numeric_limits<float>::quiet_NaN()) : a;
}

struct Rows {  // _ops.Rows, its offsets checked to be on the device
  int64_t n_rows, n_slots, uniform_len;
  OptTensor cu;
  std::vector<int64_t> shape;
  const int32_t* offsets() const { return cu ? cu->data_ptr<int32_t>() : nullptr; }
};
typedef std::tuple<int64_t, int64_t, int64_t, OptTensor, std::vector<int64_t>> RowsTuple;
Rows rows_of(const RowsTuple& t) {
  Rows r{std::get<0>(t), std::get<1>(t), std::get<2>(t), std::get<3>(t), std::get<4>(t)};
  if (r.cu && !r.cu->is_cuda())
    throw AxonError("cu_seqlens is on " + r.cu->device().str() +
                    ": the row offsets must live on the GPU (rows_of puts them on the device of the tensor it is given)");
  return r;
}

// The sums of a loss on their way to the host (axon_policy_loss_post): `also`, a tensor that earlier work of the stream has
// written, and the loss's eight sums behind it.
// One launch writes to a slot of pinned memory at a time; a slot goes back once its words have arrived.  One that nobody
// waits for any more (its loss raised behind the launch) is set aside until they have, which the next taker finds out: to wait
// in a destructor would hold the interpreter lock for the rest of the queue.  The slots, one kilobyte each, are as many as
// posts were ever under way together and live until the process ends.
struct Slot {
  uint32_t* host;
  uint32_t* device;
  uint32_t seq;
  bool arrived() const { return __atomic_load_n(host, __ATOMIC_ACQUIRE) == seq; }
};
class Slots {
 public:
  static constexpr int kWords = 16 + AXON_MAIL_MAX_WORDS + 8, kBytes = 1024, kPerBlock = 64;
  static_assert(kWords * 4 <= kBytes, "");
  static Slots& get() {
    static auto* const slots = new Slots;
    return *slots;
  }
  Slot take() {
    const std::lock_guard<std::mutex> lock(mutex_);
    const auto back = std::partition(aside_.begin(), aside_.end(), [](const Slot& s) { return !s.arrived(); });
    free_.insert(free_.end(), back, aside_.end());
    aside_.erase(back, aside_.end());
    if (free_.empty()) {
      void *host = nullptr, *device = nullptr;
      if (hipHostMalloc(&host, kBytes * kPerBlock, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) !=
              hipSuccess ||
          hipHostGetDevicePointer(&device, host, 0) != hipSuccess)
        throw AxonError("no pinned host memory for the sums of a loss");
      std::memset(host, 0, kBytes * kPerBlock);
      for (int i = 0; i < kPerBlock; ++i)
        free_.push_back(Slot{static_cast<uint32_t*>(host) + i * (kBytes / 4), static_cast<uint32_t*>(device) + i * (kBytes / 4), 0});
      made_ += kPerBlock;
    }
    Slot s = free_.back();
    free_.pop_back();
    ++s.seq;
    return s;
  }
  void give(const Slot& s) {
    const std::lock_guard<std::mutex> lock(mutex_);
    free_.push_back(s);
  }
  void set_aside(const Slot& s) {
    const std::lock_guard<std::mutex> lock(mutex_);
    aside_.push_back(s);
  }
  int made() {
    const std::lock_guard<std::mutex> lock(mutex_);
    return made_;
  }

 private:
  std::mutex mutex_;
  std::vector<Slot> free_, aside_;
  int made_ = 0;
};

class Post {
 public:
  explicit Post(OptTensor also) : also_(std::move(also)) {
    if (!also_) return;  // the launch reads nbytes() / 4 words from data_ptr() on
    require_device(*also_, "the words in front of a loss's sums");
    if (!also_->is_contiguous() || also_->nbytes() % 4 != 0 || also_->nbytes() > 4 * AXON_MAIL_MAX_WORDS)
      throw AxonError("the words in front of a loss's sums must be a contiguous tensor of whole words, at most " +
                      std::to_string(AXON_MAIL_MAX_WORDS) + "; got " + std::to_string(also_->nbytes()) + " bytes");
  }
  ~Post() {  // never waited for
    if (!sent_) return;
    try {
      Slots::get().set_aside(slot_);
    } catch (...) {  // no memory for the list: the slot is not used again
    }
  }
  const void* also() const { return also_ ? also_->data_ptr() : nullptr; }
  int64_t n_also() const { return also_ ? (int64_t)also_->nbytes() / 4 : 0; }
  const Slot& send(void* stream) {
    if (sent_) throw AxonError("these sums are on their way already");
    slot_ = Slots::get().take();
    stream_ = (hipStream_t)stream;
    return slot_;
  }
  void sent(int rc) {  // a refused launch writes nothing
    if (rc == 0) sent_ = true;
    else Slots::get().give(slot_);
  }
  bool is_sent() const { return sent_; }
  // The loss's eight sums.
  std::vector<double> sums() {
    arrive();
    float v[8];
    std::memcpy(v, slot_.host + 16 + n_also(), sizeof v);
    Slots::get().give(slot_);
    return {v, v + 8};
  }
  // All words as an fp32 tensor on the host.
  Tensor wait() {
    arrive();
    const int64_t words = n_also() + 8;
    Tensor out = at::empty({words}, at::TensorOptions().dtype(at::kFloat));
    std::memcpy(out.data_ptr(), slot_.host + 16, words * 4);
    Slots::get().give(slot_);
    return out;
  }

 private:
  // Spins while the words can be expected at once, then leaves the waiting to the runtime; the stream's end or its error
  // ends it in any case.
  void arrive() {
    if (!sent_) throw AxonError("no sums are on their way");
    sent_ = false;
    const auto start = std::chrono::steady_clock::now();
    for (int n = 1; !slot_.arrived(); ++n) {
      if (n % 1024) {
        __builtin_ia32_pause();
        continue;
      }
      if (std::chrono::steady_clock::now() - start < std::chrono::milliseconds(2)) continue;
      const hipError_t err = hipStreamSynchronize(stream_);
      if (err == hipSuccess && slot_.arrived()) break;
      // the slot is not used again: the device may be in any state
      throw AxonError(std::string("the sums of a loss did not arrive: ") + hipGetErrorString(err));
    }
  }

  OptTensor also_;
  Slot slot_{};
  hipStream_t stream_ = nullptr;
  bool sent_ = false;
};

std::tuple<Tensor, Tensor> policy_loss(int kind, const Tensor& log_probs, const Tensor& old_log_probs,
                                       const Tensor& advantages, const Tensor& mask, const OptTensor& is_weights,
                                       const RowsTuple& rows_tuple, int token_reduce, int batch_reduce,
                                       const OptTensor& per_row_count, const OptTensor& program_tokens,
                                       const OptTensor& program_steps, const OptTensor& valid, double ratio_lo,
                                       double ratio_hi, double clip_c, const OptTensor& acc_place, double loss_scale,
                                       bool one_pass, const Tensor& ws, Post* post) {
  const Rows rows = rows_of(rows_tuple);
  const int64_t n = rows.n_slots;
  same_len("policy_loss", "log_probs", n, log_probs);
  same_len("policy_loss", "old_log_probs", n, old_log_probs);
  same_len("policy_loss", "advantages", n, advantages);
  same_len("policy_loss", "mask", n, mask);
  same_len("policy_loss", "is_weights", n, is_weights);
  const Tensor lp = f32(log_probs), old = f32(old_log_probs), adv = f32(advantages), isw = f32(is_weights);
  const auto mk = mask_arg(mask);
  Tensor grad = at::empty(rows.shape, opts(lp)), acc = acc8(n, lp, acc_place);
  const float *lp_p = (const float*)ptr(lp), *old_p = (const float*)ptr(old), *adv_p = (const float*)ptr(adv),
              *isw_p = (const float*)ptr(isw);
  float *grad_p = grad.data_ptr<float>(), *acc_p = acc.data_ptr<float>(), *ws_p = ws.data_ptr<float>();
  const double *prtc_p = (const double*)ptr(per_row_count), *npt_p = (const double*)ptr(program_tokens),
               *nps_p = (const double*)ptr(program_steps), *valid_p = (const double*)ptr(valid);
  const float lo = (float)ratio_lo, hi = (float)ratio_hi, clip = (float)clip_c, scale = (float)loss_scale;
  void* const st = stream();
  // (nobody can wait inside a capture, and nothing is launched without tokens: the sums stay on the device then)
  if (post != nullptr && n > 0 && !capturing()) {
    const Slot& slot = post->send(st);
    const int rc =
        one_pass ? axon_policy_loss_post(kind, lp_p, old_p, adv_p, ptr(mk.first), mk.second, isw_p, rows.offsets(), rows.n_rows,
                                         n, rows.uniform_len, scale, valid_p, lo, hi, clip, grad_p, acc_p, ws_p,
                                         post->also(), post->n_also(), slot.device, slot.seq, st)
                 : axon_policy_loss_rows_post(kind, lp_p, old_p, adv_p, ptr(mk.first), mk.second, isw_p, rows.offsets(),
                                              rows.n_rows, n, rows.uniform_len, token_reduce, batch_reduce, prtc_p, npt_p,
                                              nps_p, valid_p, lo, hi, clip, grad_p, acc_p, ws_p, post->also(),
                                              post->n_also(), slot.device, slot.seq, st);
    post->sent(rc);
    check(rc, one_pass ? "axon_policy_loss" : "axon_policy_loss_rows");
  } else if (one_pass) {
    check(axon_policy_loss(kind, lp_p, old_p, adv_p, ptr(mk.first), mk.second, isw_p, rows.offsets(), rows.n_rows, n,
                           rows.uniform_len, nullptr, nullptr, scale, 1, valid_p, lo, hi, clip, grad_p, acc_p, ws_p, st),
          "axon_policy_loss");
  } else {
    check(axon_policy_loss_rows(kind, lp_p, old_p, adv_p, ptr(mk.first), mk.second, isw_p, rows.offsets(), rows.n_rows, n,
                                rows.uniform_len, token_reduce, batch_reduce, prtc_p, npt_p, nps_p, valid_p, lo, hi, clip,
                                grad_p, acc_p, ws_p, st),
          "axon_policy_loss_rows");
  }
  return {acc, grad};
}

Tensor group_advantage(const Tensor& rewards, const Tensor& mask, const Tensor& gidx, int64_t n_groups,
                       const RowsTuple& rows_tuple, double eps, int mode, double clamp_abs, const Tensor& ws) {
  const Rows rows = rows_of(rows_tuple);
  const int64_t n = rows.n_slots;
  same_len("group_advantage", "rewards", n, rewards);
  same_len("group_advantage", "mask", n, mask);
  same_len("group_advantage", "gidx", rows.n_rows, gidx);
  const Tensor rw = f32(rewards);
  const auto mk = mask_arg(mask);
  Tensor scratch = at::empty({2 * rows.n_rows}, opts(rw)), out = at::empty(rows.shape, opts(rw));
  check(axon_group_advantage((const float*)ptr(rw), ptr(mk.first), mk.second, rows.offsets(), rows.n_rows, n,
                             rows.uniform_len, gidx.data_ptr<int64_t>(), n_groups, (float)eps, mode, (float)clamp_abs,
                             scratch.data_ptr<float>(), out.data_ptr<float>(), ws.data_ptr<float>(), stream()),
        "axon_group_advantage");
  return out;
}

// (weights or none, new mask)
std::tuple<OptTensor, Tensor> sampler_correction_diag(
    const Tensor& old_log_probs, const Tensor& sampler_log_probs, const Tensor& mask, const RowsTuple& rows_tuple,
    int is_mode, double is_threshold, int rs_mode, double rs_lr_lo, double rs_lr_hi, std::optional<double> log_veto,
    double is_lo, double is_hi, double rs_lo, double rs_hi, double log_is_lo, double log_is_hi, double log_rs_lo,
    double log_rs_hi, const Tensor& acc, const Tensor& diag, const Tensor& part) {
  const Rows rows = rows_of(rows_tuple);
  const int64_t n = rows.n_slots;
  same_len("sampler_correction", "old_log_probs", n, old_log_probs);
  same_len("sampler_correction", "sampler_log_probs", n, sampler_log_probs);
  same_len("sampler_correction", "mask", n, mask);
  const Tensor old = f32(old_log_probs), samp = f32(sampler_log_probs);
  const auto mk = mask_arg(mask);
  OptTensor isw;
  if (is_mode) isw = at::empty(rows.shape, opts(old));
  Tensor new_mask = at::empty(rows.shape, opts(old));
  Tensor ws = at::empty({axon_sampler_correction_diag_workspace_bytes(rows.n_rows, n) / 4}, opts(old));
  check(axon_sampler_correction_diag(
        (const float*)ptr(old), (const float*)ptr(samp), ptr(mk.first), mk.second, rows.offsets(), rows.n_rows, n,
        rows.uniform_len, is_mode, (float)is_threshold, rs_mode, (float)rs_lr_lo, (float)rs_lr_hi, log_veto ? 1 : 0,
        (float)log_veto.value_or(0.0), (float)is_lo, (float)is_hi, (float)rs_lo, (float)rs_hi, (float)log_is_lo,
        (float)log_is_hi, (float)log_rs_lo, (float)log_rs_hi, isw ? isw->data_ptr<float>() : nullptr,
        new_mask.data_ptr<float>(), (float*)acc.data_ptr(), part.data_ptr<float>(), ws.data_ptr<float>(),
        diag.data_ptr<double>(), stream()),
        "axon_sampler_correction_diag");
  return {isw, new_mask};
}

// (adv or none, ret)
std::tuple<OptTensor, Tensor> reverse_scan(int mode, const Tensor& rewards, const OptTensor& values, const Tensor& mask,
                                           const RowsTuple& rows_tuple, double gamma, double lam,
                                           const OptTensor& row_baseline, bool want_adv) {
  const Rows rows = rows_of(rows_tuple);
  const int64_t n = rows.n_slots;
  same_len("reverse_scan", "rewards", n, rewards);
  same_len("reverse_scan", "values", n, values);
  same_len("reverse_scan", "mask", n, mask);
  const Tensor rw = f32(rewards), val = f32(values), base = f32(row_baseline);
  if (base.defined() && base.numel() != rows.n_rows)
    throw py::value_error("row_baseline has " + std::to_string(base.numel()) + " entries, batch has " +
                          std::to_string(rows.n_rows) + " rows");
  const auto mk = mask_arg(mask);
  OptTensor adv;
  if (want_adv) adv = at::empty(rows.shape, opts(rw));
  Tensor ret = at::empty(rows.shape, opts(rw));
  check(axon_reverse_scan(mode, (const float*)ptr(rw), (const float*)ptr(val), ptr(mk.first), mk.second, rows.offsets(),
                          rows.n_rows, n, rows.uniform_len, (float)gamma, (float)lam, (const float*)ptr(base),
                          adv ? adv->data_ptr<float>() : nullptr, ret.data_ptr<float>(), stream()),
        "axon_reverse_scan");
  return {adv, ret};
}

// x * s1 * s2 (device scalars, s2 may be missing) as a new fp32 tensor shaped like x
Tensor scale_f32(const Tensor& x, const Tensor& s1, const OptTensor& s2) {
  require_device(x, "scale_f32");  // a backward comes here without Python, with what a saved-tensor hook has handed back
  const Tensor xf = f32(x);
  const auto scalar = [&](const Tensor& s) {
    Tensor t = s.detach();
    return t.scalar_type() == at::kFloat && t.device() == xf.device() ? t : t.to(xf.device(), at::kFloat);
  };
  const Tensor a = scalar(s1), b = s2 ? scalar(*s2) : Tensor();
  Tensor out = at::empty_like(xf);
  check(axon_scale_f32((const float*)ptr(xf), (const float*)ptr(a), (const float*)ptr(b), out.data_ptr<float>(), xf.numel(),
                       stream()),
        "axon_scale_f32");
  return out.view(x.sizes());
}

// The node of a loss whose kernel has left the gradient beside it: loss = factor * acc[0], and in the backward
// grad * (factor * upstream) * acc[slot] (slot < 0: no such factor).
struct FinishedLoss : torch::autograd::Function<FinishedLoss> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& acc, const Tensor& grad,
                        double factor, int64_t slot) {
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({grad, acc});
    ctx->saved_data["factor"] = factor;
    ctx->saved_data["slot"] = slot;
    ctx->saved_data["dtype"] = (int64_t)x.scalar_type();
    if (factor != 1.0) return acc.select(0, 0) * factor;
    // acc[0] as a tensor of its own: no view (the caller may change it in place, and nothing reads it again)
    return at::empty({0}, acc.options()).set_(acc.storage(), acc.storage_offset(), {}, {});
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list upstream) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &grad = saved[0], &acc = saved[1];
    const double factor = ctx->saved_data["factor"].toDouble();
    const int64_t slot = ctx->saved_data["slot"].toInt();
    Tensor g = upstream[0].defined() ? upstream[0] : at::zeros({}, grad.options());
    if (factor != 1.0) g = g * factor;
    const Tensor out = scale_f32(grad, g, slot < 0 ? OptTensor() : OptTensor(acc.select(0, slot)));
    return {out.to((at::ScalarType)ctx->saved_data["dtype"].toInt()), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  g_error = py::object(py::module_::import("axon_amd._lib").attr("AxonAmdError")).release().ptr();
  py::register_exception_translator([](std::exception_ptr e) {
    try {
      if (e) std::rethrow_exception(e);
    } catch (const AxonError& err) {
      PyErr_SetString(g_error, err.what());
    }
  });
  // what this file was compiled against: axon_amd/_lib.py refuses another
  m.attr("abi_version") = AXON_AMD_ABI_VERSION;
  m.attr("torch_version") = AXON_TORCH_VERSION;
  const py::call_guard<py::gil_scoped_release> unlocked;
  py::class_<Post>(m, "Post")
      .def(py::init<OptTensor>())
      .def_property_readonly("sent", &Post::is_sent)
      .def("sums", &Post::sums, unlocked)
      .def("wait", &Post::wait, unlocked);
  m.def("post_slots", [] { return Slots::get().made(); });
  m.def("policy_loss", &policy_loss, unlocked);
  m.def("group_advantage", &group_advantage, unlocked);
  m.def("sampler_correction_diag", &sampler_correction_diag, unlocked);
  m.def("reverse_scan", &reverse_scan, unlocked);
  m.def("scale_f32", &scale_f32, unlocked);
  m.def("finished_loss", [](const Tensor& x, const Tensor& acc, const Tensor& grad, double factor,
                            int64_t slot) { return FinishedLoss::apply(x, acc, grad, factor, slot); }, unlocked);
}
