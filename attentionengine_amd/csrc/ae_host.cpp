// _ae_host: the host side of a repeated call, in native code.
//
// A call of an engine checks its tensors, allocates the results, fills ae_attn_params and launches.  The operators
// (core/lower/prefill_op.py, lower_decode.py, prefill_bwd_op.py) do that in Python the first time they meet a shape:
// that is where kernels are compiled, masks and splits planned, configurations measured, and where a wrong argument
// becomes an error that names it.  What they decided is then handed to a `Host` object as a PLAN - kernels, tile
// configurations, split counts, mask table - and every later call with the same extents runs here: match the
// tensors against the plan, two or three allocations, one launch function of the C ABI (with all of its checks).
// Anything a plan does not cover (other extents, other dtypes or devices, strides the kernels cannot read, tensor
// subclasses, switches in the environment that changed) returns None and the operator's Python code runs as before.
//
// Why: at batch 1 a decode or short prefill call is bound by the host.  Measured per call, one MI355X box: prefill of
// 333 tokens 15.7 -> 5.5 us, GQA decode 14.8 -> 5.7 us, paged latent decode 27.2 -> 8.4 us, forward + backward
// 77 -> 36 us of host time.  The reference's generated torch.autograd.Function and its TileLang / pybind11 callables
// do this work per call in Python as well (core/template/tl_template/attn/attn_tl.py:567-640).
//
// Threads: calls come from Python with the GIL held, which also guards the plans and the kept work buffers.  A launch
// runs without it - a full launch queue makes the caller wait, not the process - on what the call holds itself; so does
// the backward node, on autograd's own threads.

#include <torch/csrc/autograd/edge.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <memory>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "ae_hip.h"

namespace {

constexpr size_t kMaxPlans = 64;       // plans a Host keeps; the oldest goes
constexpr size_t kMaxWork = 16;        // work buffers a Host keeps, beyond those that a captured graph replays on

// Python objects that own the plan's code objects: released under the GIL whichever thread drops the last reference
struct Keep {
  PyObject* obj = nullptr;
  explicit Keep(PyObject* o) : obj(o) { Py_XINCREF(o); }
  Keep(const Keep&) = delete;
  Keep& operator=(const Keep&) = delete;
  ~Keep() {
    if (obj && Py_IsInitialized()) {
      PyGILState_STATE g = PyGILState_Ensure();
      Py_DECREF(obj);
      PyGILState_Release(g);
    }
  }
};

enum Kind { kPrefill = 0, kPrefillSplit = 1, kDecode = 2, kMla = 3, kMlaPaged = 4 };

struct BwdPlan {
  ae_kernel *delta = nullptr, *dkv = nullptr, *dq = nullptr;   // delta NULL: the dq launch forms the row sums
  ae_tile_cfg cfg{};
  int n_rs = 0;             // final row scales the kernels read (0: none)
  int planes = 2;           // fp32 planes of the work buffer
  int dkv_parts = 0;        // workgroups per kv tile of the dk/dv launch (0: kernels that do not share one out)
  int64_t work_more = 0;    // fp32 values of the work buffer behind its planes
  at::Tensor table_dq, table_dkv;     // tile classes of the two launches (mask mode 2)
  std::shared_ptr<Keep> keep;
  std::shared_ptr<Keep> again;        // weak reference to the Python operator, which can do without `work_more` (or none) ...
  int retry = 0;                      // ... and is called this many times more once it has been refused
  std::atomic<int> skip{0};           // calls left of these
};

struct Plan {
  Kind kind = kPrefill;
  int64_t B = 0, Sq = 0, Hq = 0, Hkv = 0, Skv = 0, page = 0;
  int device = -1;
  ae_kernel *k0 = nullptr, *k1 = nullptr;
  ae_tile_cfg cfg{}, ccfg{};
  bool has_ccfg = false;
  int n_split = 1, kv_per_split = 0;
  at::Tensor table;         // mask mode 2
  int mask_bm = 0, mask_bn = 0;
  std::vector<std::pair<std::string, std::string>> env;   // switches this plan was made under
  std::shared_ptr<Keep> keep;
  std::shared_ptr<BwdPlan> bwd;
  int64_t o_rows = 0, counters = 0;   // partial results a split launch writes; arrival counters behind the row scales
  int tail_slots = 0;                 // prefill: q-tile slots of an XCD that several workgroups share; paged MLA: workgroups a
                                      // head tile that share splits by the entries' lengths
};

// Work buffers of launches whose last workgroup merges: the arrival counters behind the row scales are zero when a
// launch starts, and every launch leaves them at zero (ae_decode_fwd).  Kept by the Host, per size and stream - launches
// on one stream run one after the other and may share them -, not by a plan: plans come and go with the shapes and
// settings of the calls, while a graph captured on the stream goes on using the addresses.
struct Work {
  int device;
  void* stream;
  int64_t o_rows, rs_floats, counters;
  bool captured;            // recorded into a graph: kept as long as the Host
  at::Tensor partial_o, partial_rs;
};

struct Host {
  PyObject_HEAD
  int64_t D, DV;
  at::ScalarType dtype;
  int n_custom, n_rs;
  int custom_in_dtype;      // bit i: custom input i is read in the input dtype (else fp32)
  std::vector<std::shared_ptr<Plan>>* plans;
  std::vector<Work>* work;
};

bool env_matches(const Plan& pl) {
  for (const auto& e : pl.env) {
    const char* v = getenv(e.first.c_str());
    if (e.second != (v ? v : "")) return false;
  }
  return true;
}

bool plain(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && !t.unsafeGetTensorImpl()->is_python_dispatch() && t.layout() == at::kStrided &&
         !t.is_conj() && !t.is_neg() && !t._fw_grad(0).defined();      // (forward mode: autograd.Function says it has no rule)
}

// a tensor the kernels read as it is: dense last dimension, 16-byte start, other strides multiples of 8 elements
bool readable(const at::Tensor& t) {
  const auto st = t.strides();
  const size_t n = st.size();
  if (st[n - 1] != 1 || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) != 0) return false;
  for (size_t i = 0; i + 1 < n; i++)
    if (st[i] % 8 != 0) return false;
  return true;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dt, int device) {
  return at::Tensor(at::detail::empty_cuda(sizes, dt, c10::Device(c10::kCUDA, (c10::DeviceIndex)device), std::nullopt));
}

bool is_capturing(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();              // (the default stream while another one captures)
  return true;
}

// The work buffers of a launch on `stream` (see Work).  A capture that finds none kept gets buffers of its own, which live
// in the graph's memory, and records the clearing of their counters: what a capture allocates and clears is only there
// when that graph has been replayed, so no other call may be given it.  `eager_only`: a capture always gets its own, so
// that its replays share nothing with any other call, on whatever streams they run (the clearing is one launch of about 2 us
// in a graph whose kernel takes a hundred).
std::pair<at::Tensor, at::Tensor> get_work(Host* h, int64_t o_rows, int64_t rs_floats, int64_t counters, int device, void* stream,
                                           bool eager_only) {
  const bool capturing = is_capturing(stream);
  for (auto& w : *h->work)
    if (!(eager_only && capturing) && w.device == device && w.stream == stream && w.o_rows == o_rows && w.rs_floats == rs_floats && w.counters == counters) {
      w.captured = w.captured || capturing;
      return {w.partial_o, w.partial_rs};
    }
  at::Tensor po = empty({o_rows, h->DV}, at::kFloat, device), prs = empty({rs_floats + counters}, at::kFloat, device);
  prs.narrow(0, rs_floats, counters).zero_();
  if (!capturing) {
    size_t n = 0;
    for (const auto& w : *h->work) n += !w.captured;
    if (n >= kMaxWork)
      for (auto it = h->work->begin(); it != h->work->end(); ++it)
        if (!it->captured) {
          h->work->erase(it);
          break;
        }
    h->work->push_back({device, stream, o_rows, rs_floats, counters, false, po, prs});
  }
  return {po, prs};
}

void set_strides(const at::Tensor& t, int64_t& b, int64_t& s, int64_t& h) {
  b = t.stride(0), s = t.stride(1), h = t.stride(2);
}

struct AeBackward : public torch::autograd::Node {
  std::shared_ptr<BwdPlan> plan;
  torch::autograd::SavedVariable q_, k_, v_, out_;
  std::vector<torch::autograd::SavedVariable> scales_;
  std::vector<at::Tensor> customs;

  std::string name() const override { return "AttentionEngineBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    q_.reset_data(), k_.reset_data(), v_.reset_data(), out_.reset_data();
    for (auto& s : scales_) s.reset_data();
  }
  // (dq, dk, dv) from the operator behind the weak reference: a call of it that keeps no ds
  static torch::autograd::variable_list in_python(const Keep& again, const std::vector<at::Tensor>& args) {
    PyGILState_STATE g = PyGILState_Ensure();
    PyObject *op = PyObject_CallObject(again.obj, nullptr), *res = nullptr;
    torch::autograd::variable_list grads;
    if (op && op != Py_None) {
      PyObject *t = PyTuple_New((Py_ssize_t)args.size()), *more = Py_BuildValue("{s:O}", "without_ds", Py_True);
      for (size_t i = 0; t && i < args.size(); i++) PyTuple_SET_ITEM(t, (Py_ssize_t)i, THPVariable_Wrap(args[i]));
      res = t && more ? PyObject_Call(op, t, more) : nullptr;
      Py_XDECREF(t);
      Py_XDECREF(more);
      for (Py_ssize_t i = 0; res && PyTuple_Check(res) && i < PyTuple_GET_SIZE(res); i++)
        grads.push_back(THPVariable_Unpack(PyTuple_GET_ITEM(res, i)));
    }
    const bool failed = PyErr_Occurred() != nullptr;
    python_error err;
    if (failed) err.persist();
    Py_XDECREF(res);
    Py_XDECREF(op);
    PyGILState_Release(g);
    if (failed) throw err;
    TORCH_CHECK_WITH(OutOfMemoryError, grads.size() == 3, "no memory for the work buffer of the backward, and its operator is gone");
    return grads;
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!grads[0].defined()) return torch::autograd::variable_list(3);
    at::NoGradGuard no_grad;
    BwdPlan& pl = *plan;
    const at::Tensor q = q_.unpack(), k = k_.unpack(), v = v_.unpack(), out = out_.unpack(shared_from_this());
    std::vector<at::Tensor> rs;
    for (auto& s : scales_) rs.push_back(s.unpack());
    at::Tensor dout = grads[0];
    if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
    if (!readable(dout)) dout = dout.contiguous();
    const int dev = q.get_device();
    const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), Skv = k.size(1), Hkv = k.size(2);
    if (pl.skip > 0 && pl.skip-- > 0) return in_python(*pl.again, {q, k, v, out, rs[0], dout});
    at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), work;     // (in front of ds, which a call can do without)
    try {
      work = empty({pl.planes * B * Hq * Sq + pl.work_more}, at::kFloat, dev);
    } catch (const c10::OutOfMemoryError&) {
      if (!pl.again) throw;
      dq.reset(), dk.reset(), dv.reset();
      pl.skip = pl.retry;
    }
    if (!work.defined()) return in_python(*pl.again, {q, k, v, out, rs[0], dout});
    ae_attn_bwd_params p{};
    p.q = q.const_data_ptr(), p.k = k.const_data_ptr(), p.v = v.const_data_ptr(), p.out = out.const_data_ptr();
    p.dout = dout.const_data_ptr();
    p.lse = rs.empty() ? nullptr : (const float*)rs[0].const_data_ptr();
    for (size_t i = 1; i < rs.size(); i++) p.more_rowscales[i - 1] = (const float*)rs[i].const_data_ptr();
    for (size_t i = 0; i < customs.size(); i++) p.custom[i] = customs[i].const_data_ptr();
    p.delta = (float*)work.mutable_data_ptr();
    p.dq = dq.mutable_data_ptr(), p.dk = dk.mutable_data_ptr(), p.dv = dv.mutable_data_ptr();
    set_strides(q, p.q_stride_b, p.q_stride_s, p.q_stride_h);
    set_strides(k, p.k_stride_b, p.k_stride_s, p.k_stride_h);
    set_strides(v, p.v_stride_b, p.v_stride_s, p.v_stride_h);
    set_strides(out, p.o_stride_b, p.o_stride_s, p.o_stride_h);
    set_strides(dout, p.do_stride_b, p.do_stride_s, p.do_stride_h);
    set_strides(dq, p.dq_stride_b, p.dq_stride_s, p.dq_stride_h);
    set_strides(dk, p.dk_stride_b, p.dk_stride_s, p.dk_stride_h);
    set_strides(dv, p.dv_stride_b, p.dv_stride_s, p.dv_stride_h);
    p.batch = (int)B, p.heads_q = (int)Hq, p.heads_kv = (int)Hkv, p.seqlen_q = (int)Sq, p.seqlen_kv = (int)Skv;
    p.dkv_parts = pl.dkv_parts;
    if (pl.table_dq.defined()) {
      p.mask_dq = (const int8_t*)pl.table_dq.const_data_ptr(), p.mask_dkv = (const int8_t*)pl.table_dkv.const_data_ptr();
      p.mask_b = (int)pl.table_dq.size(0), p.mask_h = (int)pl.table_dq.size(1);
    }
    // (autograd has made the forward's device and stream current on this thread)
    const int rc = ae_prefill_bwd(pl.delta, pl.dkv, pl.dq, &p, &pl.cfg,
                                  (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
    TORCH_CHECK(rc == 0, "[ae status ", rc, "] ", ae_last_error());
    return {dq, dk, dv};
  }
};

// ---- forward ---------------------------------------------------------------------------------------------------------
struct Call {
  at::Tensor q, k, v, q2, k2, block_table, seqlens;
  int64_t B, Sq, Hq, Hkv, Skv, page = 0;
  Kind kind;             // kPrefill stands for prefill, split prefill and GQA decode: the plan says which
};

std::shared_ptr<Plan> find(Host* h, const Call& c, int device) {
  auto& v = *h->plans;
  for (size_t i = 0; i < v.size(); i++) {
    const Plan& pl = *v[i];
    if (pl.B == c.B && pl.Sq == c.Sq && pl.Hq == c.Hq && pl.Hkv == c.Hkv && pl.Skv == c.Skv && pl.device == device &&
        pl.page == c.page && (pl.kind >= kMla ? pl.kind == c.kind : c.kind == kPrefill)) {
      if (i) std::swap(v[i], v[0]);
      return v[0];
    }
  }
  return nullptr;
}

// (torch.Tensor and torch.nn.Parameter themselves: a subclass may override what its calls do, __torch_function__)
const at::Tensor* tensor_arg(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

// The call's tensors as the plan's kernel takes them; false: not a call for this path
bool gather(Host* h, PyObject* const* args, Py_ssize_t n, bool mla, Call& c) {
  const at::Tensor* t[4] = {nullptr, nullptr, nullptr, nullptr};
  const int nt = mla ? (int)n : 3;
  for (int i = 0; i < nt; i++) {
    t[i] = tensor_arg(args[i]);
    if (!t[i] || !plain(*t[i])) return false;
  }
  if (!mla) {
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2];
    if (q.scalar_type() != h->dtype || k.scalar_type() != h->dtype || v.scalar_type() != h->dtype) return false;
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
    c.B = q.size(0), c.Sq = q.size(1), c.Hq = q.size(2), c.Skv = k.size(1), c.Hkv = k.size(2);
    if (q.size(3) != h->D || k.size(3) != h->D || v.size(3) != h->DV || k.size(0) != c.B || v.size(0) != c.B ||
        v.size(1) != c.Skv || v.size(2) != c.Hkv)
      return false;
    if (k.get_device() != q.get_device() || v.get_device() != q.get_device()) return false;
    if (!readable(q) || !readable(k) || !readable(v)) return false;
    c.q = q, c.k = k, c.v = v, c.kind = kPrefill;
    return true;
  }
  const int64_t D2 = h->D - h->DV;
  if (t[0]->scalar_type() != h->dtype || t[1]->scalar_type() != h->dtype || t[0]->dim() != 4 || t[1]->dim() != 4) return false;
  for (int i = 1; i < nt; i++)
    if (t[i]->get_device() != t[0]->get_device()) return false;
  const at::Tensor& q = *t[0];
  c.B = q.size(0), c.Sq = q.size(1), c.Hq = q.size(2);
  if (c.Sq != 1 || !readable(q)) return false;
  if (n == 2 || (n == 4 && t[2]->scalar_type() == at::kInt)) {        // mod(q, kv_cache), perhaps with its page table
    const at::Tensor& cache = *t[1];
    if (q.size(3) != h->D || cache.size(3) != h->D) return false;
    c.Hkv = cache.size(2);
    if (n == 4) {
      const at::Tensor &bt = *t[2], &sl = *t[3];
      if (sl.scalar_type() != at::kInt || bt.dim() != 2 || bt.size(0) != c.B || bt.stride(1) != 1 || sl.dim() != 1 ||
          sl.size(0) != c.B || !sl.is_contiguous() || !readable(cache))
        return false;
      c.page = cache.size(1), c.Skv = bt.size(1) * c.page;
      c.block_table = bt, c.seqlens = sl, c.kind = kMlaPaged;
      c.k = cache, c.q = q;
      return true;
    }
    if (!cache.is_contiguous() || (reinterpret_cast<uintptr_t>(cache.const_data_ptr()) & 15) != 0) return false;
    const int64_t rows = cache.size(0) * cache.size(1);
    if (c.B == 0 || rows % c.B) return false;
    c.Skv = rows / c.B, c.kind = kMla, c.k = cache, c.q = q;
    return true;
  }
  if (n != 4 || t[2]->dim() != 4 || t[3]->dim() != 4 || t[2]->scalar_type() != h->dtype || t[3]->scalar_type() != h->dtype) return false;
  const at::Tensor &q2 = *t[1], &k1 = *t[2], &k2 = *t[3];
  c.Skv = k1.size(1), c.Hkv = k1.size(2);
  if (q.size(3) != h->DV || q2.size(3) != D2 || k1.size(3) != h->DV || k2.size(3) != D2 || k1.size(0) != c.B || k2.size(0) != c.B ||
      k2.size(1) != c.Skv || k2.size(2) != c.Hkv || q2.size(0) != c.B || q2.size(1) != 1 || q2.size(2) != c.Hq)
    return false;
  if (!readable(q2) || !readable(k1) || !readable(k2)) return false;
  c.q = q, c.q2 = q2, c.k = k1, c.k2 = k2, c.kind = kMla;
  return true;
}

PyObject* raise_status(int rc) {
  // the same exception the ctypes binding raises (core.runtime.hip_rt.AEError, a RuntimeError)
  static PyObject* type = nullptr;
  if (!type) {
    PyObject* m = PyImport_ImportModule("core.runtime.hip_rt");
    if (m) {
      type = PyObject_GetAttrString(m, "AEError");
      Py_DECREF(m);
    }
    PyErr_Clear();
  }
  PyErr_Format(type ? type : PyExc_RuntimeError, "[ae status %d] %s", rc, ae_last_error());
  return nullptr;
}

// run(q, k, v, *customs) / run(q, q_pe, kv, k_pe) / run(q, cache[, block_table, seqlens]) -> (out, *row scales) or None
PyObject* run(Host* h, PyObject* const* args, Py_ssize_t nargs, bool mla) {
  if (h->plans->empty()) Py_RETURN_NONE;
  if (mla ? (nargs != 2 && nargs != 4) : nargs != 3 + h->n_custom) Py_RETURN_NONE;
  Call c;
  if (!gather(h, args, nargs, mla, c)) Py_RETURN_NONE;
  const int dev = c.q.get_device();
  if ((int)c10::hip::current_device() != dev) Py_RETURN_NONE;
  const std::shared_ptr<Plan> plp = find(h, c, dev);
  if (!plp || !env_matches(*plp)) Py_RETURN_NONE;
  Plan& pl = *plp;
  const at::Tensor* customs[AE_MAX_CUSTOM];
  const int n_custom = mla ? 0 : h->n_custom;
  for (int i = 0; i < n_custom; i++) {
    const at::Tensor* t = tensor_arg(args[3 + i]);
    if (!t || !plain(*t) || t->get_device() != dev || !t->is_contiguous() || t->requires_grad() ||
        t->scalar_type() != ((h->custom_in_dtype >> i) & 1 ? h->dtype : at::kFloat))
      Py_RETURN_NONE;
    customs[i] = t;
  }
  bool wants_grad = false;
  if (!mla && at::GradMode::is_enabled()) wants_grad = c.q.requires_grad() || c.k.requires_grad() || c.v.requires_grad();
  if (wants_grad && !pl.bwd) Py_RETURN_NONE;
  const bool at_row = pl.kind == kDecode || mla;        // one query token: row scales are [B, Hq, 1]
  void* stream = (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
  const int64_t B = c.B, Sq = c.Sq, Hq = c.Hq;

  at::Tensor out = empty({B, Sq, Hq, h->DV}, h->dtype, dev);
  at::Tensor rs[AE_MAX_ROWSCALES];
  ae_attn_params p{};
  for (int i = 0; i < h->n_rs; i++) {
    rs[i] = at_row ? empty({B, Hq, 1}, at::kFloat, dev) : empty({B, Hq, Sq}, at::kFloat, dev);
    p.rowscale_out[i] = (float*)rs[i].mutable_data_ptr();
  }
  p.q = c.q.const_data_ptr(), p.k = c.k.const_data_ptr(), p.out = out.mutable_data_ptr();
  set_strides(c.q, p.q_stride_b, p.q_stride_s, p.q_stride_h);
  set_strides(c.k, p.k_stride_b, p.k_stride_s, p.k_stride_h);
  set_strides(out, p.o_stride_b, p.o_stride_s, p.o_stride_h);
  if (mla) {
    p.v = p.k;
    if (c.kind == kMla && !c.q2.defined()) {             // a dense cache of pages in order, read as [B, Skv, Hkv, D]
      p.k_stride_b = c.Skv * c.Hkv * h->D, p.k_stride_s = c.Hkv * h->D, p.k_stride_h = h->D;
    }
    if (c.q2.defined()) {
      p.q2 = c.q2.const_data_ptr(), p.k2 = c.k2.const_data_ptr();
      set_strides(c.q2, p.q2_stride_b, p.q2_stride_s, p.q2_stride_h);
      set_strides(c.k2, p.k2_stride_b, p.k2_stride_s, p.k2_stride_h);
    } else {                                             // the rope part: the last columns of the same tensors
      p.q2 = (const char*)p.q + h->DV * 2, p.k2 = (const char*)p.k + h->DV * 2;
      p.q2_stride_b = p.q_stride_b, p.q2_stride_s = p.q_stride_s, p.q2_stride_h = p.q_stride_h;
      p.k2_stride_b = p.k_stride_b, p.k2_stride_s = p.k_stride_s, p.k2_stride_h = p.k_stride_h;
    }
    p.v_stride_b = p.k_stride_b, p.v_stride_s = p.k_stride_s, p.v_stride_h = p.k_stride_h;
    if (c.kind == kMlaPaged) {
      p.block_table = (const int32_t*)c.block_table.const_data_ptr(), p.seqlens_k = (const int32_t*)c.seqlens.const_data_ptr();
      p.block_table_stride = (int)c.block_table.stride(0), p.page_block_size = (int)c.page, p.num_pages = (int)c.k.size(0);
    }
  } else {
    p.v = c.v.const_data_ptr();
    set_strides(c.v, p.v_stride_b, p.v_stride_s, p.v_stride_h);
  }
  p.batch = (int)B, p.heads_q = (int)Hq, p.heads_kv = (int)c.Hkv, p.seqlen_q = (int)Sq, p.seqlen_kv = (int)c.Skv;
  for (int i = 0; i < n_custom; i++) p.custom[i] = customs[i]->const_data_ptr();
  if (pl.table.defined()) {
    p.block_mask = (const int8_t*)pl.table.const_data_ptr();
    p.mask_b = (int)pl.table.size(0), p.mask_h = (int)pl.table.size(1);
    p.mask_nq = (int)pl.table.size(2), p.mask_nkv = (int)pl.table.size(3);
    p.mask_block_m = pl.mask_bm, p.mask_block_n = pl.mask_bn;
  }
  ae_tile_cfg cfg = pl.cfg;
  const int64_t rs_floats = (h->n_rs > 0 ? h->n_rs : 1) * B * Sq * Hq * pl.n_split;
  at::Tensor po, prs;
  if (pl.kind != kPrefill || pl.tail_slots) p.num_splits = pl.n_split, p.kv_per_split = pl.kv_per_split;
  if (pl.kind == kMlaPaged) p.tail_slots = pl.tail_slots;
  if (pl.kind != kMlaPaged && pl.tail_slots) {      // (only the counters are kept: the partial results are the size of a few thousand rows)
    p.tail_slots = pl.tail_slots;
    po = empty({pl.o_rows, h->DV}, at::kFloat, dev);
    prs = get_work(h, 1, 1, pl.counters, dev, stream, true).second.narrow(0, 1, pl.counters);
  } else if (pl.kind == kPrefillSplit && pl.counters && !is_capturing(stream)) {
    // (the last workgroup merges; not in a graph, where the clearing of its counters costs what the merge launch does:
    // B3 H8 Sq8 Skv1680 D64 9.1 us a replay, 10.2 so)
    cfg.merge_in_wg = 2;
    po = empty({pl.o_rows, h->DV}, at::kFloat, dev);
    prs = get_work(h, 1, rs_floats, pl.counters, dev, stream, true).second;
  } else if (pl.cfg.merge_in_wg == 2) {
    std::tie(po, prs) = get_work(h, pl.o_rows, rs_floats, pl.counters, dev, stream, false);
  } else if (pl.n_split > 1 && pl.cfg.merge_in_wg == 0) {
    po = empty({pl.o_rows, h->DV}, at::kFloat, dev);
    prs = empty({rs_floats + (pl.tail_slots ? B : 0)}, at::kFloat, dev);
  }
  if (po.defined()) p.partial_o = (float*)po.mutable_data_ptr(), p.partial_rs = (float*)prs.mutable_data_ptr();

  int rc;
  PyThreadState* thread = PyEval_SaveThread();
  switch (pl.kind) {
    case kPrefill: rc = ae_prefill_fwd(pl.k0, &p, &cfg, stream); break;
    case kPrefillSplit: rc = ae_prefill_split_fwd(pl.k0, pl.k1, &p, &cfg, &pl.ccfg, stream); break;
    case kDecode: rc = ae_decode_fwd(pl.k0, pl.k1, &p, &pl.cfg, pl.has_ccfg ? &pl.ccfg : nullptr, stream); break;
    default: rc = ae_mla_decode_fwd(pl.k0, pl.k1, &p, &pl.cfg, &pl.ccfg, stream); break;
  }
  PyEval_RestoreThread(thread);
  if (rc) return raise_status(rc);

  if (wants_grad) {
    auto fn = std::shared_ptr<AeBackward>(new AeBackward(), torch::autograd::deleteNode);
    fn->set_next_edges(torch::autograd::collect_next_edges(c.q, c.k, c.v));
    fn->plan = pl.bwd;
    fn->q_ = torch::autograd::SavedVariable(c.q, false);
    fn->k_ = torch::autograd::SavedVariable(c.k, false);
    fn->v_ = torch::autograd::SavedVariable(c.v, false);
    for (int i = 0; i < pl.bwd->n_rs; i++) fn->scales_.emplace_back(rs[i], false);
    for (int i = 0; i < n_custom; i++) fn->customs.push_back(*customs[i]);
    torch::autograd::set_history(out, fn);
    fn->out_ = torch::autograd::SavedVariable(out, true);
  }
  PyObject* res = PyTuple_New(1 + h->n_rs);
  if (!res) return nullptr;
  PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(out));
  for (int i = 0; i < h->n_rs; i++) PyTuple_SET_ITEM(res, 1 + i, THPVariable_Wrap(rs[i]));
  return res;
}

template <bool MLA>
PyObject* host_run(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  return run((Host*)self, args, nargs, MLA);
  END_HANDLE_TH_ERRORS
}

// ---- plans from Python ----------------------------------------------------------------------------------------------
int64_t get_int(PyObject* d, const char* key, int64_t dflt = 0) {
  PyObject* o = PyDict_GetItemString(d, key);
  if (!o || o == Py_None) return dflt;
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
bool get_cfg(PyObject* d, const char* key, ae_tile_cfg& cfg) {
  PyObject* o = PyDict_GetItemString(d, key);
  if (!o || o == Py_None) return false;
  char* data;
  Py_ssize_t n;
  if (PyBytes_AsStringAndSize(o, &data, &n) < 0) throw python_error();
  TORCH_CHECK(n == (Py_ssize_t)sizeof cfg, key, ": ", n, " bytes");
  memcpy(&cfg, data, sizeof cfg);
  return true;
}
at::Tensor get_tensor(PyObject* d, const char* key) {
  PyObject* o = PyDict_GetItemString(d, key);
  if (!o || o == Py_None) return at::Tensor();
  TORCH_CHECK(THPVariable_Check(o), key, " is not a tensor");
  return THPVariable_Unpack(o);
}

// add(dict): see core/runtime/host.py for the keys
PyObject* host_add(PyObject* self, PyObject* d) {
  HANDLE_TH_ERRORS
  Host* h = (Host*)self;
  TORCH_CHECK(PyDict_Check(d), "add() takes a dict");
  auto pl = std::make_shared<Plan>();
  pl->kind = (Kind)get_int(d, "kind");
  pl->B = get_int(d, "B"), pl->Sq = get_int(d, "Sq"), pl->Hq = get_int(d, "Hq"), pl->Hkv = get_int(d, "Hkv");
  pl->Skv = get_int(d, "Skv"), pl->page = get_int(d, "page");
  pl->device = (int)get_int(d, "device");
  pl->k0 = (ae_kernel*)(uintptr_t)get_int(d, "k0"), pl->k1 = (ae_kernel*)(uintptr_t)get_int(d, "k1");
  TORCH_CHECK(pl->k0 && get_cfg(d, "cfg", pl->cfg), "a plan needs a kernel and its tile configuration");
  pl->has_ccfg = get_cfg(d, "ccfg", pl->ccfg);
  pl->n_split = (int)get_int(d, "n_split", 1), pl->kv_per_split = (int)get_int(d, "kv_per_split");
  pl->o_rows = get_int(d, "o_rows", pl->B * pl->Sq * pl->Hq * pl->n_split), pl->counters = get_int(d, "counters");
  pl->tail_slots = (int)get_int(d, "tail_slots");
  TORCH_CHECK(pl->cfg.merge_in_wg != 2 || pl->counters > 0, "a launch whose last workgroup merges needs arrival counters");
  pl->table = get_tensor(d, "table");
  pl->mask_bm = (int)get_int(d, "mask_bm"), pl->mask_bn = (int)get_int(d, "mask_bn");
  if (PyObject* env = PyDict_GetItemString(d, "env")) {
    PyObject *key, *value;
    Py_ssize_t pos = 0;
    while (PyDict_Next(env, &pos, &key, &value)) pl->env.emplace_back(PyUnicode_AsUTF8(key), PyUnicode_AsUTF8(value));
  }
  pl->keep = std::make_shared<Keep>(PyDict_GetItemString(d, "keep"));
  auto& v = *h->plans;
  for (size_t i = 0; i < v.size(); i++)      // a new plan for the same call replaces the old one
    if (v[i]->B == pl->B && v[i]->Sq == pl->Sq && v[i]->Hq == pl->Hq && v[i]->Hkv == pl->Hkv && v[i]->Skv == pl->Skv &&
        v[i]->device == pl->device && v[i]->page == pl->page && (v[i]->kind == kMlaPaged) == (pl->kind == kMlaPaged)) {
      pl->bwd = v[i]->bwd;
      v.erase(v.begin() + (long)i);
      break;
    }
  if (v.size() >= kMaxPlans) v.pop_back();
  v.insert(v.begin(), pl);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// add_backward(dict): attaches the backward of the plan with these extents (no such plan: nothing happens)
PyObject* host_add_backward(PyObject* self, PyObject* d) {
  HANDLE_TH_ERRORS
  Host* h = (Host*)self;
  TORCH_CHECK(PyDict_Check(d), "add_backward() takes a dict");
  auto bw = std::make_shared<BwdPlan>();
  bw->delta = (ae_kernel*)(uintptr_t)get_int(d, "delta"), bw->dkv = (ae_kernel*)(uintptr_t)get_int(d, "dkv");
  bw->dq = (ae_kernel*)(uintptr_t)get_int(d, "dq");
  TORCH_CHECK(bw->dkv && bw->dq && get_cfg(d, "cfg", bw->cfg), "a backward plan needs its kernels and their tile configuration");
  bw->n_rs = (int)get_int(d, "n_rs"), bw->planes = (int)get_int(d, "planes", 2);
  bw->dkv_parts = (int)get_int(d, "dkv_parts"), bw->work_more = get_int(d, "work_more");
  bw->table_dq = get_tensor(d, "table_dq"), bw->table_dkv = get_tensor(d, "table_dkv");
  bw->keep = std::make_shared<Keep>(PyDict_GetItemString(d, "keep"));
  PyObject* again = PyDict_GetItemString(d, "again");
  if (again && again != Py_None)
    bw->again = std::make_shared<Keep>(again), bw->retry = (int)get_int(d, "retry"), bw->skip = (int)get_int(d, "skip");
  for (auto& pl : *h->plans)
    if (pl->kind == kPrefill && pl->B == get_int(d, "B") && pl->Sq == get_int(d, "Sq") && pl->Hq == get_int(d, "Hq") &&
        pl->Hkv == get_int(d, "Hkv") && pl->Skv == get_int(d, "Skv") && pl->device == (int)get_int(d, "device"))
      pl->bwd = bw;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// work(o_rows, rs_floats, counters, device, stream, eager_only) -> (partial_o, partial_rs)
PyObject* host_work(PyObject* self, PyObject* args) {
  HANDLE_TH_ERRORS
  long long o_rows, rs_floats, counters, stream;
  int device, eager_only = 0;
  if (!PyArg_ParseTuple(args, "LLLiL|p", &o_rows, &rs_floats, &counters, &device, &stream, &eager_only)) return nullptr;
  TORCH_CHECK(o_rows > 0 && rs_floats > 0 && counters > 0, "work(): sizes must be positive");
  auto w = get_work((Host*)self, o_rows, rs_floats, counters, device, (void*)(uintptr_t)stream, eager_only != 0);
  PyObject* res = PyTuple_New(2);
  if (!res) return nullptr;
  PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(w.first));
  PyTuple_SET_ITEM(res, 1, THPVariable_Wrap(w.second));
  return res;
  END_HANDLE_TH_ERRORS
}

PyObject* host_clear(PyObject* self, PyObject*) {
  ((Host*)self)->plans->clear();
  Py_RETURN_NONE;
}
Py_ssize_t host_len(PyObject* self) { return (Py_ssize_t)((Host*)self)->plans->size(); }

PyObject* host_new(PyTypeObject* type, PyObject* args, PyObject*) {
  long long D, DV;
  int bf16, n_custom, in_dtype, n_rs;
  if (!PyArg_ParseTuple(args, "LLpiii", &D, &DV, &bf16, &n_custom, &in_dtype, &n_rs)) return nullptr;
  if (n_custom < 0 || n_custom > AE_MAX_CUSTOM || n_rs < 0 || n_rs > AE_MAX_ROWSCALES) {
    PyErr_SetString(PyExc_ValueError, "too many custom inputs / row scales");
    return nullptr;
  }
  Host* h = (Host*)type->tp_alloc(type, 0);
  if (!h) return nullptr;
  h->D = D, h->DV = DV, h->dtype = bf16 ? at::kBFloat16 : at::kHalf, h->n_custom = n_custom, h->n_rs = n_rs;
  h->custom_in_dtype = in_dtype;
  h->plans = new std::vector<std::shared_ptr<Plan>>();
  h->work = new std::vector<Work>();
  return (PyObject*)h;
}
void host_dealloc(PyObject* self) {
  delete ((Host*)self)->plans;
  delete ((Host*)self)->work;
  PyTypeObject* tp = Py_TYPE(self);
  tp->tp_free(self);
  Py_DECREF(tp);
}

PyMethodDef host_methods[] = {
    {"run", (PyCFunction)(void (*)(void))host_run<false>, METH_FASTCALL, "run(q, k, v, *customs) -> (out, *row scales) or None"},
    {"run_mla", (PyCFunction)(void (*)(void))host_run<true>, METH_FASTCALL,
     "run_mla(q, q_pe, kv, k_pe) or run_mla(q, cache[, block_table, cache_seqlens]) -> (out, *row scales) or None"},
    {"add", host_add, METH_O, "add(plan dict)"},
    {"add_backward", host_add_backward, METH_O, "add_backward(plan dict)"},
    {"work", host_work, METH_VARARGS, "work(o_rows, rs_floats, counters, device, stream[, eager_only]) -> (partial_o, partial_rs) with zero counters"},
    {"clear", host_clear, METH_NOARGS, "drop every plan"},
    {nullptr, nullptr, 0, nullptr}};
PyType_Slot host_slots[] = {{Py_tp_new, (void*)host_new}, {Py_tp_dealloc, (void*)host_dealloc}, {Py_tp_methods, host_methods},
                            {Py_sq_length, (void*)host_len}, {0, nullptr}};
PyType_Spec host_spec = {"_ae_host.Host", sizeof(Host), 0, Py_TPFLAGS_DEFAULT, host_slots};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ae_host", "native host path of repeated calls", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ae_host() {
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  PyObject* t = PyType_FromSpec(&host_spec);
  if (!t || PyModule_AddObject(m, "Host", t) < 0 || PyModule_AddIntConstant(m, "ABI_VERSION", AE_ABI_VERSION) < 0) return nullptr;
  return m;
}
