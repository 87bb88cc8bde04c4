// The host side of the calls a model makes most often, native: the fused forward of one projection, and the autograd
// functions rms_norm, add_lora and fused_add_lora.  A launch takes the host 3 us; what came around it in Python made small
// batches wait.  us, whole passes in Python / so: RMSNorm forward and backward of 4224 rows 99 / 57 (41 in its kernels),
// add_lora forward and backward of three sequences of 200 rows 278 / 112, seven layers' forward of eight decoded rows
// 150 / 116, four layers' forward and backward of 4224 rows 600-820 / 390-530 (290 in their kernels).  What is left is
// mostly autograd's hand-over to its device thread, 20 to 50 a backward, and the launches.
//
// Every function here takes a call only in its plain form (tensors that are exactly torch's, on the current device, of
// the shapes and types the operator wants; no tracing, no functorch transform, no dispatch mode, no forward-mode
// tangent) and otherwise hands it back, having done nothing: the Python functions of the same names remain the general
// path and raise the errors.  Nothing is kept from one call to the next but the device tables of the gradients' addresses
// that the layers' backward keeps in either language (grad_tabs).
#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/version.h>

#include <string.h>

#include "smlm.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// ---- the operator library: loaded by Python, which hands over the addresses ----
struct Lib {
  decltype(&smlm_strerror) strerror;
  decltype(&smlm_plan_size) plan_size;
  decltype(&smlm_lora_fwd_multi_workspace_size) fwd_size;
  decltype(&smlm_lora_fwd_multi_ex) fwd;
  decltype(&smlm_lora_bwd_multi_workspace_size) bwd_size;
  decltype(&smlm_lora_bwd_multi_ex) bwd;
  decltype(&smlm_rms_norm_fwd) rms_fwd;
  decltype(&smlm_rms_norm_bwd_workspace_size) rms_bwd_size;
  decltype(&smlm_rms_norm_bwd) rms_bwd;
  decltype(&smlm_put_words) put;
} lib;
PyObject* default_workspace = nullptr;  // ops._kernels._workspace

struct Names {
  PyObject *T, *S, *kind, *built, *buf, *segment, *seg_key, *seg_key2, *ws_buf, *reserve, *workspace, *packed, *wa_table,
      *wb_table, *seg_scale, *plan, *rank, *train_len, *train_partition, *dropout, *adapter_rank, *part_segments, *bwd_plan,
      *part_adapter, *a_tab, *b_tab, *grad_layout, *gather, *grad_uniform, *grad_tabs, *grad_offsets_a, *grad_offsets_b;
} names;

void check(int rc, const char* what) {
  TORCH_CHECK(rc == SMLM_OK, what, ": ", lib.strerror(rc), " (code ", rc, ")");
}

struct Gil {
  PyGILState_STATE state = PyGILState_Ensure();
  ~Gil() { PyGILState_Release(state); }
};
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
struct python_raised {};  // the Python error is set

THPObjectPtr attr(PyObject* o, PyObject* name) {
  THPObjectPtr v(PyObject_GetAttr(o, name));
  if (!v) throw python_raised();
  return v;
}
int64_t integer(PyObject* o) {
  THPObjectPtr n(PyNumber_Index(o));  // (of numpy's integers too)
  if (!n) throw python_raised();
  const int64_t v = PyLong_AsLongLong(n);
  if (v == -1 && PyErr_Occurred()) throw python_raised();
  return v;
}

// ---- what makes a call plain ----
bool plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet kOther({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                        c10::DispatchKey::Batched, c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                        c10::DispatchKey::ZeroTensor, c10::DispatchKey::Python});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kOther) &&
         !t._fw_grad(0).defined();
}
bool plain_thread() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing();
}
bool half(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
int dtype_code(const Tensor& t) { return t.scalar_type() == at::kHalf ? SMLM_DTYPE_F16 : SMLM_DTYPE_BF16; }
bool here(const Tensor& t) { return t.device().index() == c10::hip::current_device(); }
bool is(const Tensor& t, at::ScalarType type, int64_t dim) {
  return t.scalar_type() == type && t.dim() == dim && t.is_contiguous();
}
void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false));
}
// A saved tensor comes back from whatever hooks its program has set (torch.autograd.graph.saved_tensors_hooks), which torch
// does not look at: what the kernels take for granted is checked in every backward, with the Python functions' words.
void check_input(const Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}
const Tensor* optional(PyObject* o, bool* ok) {
  if (o == Py_None) return nullptr;
  *ok = *ok && plain(o);
  return *ok ? &THPVariable_Unpack(o) : nullptr;
}

// ops._kernels.SegmentPlan
struct Plan {
  PyObject* o;
  int T, S, kind;
  bool built, ok = true;
  THPObjectPtr buf, segment, key, key2;
  explicit Plan(PyObject* plan) : o(plan) {
    T = (int)integer(attr(o, names.T));
    S = (int)integer(attr(o, names.S));
    kind = (int)integer(attr(o, names.kind));
    built = attr(o, names.built).get() == Py_True;
    buf = attr(o, names.buf);
    ok = plain(buf);
    if (!built) {
      segment = attr(o, names.segment);
      key = attr(o, names.seg_key);
      key2 = attr(o, names.seg_key2);
      ok = ok && plain(segment) && plain(key) && (key2.get() == Py_None || plain(key2)) &&
           (kind == SMLM_KEY_I32 || kind == SMLM_KEY_PTR2);
    }
  }
  void* ptr() { return THPVariable_Unpack(buf.get()).data_ptr(); }
  // the call builds the plan
  void build(smlm_lora_opts* opts) {
    auto at = [](THPObjectPtr& p) { return THPVariable_Unpack(p.get()).data_ptr(); };
    opts->build_seg_indptr = (const int32_t*)at(segment);
    if (kind == SMLM_KEY_PTR2) {
      opts->build_seg_key_a = (const void* const*)at(key);
      opts->build_seg_key_b = (const void* const*)at(key2);
    } else {
      opts->build_seg_adapter = (const int32_t*)at(key);
    }
  }
  void set_built() {
    if (!built && PyObject_SetAttr(o, names.built, Py_True) < 0) throw python_raised();
  }
};

// the bytes a call needs, of a Workspace or (None) of the one kept for the device and stream
Tensor scratch(PyObject* ws, size_t need, const Tensor& like) {
  THPObjectPtr buf;
  if (ws == Py_None) {
    THPObjectPtr dev(THPDevice_New(like.device()));
    buf = THPObjectPtr(PyObject_CallFunction(default_workspace, "On", dev.get(), (Py_ssize_t)need));
  } else {
    buf = attr(ws, names.ws_buf);
    if (buf.get() == Py_None || (size_t)THPVariable_Unpack(buf.get()).numel() < need) {
      THPObjectPtr n(PyLong_FromSize_t(need));
      buf = THPObjectPtr(PyObject_CallMethodObjArgs(ws, names.reserve, n.get(), nullptr));
    }
  }
  if (!buf) throw python_raised();
  const Tensor t = THPVariable_Unpack(buf.get());
  TORCH_CHECK(t.device() == like.device(), "workspace lives on ", t.device(), ", the tensors on ", like.device());
  return t;
}

// ---- the fused forward of one projection (ops._kernels.smlm_lora_forward without dropout); false: not plain ----
bool lora_forward(const Tensor& y, const Tensor& x, const Tensor& a, const Tensor& b, Plan& plan, int64_t rank,
                  const Tensor* scale, double beta, const Tensor* v, const Tensor* ranks, PyObject* ws, bool packed) {
  const int64_t n_weights = a.size(0) < b.size(0) ? a.size(0) : b.size(0);
  if (!plan.ok || !half(x) || y.scalar_type() != x.scalar_type() || !is(x, x.scalar_type(), 2) ||
      !is(y, x.scalar_type(), 2) || x.size(0) != plan.T || y.size(0) != plan.T || y.device() != x.device() || !here(x) ||
      rank <= 0 || (packed && !ranks))
    return false;
  if (plan.kind != SMLM_KEY_I32 && (a.size(0) != plan.S || b.size(0) != plan.S)) return false;
  if (scale && !(is(*scale, at::kFloat, 1) && scale->size(0) == plan.S)) return false;
  if (v && !(is(*v, x.scalar_type(), 2) && v->size(0) == plan.T && v->size(1) == rank)) return false;
  if (ranks && !(is(*ranks, at::kInt, 1) && ranks->size(0) >= n_weights)) return false;
  const int h_in = (int)x.size(1), h_out = (int)y.size(1);
  size_t need = 0;
  check(lib.fwd_size(1, plan.T, &h_in, (int)rank, &need), "smlm_lora_fwd_multi_workspace_size");
  const Tensor mem = scratch(ws, need, x);
  smlm_lora_opts opts{};
  opts.adapter_rank = ranks ? (const int32_t*)ranks->data_ptr() : nullptr;
  opts.packed_ranks = packed;
  if (!plan.built) plan.build(&opts);
  void *yp = y.data_ptr(), *vp = v ? v->data_ptr() : nullptr;
  const void* xp = x.data_ptr();
  const void* const* ap = (const void* const*)a.data_ptr();
  const void* const* bp = (const void* const*)b.data_ptr();
  int rc;
  {
    void *pp = plan.ptr(), *st = stream(x);
    NoGil no_gil;
    rc = lib.fwd(1, &yp, &xp, v ? &vp : nullptr, &ap, &bp, (int)n_weights, &h_in, &h_out, pp, mem.data_ptr(),
                 (size_t)mem.numel(), plan.T, plan.S, (int)rank, dtype_code(x), (float)beta,
                 scale ? (const float*)scale->data_ptr() : nullptr, SMLM_STAGE_SHRINK | SMLM_STAGE_EXPAND, &opts, st);
  }
  check(rc, "smlm_lora_forward");
  plan.set_built();
  return true;
}

// ---- rms_norm ----
struct RmsNorm : public Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    Tensor m = at::empty({x.size(0), 1}, x.options().dtype(at::kFloat)), o = at::empty_like(x);
    check(lib.rms_fwd(o.data_ptr(), (float*)m.data_ptr(), x.data_ptr(), w.data_ptr(), (int)x.size(0), (int)x.size(1),
                      (float)eps, dtype_code(x), stream(x)),
          "rms_norm");
    ctx->save_for_backward({x, w, m});
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w = s[1], &m = s[2];
    const Tensor g = grads[0].contiguous();
    Tensor dx = at::empty_like(x), dw = at::empty_like(w);
    check_input(dx, "dx"), check_input(dw, "dw"), check_input(g, "grad_output");
    check_input(x, "x"), check_input(w, "w"), check_input(m, "rms");
    TORCH_CHECK(g.sizes() == x.sizes(), "dx / grad_output must match x and dw must match w");
    TORCH_CHECK(w.dim() == 1 && w.size(0) == x.size(1), "w must have one entry per column of x");
    TORCH_CHECK(m.scalar_type() == at::kFloat && m.numel() == x.size(0), "rms must be float32 with one entry per row");
    TORCH_CHECK(x.scalar_type() == g.scalar_type() && w.scalar_type() == g.scalar_type(),
                "dx, dw, grad_output, x, w must share one dtype");
    TORCH_CHECK(x.device() == g.device() && w.device() == g.device() && m.device() == g.device(),
                "dx, dw, grad_output, x, w, rms must share one device");
    const int rows = (int)x.size(0), cols = (int)x.size(1);
    size_t need = 0;
    check(lib.rms_bwd_size(rows, cols, &need), "smlm_rms_norm_bwd_workspace_size");
    const Tensor mem = bytes(need, x);
    check(lib.rms_bwd(dx.data_ptr(), dw.data_ptr(), g.data_ptr(), x.data_ptr(), w.data_ptr(), (const float*)m.data_ptr(),
                      mem.data_ptr(), need, rows, cols, dtype_code(x), stream(x)),
          "rms_norm_backward");
    return {dx, dw, Tensor()};
  }
};

// ---- what the two LoRA functions' backward shares ----
struct Backward {
  Tensor g, dx;
  int rows, tail;  // rows of the plan; rows of dx when the call is to clear those past the plan's
  // x, v: as they came back from the forward, where x had h_in columns and v `rank`
  Backward(const Tensor& grad, const Tensor& x, const Tensor& v, int64_t first, int64_t rows_, int64_t h_in, int64_t rank)
      : g(grad.contiguous()), rows((int)rows_) {
    check_input(x, "x");
    TORCH_CHECK(g.size(0) >= rows && x.dim() == 2 && x.size(0) >= rows, "dy, x and dx need at least plan.T rows");
    TORCH_CHECK(x.scalar_type() == g.scalar_type() && v.scalar_type() == g.scalar_type(),
                "dx, dy, x, v must share one dtype");
    TORCH_CHECK(v.dim() == 2 && v.size(0) >= rows && v.size(1) == rank && v.is_contiguous(),
                "v must be a contiguous [>=n_rows, rank] tensor (of every projection or of none)");
    TORCH_CHECK(x.size(1) == h_in, "dx and x must have the same width");
    TORCH_CHECK(x.device() == g.device() && v.device() == g.device(), "dx, dy, x, v must share one device");
    dx = at::empty({g.size(0), x.size(1)}, g.options());
    if (first > 0) dx.narrow(0, 0, first).zero_();
    tail = rows < g.size(0) ? (int)g.size(0) : 0;
  }
  size_t need(const Tensor& x, int S, int NA, int rank) const {
    const int h_in = (int)x.size(1), h_out = (int)g.size(1);
    size_t n = 0;
    check(lib.bwd_size(1, rows, S, NA, &h_in, &h_out, rank, &n), "smlm_lora_bwd_multi_workspace_size");
    return n;
  }
  void run(const Tensor& x, const Tensor& v, void* const* da, void* const* db, const void* const* a, const void* const* b,
           const void* plan, void* ws, size_t ws_bytes, int S, int NA, int rank, const float* scale,
           smlm_lora_opts* opts) const {
    const int h_in = (int)x.size(1), h_out = (int)g.size(1);
    void* dxp = dx.data_ptr();
    const void *gp = g.data_ptr(), *xp = x.data_ptr(), *vp = v.data_ptr();
    opts->dx_rows = tail;
    check(lib.bwd(1, &dxp, &da, &db, &gp, &xp, &vp, &a, &b, plan, ws, ws_bytes, rows, S, NA, &h_in, &h_out, rank,
                  dtype_code(x), scale, opts, stream(x)),
          "smlm_lora_backward");
  }
};

// the places of a tensor's elements (the stride of a dimension of one names none)
struct Layout {
  c10::DimVector sizes, strides;
  explicit Layout(const Tensor& t) : sizes(t.sizes()), strides(t.strides()) {}
  bool of(const Tensor& t) const {
    if (t.sizes() != c10::IntArrayRef(sizes)) return false;
    for (size_t i = 0; i < sizes.size(); ++i)
      if (sizes[i] != 1 && t.stride((int64_t)i) != strides[i]) return false;
    return true;
  }
};

// ---- add_lora: everything a backward needs besides the saved tensors ----
struct AddState : torch::CustomClassHolder {
  PyObject *wa, *wb, *s;  // during the forward only
  std::vector<int64_t> tp;
  std::vector<Layout> layouts;  // of the weights
  int64_t rank, train_len, h_in, h_out;
};

struct AddLora : public Function<AddLora> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const c10::intrusive_ptr<AddState>& st,
                        at::TensorList weights) {
    const int T = (int)x.size(0), h_in = (int)x.size(1), h_out = (int)st->h_out, rank = (int)st->rank;
    const Tensor &wa = THPVariable_Unpack(st->wa), &wb = THPVariable_Unpack(st->wb), &s = THPVariable_Unpack(st->s);
    const int S = (int)s.size(0) - 1;
    Tensor y = at::empty({T, h_out}, x.options()), v = at::empty({T, rank}, x.options());
    size_t plan = 0, need = 0;
    check(lib.plan_size(T, S, &plan), "smlm_plan_size");
    check(lib.fwd_size(1, T, &h_in, rank, &need), "smlm_lora_fwd_multi_workspace_size");
    const Tensor mem = bytes(plan + 256 + need, x);  // the plan, a multiple of 256 bytes, and the scratch
    char* at_ws = (char*)mem.data_ptr() + (plan + 255) / 256 * 256;
    smlm_lora_opts opts{};
    opts.build_seg_indptr = (const int32_t*)s.data_ptr();
    const void* const* ap = (const void* const*)wa.data_ptr();
    const void* const* bp = (const void* const*)wb.data_ptr();
    opts.build_seg_key_a = ap;
    opts.build_seg_key_b = bp;
    void *yp = y.data_ptr(), *vp = v.data_ptr();
    const void* xp = x.data_ptr();
    check(lib.fwd(1, &yp, &xp, &vp, &ap, &bp, S, &h_in, &h_out, mem.data_ptr(), at_ws, need, T, S, rank, dtype_code(x),
                  0.0f, nullptr, SMLM_STAGE_SHRINK | SMLM_STAGE_EXPAND, &opts, stream(x)),
          "smlm_lora_forward");
    st->wa = st->wb = st->s = nullptr;
    variable_list saved{x.narrow(0, 0, st->train_len), v.narrow(0, 0, st->train_len)};
    saved.insert(saved.end(), weights.begin(), weights.end());
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["state"] = c10::IValue::make_capsule(st);
    return y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const auto st = c10::static_intrusive_pointer_cast<AddState>(ctx->saved_data["state"].toCapsule());
    const Tensor &x = s[0], &v = s[1];
    const int P = (int)st->tp.size() - 1, rank = (int)st->rank;
    // partitions that train the same adapter share one gradient, returned for the first of them
    std::vector<int32_t> part_adapter;
    std::vector<int> first;  // partition of each adapter
    for (int p = 0; p < P; ++p) {
      size_t a = 0;
      while (a < first.size() && !(s[2 + 2 * first[a]].data_ptr() == s[2 + 2 * p].data_ptr() &&
                                   s[3 + 2 * first[a]].data_ptr() == s[3 + 2 * p].data_ptr()))
        ++a;
      if (a == first.size()) first.push_back(p);
      part_adapter.push_back((int32_t)a);
    }
    const int NA = (int)first.size();
    const Backward call(grads[0], x, v, st->tp[0], st->tp[P], st->h_in, rank);
    for (int p = 0; p < 2 * P; ++p) {
      TORCH_CHECK(s[2 + p].device() == call.g.device() && s[2 + p].scalar_type() == call.g.scalar_type(),
                  "the weights must share dy's dtype and device");
      TORCH_CHECK(st->layouts[p].of(s[2 + p]), "the weights must come back laid out as they were saved");
    }
    variable_list out(2 + s.size() - 2);
    out[0] = call.dx;
    // addresses of dA, dB, A and B, then where the partitions start and their adapters
    std::vector<int64_t> words(4 * (size_t)NA + (2 * (size_t)P + 2) / 2);
    for (int a = 0; a < NA; ++a)
      for (int w = 0; w < 2; ++w) {
        const Tensor& weight = s[2 + 2 * first[a] + w];
        Tensor grad = at::empty_like(weight);
        words[w * NA + a] = (int64_t)grad.data_ptr();
        words[(2 + w) * NA + a] = (int64_t)weight.data_ptr();
        out[2 + 2 * first[a] + w] = std::move(grad);
      }
    int32_t* parts = (int32_t*)(words.data() + 4 * (size_t)NA);
    for (int p = 0; p <= P; ++p) parts[p] = (int32_t)st->tp[p];
    memcpy(parts + P + 1, part_adapter.data(), (size_t)P * 4);
    Tensor tab;
    const auto ints = x.options().dtype(at::kLong);
    if (words.size() * 8 > 4 * 3584) {  // (more than four launches carry)
      tab = at::from_blob(words.data(), {(int64_t)words.size()}, at::kLong).to(x.device());
    } else {
      tab = at::empty({(int64_t)words.size()}, ints);
      check(lib.put(tab.data_ptr(), words.data(), words.size() * 8, stream(x)), "put_ints");
    }
    int64_t* t = (int64_t*)tab.data_ptr();
    const int32_t* parts_at = (const int32_t*)(t + 4 * (size_t)NA);
    size_t plan = 0;
    check(lib.plan_size(call.rows, P, &plan), "smlm_plan_size");
    const size_t need = call.need(x, P, NA, rank), plan_end = (plan + 255) / 256 * 256;
    const Tensor mem = bytes(plan_end + need, x);
    smlm_lora_opts opts{};
    opts.build_seg_indptr = parts_at;
    opts.build_seg_adapter = parts_at + P + 1;
    call.run(x, v, (void* const*)t, (void* const*)(t + NA), (const void* const*)(t + 2 * NA),
             (const void* const*)(t + 3 * NA), mem.data_ptr(), (char*)mem.data_ptr() + plan_end, need, P, NA, rank, nullptr,
             &opts);
    return out;
  }
};

// ---- fused_add_lora: the step's tables stay Python's ----
struct FusedState : torch::CustomClassHolder {
  PyObject* step = nullptr;  // mixed_lora.LayerStep
  int64_t rank, h_in, first;  // first: rows before the first partition
  Tensor part_scale, train_rank;
  std::vector<int64_t> part_adapter;
  std::vector<int64_t> shape_a, shape_b;  // of all dA, all dB: [adapters, ...]
  bool packed;
  ~FusedState() override {
    if (step && Py_IsInitialized()) {
      Gil gil;
      Py_DECREF(step);
    }
  }
};

struct FusedAddLora : public Function<FusedAddLora> {
  static Tensor forward(AutogradContext* ctx, const Tensor& result, const Tensor& x, const Tensor& v,
                        const c10::intrusive_ptr<FusedState>& st, at::TensorList weights) {
    (void)v;  // (already computed, as `result` is: FusedAddLora only records)
    ctx->mark_dirty({result});
    variable_list saved{x, v};
    saved.insert(saved.end(), weights.begin(), weights.end());
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["state"] = c10::IValue::make_capsule(st);
    return result;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const auto st = c10::static_intrusive_pointer_cast<FusedState>(ctx->saved_data["state"].toCapsule());
    const Tensor &x = s[0], &v = s[1];
    variable_list out(4 + s.size() - 2);
    Gil gil;
    try {
      Plan plan(attr(st->step, names.bwd_plan));
      THPObjectPtr a_tab = attr(st->step, names.a_tab), b_tab = attr(st->step, names.b_tab);
      THPObjectPtr lay = attr(st->step, names.grad_layout), ws = attr(st->step, names.workspace);
      const Tensor &a = THPVariable_Unpack(a_tab.get()), &b = THPVariable_Unpack(b_tab.get());
      const Backward call(grads[0], x, v, st->first, plan.T, st->h_in, st->rank);
      const Tensor ga = at::empty(st->shape_a, call.g.options()), gb = at::empty(st->shape_b, call.g.options());
      // the device tables of the gradients' addresses, kept by stream and address: torch's allocator hands the same blocks
      // out step after step.  Not while a graph is recorded: a table made then holds its words from the graph's first
      // replay on, and one that was kept may be dropped before the graph is.
      auto item = [](PyObject* dict, PyObject* key) {
        PyObject* o = PyDict_GetItemWithError(dict, key);
        if (!o) {
          if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, key);
          throw python_raised();
        }
        return o;
      };
      PyObject* known = item(lay, names.grad_tabs);
      const bool keep = c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
      THPObjectPtr where(Py_BuildValue("(KKK)", (unsigned long long)ga.data_ptr(), (unsigned long long)gb.data_ptr(),
                                       (unsigned long long)stream(ga)));
      if (!where) throw python_raised();
      THPObjectPtr tabs;
      if (PyObject* hit = keep ? PyDict_GetItemWithError(known, where) : nullptr) {
        Py_INCREF(hit);
        tabs = THPObjectPtr(hit);
      } else {
        if (PyErr_Occurred()) throw python_raised();
        const Tensor& oa = THPVariable_Unpack(item(lay, names.grad_offsets_a));
        const Tensor& ob = THPVariable_Unpack(item(lay, names.grad_offsets_b));
        THPObjectPtr ta(THPVariable_Wrap(at::add(oa, (int64_t)ga.data_ptr())));
        THPObjectPtr tb(THPVariable_Wrap(at::add(ob, (int64_t)gb.data_ptr())));
        tabs = THPObjectPtr(PyTuple_Pack(2, ta.get(), tb.get()));
        if (!tabs) throw python_raised();
        if (keep && PyDict_Size(known) >= 64) PyDict_Clear(known);
        if (keep && PyDict_SetItem(known, where, tabs) < 0) throw python_raised();
      }
      const Tensor ta = THPVariable_Unpack(PyTuple_GET_ITEM(tabs.get(), 0));
      const Tensor tb = THPVariable_Unpack(PyTuple_GET_ITEM(tabs.get(), 1));
      const int NA = (int)a.size(0), rank = (int)st->rank;
      const Tensor mem = scratch(ws, call.need(x, plan.S, NA, rank), x);
      smlm_lora_opts opts{};
      if (st->train_rank.defined()) opts.adapter_rank = (const int32_t*)st->train_rank.data_ptr();
      opts.packed_ranks = st->packed;
      if (!plan.built) plan.build(&opts);
      {
        void* pp = plan.ptr();
        NoGil no_gil;
        call.run(x, v, (void* const*)ta.data_ptr(), (void* const*)tb.data_ptr(), (const void* const*)a.data_ptr(),
                 (const void* const*)b.data_ptr(), pp, mem.data_ptr(), (size_t)mem.numel(), plan.S, NA, rank,
                 st->part_scale.defined() ? (const float*)st->part_scale.data_ptr() : nullptr, &opts);
      }
      plan.set_built();
      out[0] = grads[0];
      out[1] = call.dx;
      const auto da = ga.unbind(0), db = gb.unbind(0);
      std::vector<bool> seen(da.size(), false);
      for (size_t p = 0; p < st->part_adapter.size(); ++p) {
        const int64_t ad = st->part_adapter[p];
        if (seen[ad]) continue;
        seen[ad] = true;
        out[4 + 2 * p] = da[ad];
        out[5 + 2 * p] = db[ad];
      }
    } catch (const python_raised&) {
      python_error e;
      e.persist();
      throw std::move(e);
    }
    return out;
  }
};

// ------------------------------------------------------------------ entries --
#define SMLM_PY_TRY HANDLE_TH_ERRORS try {
#define SMLM_PY_END                    \
  }                                    \
  catch (const python_raised&) {       \
    return nullptr;                    \
  }                                    \
  END_HANDLE_TH_ERRORS

// forward(y, x, a_ptrs, b_ptrs, plan, rank, seg_scale, beta, v_out, adapter_rank, workspace, packed) -> whether it was done
PyObject* py_forward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  SMLM_PY_TRY
  TORCH_CHECK(n == 12, "forward takes 12 arguments");
  bool ok = plain_thread() && plain(p[0]) && plain(p[1]) && plain(p[2]) && plain(p[3]);
  const Tensor *scale = optional(p[6], &ok), *v = optional(p[8], &ok), *ranks = optional(p[9], &ok);
  if (!ok) Py_RETURN_FALSE;
  const Tensor &y = THPVariable_Unpack(p[0]), &x = THPVariable_Unpack(p[1]), &a = THPVariable_Unpack(p[2]),
               &b = THPVariable_Unpack(p[3]);
  if (!is(a, at::kLong, 1) || !is(b, at::kLong, 1)) Py_RETURN_FALSE;
  Plan plan(p[4]);
  const double beta = PyFloat_AsDouble(p[7]);
  if (beta == -1.0 && PyErr_Occurred()) throw python_raised();
  const int packed = PyObject_IsTrue(p[11]);
  if (lora_forward(y, x, a, b, plan, integer(p[5]), scale, beta, v, ranks, p[10], packed == 1)) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
  SMLM_PY_END
}

// rms_norm(x, w, eps) -> output, or None
PyObject* py_rms_norm(PyObject*, PyObject* const* p, Py_ssize_t n) {
  SMLM_PY_TRY
  if (n < 2 || n > 3 || !plain_thread() || !plain(p[0]) || !plain(p[1])) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(p[0]), &w = THPVariable_Unpack(p[1]);
  if (!half(x) || !is(x, x.scalar_type(), 2) || !is(w, x.scalar_type(), 1) || w.size(0) != x.size(1) || x.size(0) == 0 ||
      x.size(1) % 8 != 0 || x.size(1) == 0 || x.device() != w.device() || !here(x))
    Py_RETURN_NONE;
  double eps = 1e-6;
  if (n == 3) eps = PyFloat_AsDouble(p[2]);
  if (eps == -1.0 && PyErr_Occurred()) throw python_raised();
  Tensor o;
  {
    NoGil no_gil;
    o = RmsNorm::apply(x, w, eps);
  }
  return THPVariable_Wrap(std::move(o));
  SMLM_PY_END
}

// add_lora(y_shape, x, wa_ptr, wb_ptr, s, lora_rank, train_len, train_partition, *weights) -> output, or None
PyObject* py_add_lora(PyObject*, PyObject* const* p, Py_ssize_t n) {
  SMLM_PY_TRY
  const Py_ssize_t n_weights = n - 8;
  if (n_weights < 2 || n_weights % 2 != 0 || !plain_thread()) Py_RETURN_NONE;
  for (int i = 1; i <= 4; ++i)
    if (!plain(p[i])) Py_RETURN_NONE;
  variable_list weights;
  weights.reserve(n_weights);
  for (Py_ssize_t i = 0; i < n_weights; ++i) {
    if (!plain(p[8 + i])) Py_RETURN_NONE;
    weights.push_back(THPVariable_Unpack(p[8 + i]));
  }
  const Tensor &x = THPVariable_Unpack(p[1]), &wa = THPVariable_Unpack(p[2]), &wb = THPVariable_Unpack(p[3]),
               &s = THPVariable_Unpack(p[4]);
  auto st = c10::make_intrusive<AddState>();
  if (!PyTuple_Check(p[0]) || PyTuple_GET_SIZE(p[0]) != 2 || !half(x) || !is(x, x.scalar_type(), 2) || !here(x) ||
      !is(s, at::kInt, 1) || s.size(0) < 2 || !is(wa, at::kLong, 1) || !is(wb, at::kLong, 1) ||
      wa.size(0) != s.size(0) - 1 || wb.size(0) != s.size(0) - 1 || s.device() != x.device())
    Py_RETURN_NONE;
  st->h_in = x.size(1);
  st->h_out = integer(PyTuple_GET_ITEM(p[0], 1));
  st->rank = integer(p[5]);
  st->train_len = integer(p[6]);
  if (integer(PyTuple_GET_ITEM(p[0], 0)) != x.size(0) || st->h_out <= 0 || st->rank <= 0 || st->train_len <= 0 ||
      st->train_len > x.size(0))
    Py_RETURN_NONE;
  THPObjectPtr tp(PySequence_Fast(p[7], "train_partition must be a sequence"));
  if (!tp) throw python_raised();
  Py_ssize_t parts = PySequence_Fast_GET_SIZE(tp.get()) - 1;
  if (parts > n_weights / 2) parts = n_weights / 2;
  for (Py_ssize_t i = 0; i <= parts; ++i) st->tp.push_back(integer(PySequence_Fast_GET_ITEM(tp.get(), i)));
  if (parts < 1 || st->tp[parts] <= 0 || st->tp[parts] > st->train_len) Py_RETURN_NONE;
  for (const Tensor& w : weights)
    if (w.device() != x.device() || w.scalar_type() != x.scalar_type()) Py_RETURN_NONE;
  st->layouts.reserve(2 * parts);
  for (Py_ssize_t i = 0; i < 2 * parts; ++i) st->layouts.emplace_back(weights[i]);
  st->wa = p[2], st->wb = p[3], st->s = p[4];
  Tensor y;
  {
    NoGil no_gil;
    y = AddLora::apply(x, st, at::TensorList(weights));
  }
  return THPVariable_Wrap(std::move(y));
  SMLM_PY_END
}

// fused_add_lora(result, x, step, *weights) -> result, or None
PyObject* py_fused_add_lora(PyObject*, PyObject* const* p, Py_ssize_t n) {
  SMLM_PY_TRY
  const Py_ssize_t n_weights = n - 3;
  if (n_weights < 2 || n_weights % 2 != 0 || !plain_thread() || !plain(p[0]) || !plain(p[1])) Py_RETURN_NONE;
  variable_list weights;
  weights.reserve(n_weights);
  for (Py_ssize_t i = 0; i < n_weights; ++i) {
    if (!plain(p[3 + i])) Py_RETURN_NONE;
    weights.push_back(THPVariable_Unpack(p[3 + i]));
  }
  PyObject* step = p[2];
  THPObjectPtr lay = attr(step, names.grad_layout), bwd = attr(step, names.bwd_plan),
                     drop = attr(step, names.dropout), segs = attr(step, names.part_segments),
                     ranks_o = attr(step, names.adapter_rank), scale_o = attr(step, names.seg_scale);
  if (lay.get() == Py_None || bwd.get() == Py_None || drop.get() != Py_None || segs.get() == Py_None ||
      !PyDict_Check(lay.get()))
    Py_RETURN_NONE;
  PyObject* uniform = PyDict_GetItemWithError(lay, names.grad_uniform);
  if (!uniform || uniform == Py_None) {
    if (PyErr_Occurred()) throw python_raised();
    Py_RETURN_NONE;
  }
  auto st = c10::make_intrusive<FusedState>();
  Py_INCREF(step);
  st->step = step;
  st->rank = integer(attr(step, names.rank));
  st->packed = PyObject_IsTrue(attr(step, names.packed)) == 1;
  THPObjectPtr pa(PySequence_Fast(attr(step, names.part_adapter), "part_adapter must be a sequence"));
  if (!pa) throw python_raised();
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(pa.get()); ++i)
    st->part_adapter.push_back(integer(PySequence_Fast_GET_ITEM(pa.get(), i)));
  const int64_t NA = integer(PyTuple_GET_ITEM(uniform, 0));
  auto shape = [&](PyObject* t) {
    return std::vector<int64_t>{NA, integer(PyTuple_GET_ITEM(t, 0)), integer(PyTuple_GET_ITEM(t, 1))};
  };
  st->shape_a = shape(PyTuple_GET_ITEM(uniform, 1));
  st->shape_b = shape(PyTuple_GET_ITEM(uniform, 2));
  Plan plan(attr(step, names.plan));
  Plan bplan(bwd);
  THPObjectPtr tp = attr(step, names.train_partition), wa_o = attr(step, names.wa_table),
                     wb_o = attr(step, names.wb_table), ws = attr(step, names.workspace), a_tab = attr(step, names.a_tab),
                     b_tab = attr(step, names.b_tab);
  {
    THPObjectPtr first(PySequence_GetItem(tp, 0));
    if (!first) throw python_raised();
    st->first = integer(first);
  }
  bool ok = true;
  const Tensor* scale = optional(scale_o, &ok);
  const Tensor* ranks = nullptr;
  if (ranks_o.get() != Py_None) {
    if (!PyTuple_Check(ranks_o.get()) || PyTuple_GET_SIZE(ranks_o.get()) != 2) Py_RETURN_NONE;
    ranks = optional(PyTuple_GET_ITEM(ranks_o.get(), 0), &ok);
    const Tensor* train = optional(PyTuple_GET_ITEM(ranks_o.get(), 1), &ok);
    if (!ok || !train || !is(*train, at::kInt, 1) || train->size(0) < NA) Py_RETURN_NONE;
    st->train_rank = *train;
  }
  const Tensor &result = THPVariable_Unpack(p[0]), &x = THPVariable_Unpack(p[1]);
  ok = ok && plain(wa_o) && plain(wb_o) && plain(a_tab) && plain(b_tab) && bplan.ok && bplan.kind == SMLM_KEY_I32 &&
       ws.get() != Py_None && bplan.T > 0 && bplan.T <= plan.T && bplan.S == (int)st->part_adapter.size() &&
       2 * (Py_ssize_t)st->part_adapter.size() <= n_weights && integer(attr(step, names.train_len)) > 0;
  for (const int64_t ad : st->part_adapter) ok = ok && ad >= 0 && ad < NA;
  if (!ok) Py_RETURN_NONE;
  const Tensor &wa = THPVariable_Unpack(wa_o.get()), &wb = THPVariable_Unpack(wb_o.get()),
               &at_ = THPVariable_Unpack(a_tab.get()), &bt_ = THPVariable_Unpack(b_tab.get());
  if (!is(wa, at::kLong, 1) || !is(wb, at::kLong, 1) || !is(at_, at::kLong, 1) || !is(bt_, at::kLong, 1) ||
      at_.size(0) != NA || bt_.size(0) != NA || x.dim() != 2 || result.dim() != 2)
    Py_RETURN_NONE;
  // what autograd would refuse is left to the general path, which refuses it before anything is computed
  if (at::GradMode::is_enabled() && (result.requires_grad() && result.is_leaf())) Py_RETURN_NONE;
  if (result.is_inference() || x.is_inference()) Py_RETURN_NONE;
  st->h_in = x.size(1);
  const Tensor v = at::empty({x.size(0), st->rank}, x.options());
  if (scale) {
    THPObjectPtr g(PyObject_CallMethodObjArgs(step, names.gather, scale_o.get(), segs.get(), nullptr));
    if (!g) throw python_raised();
    st->part_scale = THPVariable_Unpack(g.get());
    if (!is(st->part_scale, at::kFloat, 1) || st->part_scale.size(0) != bplan.S) Py_RETURN_NONE;
  }
  if (!lora_forward(result, x, wa, wb, plan, st->rank, scale, 1.0, &v, ranks, ws, st->packed)) Py_RETURN_NONE;
  Tensor out;
  {
    NoGil no_gil;
    out = FusedAddLora::apply(result, x, v, st, at::TensorList(weights));
  }
  return THPVariable_Wrap(std::move(out));
  SMLM_PY_END
}

// bind({entry: address}, default_workspace)
PyObject* py_bind(PyObject*, PyObject* args) {
  SMLM_PY_TRY
  PyObject *addr, *ws;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &addr, &ws)) return nullptr;
  auto get = [&](const char* name, auto* f) {
    PyObject* o = PyDict_GetItemString(addr, name);
    TORCH_CHECK(o, name, " is missing");
    *f = reinterpret_cast<std::remove_pointer_t<decltype(f)>>(PyLong_AsVoidPtr(o));
    if (PyErr_Occurred()) throw python_raised();
  };
  get("smlm_strerror", &lib.strerror);
  get("smlm_plan_size", &lib.plan_size);
  get("smlm_lora_fwd_multi_workspace_size", &lib.fwd_size);
  get("smlm_lora_fwd_multi_ex", &lib.fwd);
  get("smlm_lora_bwd_multi_workspace_size", &lib.bwd_size);
  get("smlm_lora_bwd_multi_ex", &lib.bwd);
  get("smlm_rms_norm_fwd", &lib.rms_fwd);
  get("smlm_rms_norm_bwd_workspace_size", &lib.rms_bwd_size);
  get("smlm_rms_norm_bwd", &lib.rms_bwd);
  get("smlm_put_words", &lib.put);
  Py_INCREF(ws);
  Py_XSETREF(default_workspace, ws);
  Py_RETURN_NONE;
  SMLM_PY_END
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"forward", (PyCFunction)(void (*)(void))py_forward, METH_FASTCALL, nullptr},
    {"rms_norm", (PyCFunction)(void (*)(void))py_rms_norm, METH_FASTCALL, nullptr},
    {"add_lora", (PyCFunction)(void (*)(void))py_add_lora, METH_FASTCALL, nullptr},
    {"fused_add_lora", (PyCFunction)(void (*)(void))py_fused_add_lora, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_smlm_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__smlm_host(void) {
  auto s = [](const char* n) { return PyUnicode_InternFromString(n); };
  names = {s("T"), s("S"), s("kind"), s("built"), s("buf"), s("segment"), s("seg_key"), s("seg_key2"), s("_buf"),
           s("reserve"), s("workspace"), s("packed"), s("wa_table"), s("wb_table"), s("seg_scale"), s("plan"), s("rank"),
           s("train_len"), s("train_partition"), s("dropout"), s("adapter_rank"), s("part_segments"), s("bwd_plan"),
           s("part_adapter"), s("a_tab"), s("b_tab"), s("grad_layout"), s("gather"), s("grad_uniform"), s("grad_tabs"),
           s("grad_offsets_a"), s("grad_offsets_b")};
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
