// The operator's call from Python in native code: tensors in, one acct_fa_fwd, outputs and (where a gradient is asked for)
// an autograd node whose backward is one acct_fa_bwd.  Built as acctransformer_amd/_native.so, host code only.
//
// A step on small inputs is bound by the host: with a Python autograd function and ctypes calls the (4, 8, 128, 80) training
// step took 121 us for 28 us of kernels, now 71 (44 are torch's own for a step of one built-in operator: the hand-over to the
// autograd thread and back), a (1, 4, 512, 64) forward 13.4, now 8.2 (us).  A mask tensor that is new in every step still has its
// record made in Python: 209 us and 162.  A backward here runs without the interpreter lock.  Calls that are not plain --
// transforms, tracing, forward mode, tensor subclasses, side inputs that ask for a gradient -- and whatever this file does not
// recognise stay with the Python function (flash_attention_impl.py), which also words the errors.
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/dynamo/compiled_autograd.h>
#include <torch/csrc/PyInterpreter.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/SafePyObject.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <array>
#include <cstring>
#include <mutex>

#include "../../include/acct_fa.h"

namespace {

using at::Tensor;

// the library's entry points, as the Python binding loaded them (one library in the process, whichever file it came from)
struct Library {
  decltype(&acct_fa_fwd) fwd;
  decltype(&acct_fa_bwd) bwd;
  decltype(&acct_fa_fwd_split_workspace_bytes) fwd_workspace_bytes;
  decltype(&acct_fa_bwd_workspace_bytes) bwd_workspace_bytes;
  decltype(&acct_fa_drop_bits_bytes) drop_bits_bytes;
  decltype(&acct_last_error) last_error;
} g_lib;
PyObject* g_error = nullptr;         // AcctError
PyObject* g_params_view = nullptr;   // (bytes of acct_fa_params, tensors, mask_bits entry) -> AcctFaParams

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// runs with the interpreter lock held
void set_error(int rc) {
  PyObject* e = PyObject_CallFunction(g_error, "is", rc, g_lib.last_error());
  if (!e) return;
  PyErr_SetObject(g_error, e);
  Py_DECREF(e);
}

void take_strides(const Tensor& t, int64_t (&s)[3]) {
  for (int i = 0; i < 3; i++) s[i] = t.stride(i);
  if (!s[0] && !s[1] && !s[2]) s[2] = t.size(3);       // one row for all (to the library, three zeros are a contiguous tensor)
}

// One call: its parameters without addresses, and the tensors beside q, k, v that they go with.
struct Problem {
  acct_fa_params p{};
  Tensor mask, drop, alibi, mask_bits, drop_bits;

  std::array<Tensor*, 5> tensors() { return {&mask, &drop, &alibi, &mask_bits, &drop_bits}; }
  std::array<const Tensor*, 5> tensors() const { return {&mask, &drop, &alibi, &mask_bits, &drop_bits}; }
  void point(const Tensor& q, const Tensor& k, const Tensor& v) {
    auto at = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
    p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr();
    take_strides(q, p.q_stride); take_strides(k, p.k_stride); take_strides(v, p.v_stride);
    p.attn_mask = at(mask); p.drop_mask = at(drop); p.alibi = at(alibi);
    p.mask_bits = at(mask_bits); p.drop_bits = at(drop_bits);
  }
};

Tensor bytes_like(const Tensor& like, size_t n) {
  return n ? at::empty({(int64_t)n}, like.options().dtype(at::kByte)) : Tensor();
}

// Makes `t` a copy of it where elements may share memory (an expanded operand): its gradient has the same layout and needs a
// place of its own for every element.  A copy also where rows are further apart than the library's backward takes.
constexpr int64_t kRowStrideEnd = 34087040, kFwdRowStrideEnd = 16909320;
void take_apart(Tensor& t) {
  bool apart = t.stride(2) < kRowStrideEnd;
  if (apart && t.is_non_overlapping_and_dense()) return;
  std::array<std::pair<int64_t, int64_t>, 4> dims;
  for (int i = 0; i < 4; i++) dims[i] = {t.stride(i), t.size(i)};
  std::sort(dims.begin(), dims.end());
  int64_t room = 1;
  for (const auto& [stride, size] : dims) {
    if (size <= 1) continue;
    apart = apart && stride >= room;
    room += stride * (size - 1);
  }
  if (!apart) t = t.contiguous();
}

struct FlashAttentionBackward : public torch::autograd::Node {
  Problem problem;
  std::shared_ptr<c10::SafePyObject> entry;    // the operator's record of the mask_bits buffer, for `params`
  torch::autograd::SavedVariable q_, k_, v_, o_, lse_;

  std::string name() const override { return "_FlashAttentionFnBackward"; }
  // what a reader on another thread sees while a backward ends (called with the interpreter lock, waits without it)
  std::pair<Problem, std::shared_ptr<c10::SafePyObject>> record() {
    pybind11::gil_scoped_release free_python;
    std::lock_guard<std::mutex> lock(mutex_);
    return {problem, entry};
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* s : {&q_, &k_, &v_, &o_, &lse_}) s->reset_data();
    // (no backward can follow, and whoever still holds an output would hold the keep bits of its dropout with it)
    problem = Problem{problem.p};
    acct_fa_params& p = problem.p;
    p.q = p.k = p.v = p.attn_mask = p.drop_mask = p.alibi = nullptr;
    p.mask_bits = p.drop_bits = nullptr;
    entry.reset();
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    return backward(problem, q_.unpack(), k_.unpack(), v_.unpack(), o_.unpack(shared_from_this()), lse_.unpack(), grads[0]);
  }
  // Compiled autograd records the backward as a call of `compiled`, with the tensors and (as one more of them) the parameters
  // as its arguments.
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override {
    for (const auto* s : {&q_, &k_, &v_, &lse_}) args.collect(*s, false);
    args.collect(o_, true);
    params_ = at::empty({(int64_t)sizeof(acct_fa_params)}, at::kByte);
    std::memcpy(params_.data_ptr(), &problem.p, sizeof(acct_fa_params));
    args.collect(params_);
    for (const Tensor* t : problem.tensors()) args.collect(*t);
  }
  torch::autograd::variable_list apply_with_saved(const torch::autograd::variable_list& grads,
                                                  torch::dynamo::autograd::SwapSavedVariables& saved) override {
    using namespace torch::dynamo::autograd;
    for (auto* s : {&q_, &k_, &v_, &lse_, &o_}) saved.before(*s);
    saved.before(params_);
    for (Tensor* t : problem.tensors()) saved.before(*t);
    PackedArgs args;
    for (const Tensor& t : {q_.unpack(), k_.unpack(), v_.unpack(), o_.unpack(shared_from_this()), lse_.unpack(), params_}) args.pack(t);
    for (Tensor* t : problem.tensors()) args.pack(t->defined() ? *t : params_);      // (absent: null in the parameters, and not looked at)
    const auto& compiler = getPyCompilerInterface();
    const std::string fn = compiler->bind_function(saved.get_py_compiler(), name(), compiled,
                                                   std::vector<at::TypePtr>(11, at::TensorType::get()), true, false);
    auto metadata = IValuePacker<std::vector<std::optional<torch::autograd::InputMetadata>>>::pack(get_input_metadata(next_edges()));
    auto out = compiler->call_function(saved.get_py_compiler(), "apply_functional", fn, grads, args.vec(), metadata);
    for (auto* s : {&q_, &k_, &v_, &lse_, &o_}) saved.after(*s);
    saved.after(params_);
    for (Tensor* t : problem.tensors()) saved.after(*t);
    return out;
  }

 private:
  mutable Tensor params_;

  static torch::autograd::variable_list compiled(const torch::autograd::variable_list& grads, const std::vector<c10::IValue>& a) {
    Problem c;
    const Tensor params = a[5].toTensor();
    std::memcpy(&c.p, params.data_ptr(), sizeof(c.p));
    const void* there[] = {c.p.attn_mask, c.p.drop_mask, c.p.alibi, c.p.mask_bits, c.p.drop_bits};
    auto side = c.tensors();
    for (int i = 0; i < 5; i++)
      if (there[i]) *side[i] = a[6 + i].toTensor();
    return backward(c, a[0].toTensor(), a[1].toTensor(), a[2].toTensor(), a[3].toTensor(), a[4].toTensor(), grads[0]);
  }

  static torch::autograd::variable_list backward(Problem c, Tensor q, Tensor k, Tensor v, Tensor o, const Tensor& lse, Tensor dout) {
    c10::DeviceGuard device(q.device());
    at::AutoDispatchBelowADInplaceOrView below;
    take_apart(q); take_apart(k); take_apart(v);
    if (o.stride(2) >= kRowStrideEnd) o = o.contiguous();
    if (!dout.defined()) dout = at::zeros_like(o);
    if (dout.strides() != o.strides()) {       // the kernels read dO with O's strides
      Tensor t = at::empty_strided(o.sizes(), o.strides(), o.options());
      t.copy_(dout);
      dout = t;
    }
    c.point(q, k, v);                          // (a backward may run twice, and on other copies of the saved tensors)
    take_strides(o, c.p.o_stride);
    Tensor dq = at::empty_strided(q.sizes(), q.strides(), q.options()), dk = at::empty_strided(k.sizes(), k.strides(), k.options()),
           dv = at::empty_strided(v.sizes(), v.strides(), v.options());
    const size_t n = g_lib.bwd_workspace_bytes(&c.p);
    const Tensor ws = bytes_like(q, n);
    const int rc = g_lib.bwd(&c.p, o.data_ptr(), dout.data_ptr(), lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                             n ? ws.data_ptr() : nullptr, n, stream_of(q));
    if (rc != ACCT_OK) {
      pybind11::gil_scoped_acquire lock_python;
      set_error(rc);
      python_error e;
      e.persist();
      throw std::move(e);
    }
    return {dq, dk, dv};
  }
};

FlashAttentionBackward* node_of(PyObject* self) {
  return static_cast<FlashAttentionBackward*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get());
}

PyObject* get_params(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  const auto [c, entry] = node_of(self)->record();
  THPObjectPtr tensors(PyList_New(0));
  if (!tensors) return nullptr;
  for (const Tensor* t : c.tensors())
    if (t->defined()) {
      THPObjectPtr w(THPVariable_Wrap(*t));
      if (!w || PyList_Append(tensors.get(), w.get())) return nullptr;
    }
  THPObjectPtr raw(PyBytes_FromStringAndSize(reinterpret_cast<const char*>(&c.p), sizeof(c.p)));
  if (!raw) return nullptr;
  PyObject* e = entry ? entry->ptr(getPyInterpreter()) : Py_None;
  return PyObject_CallFunctionObjArgs(g_params_view, raw.get(), tensors.get(), e, nullptr);
  END_HANDLE_TH_ERRORS
}

PyObject* get_drop_bits(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  const Tensor t = node_of(self)->record().first.drop_bits;
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
  END_HANDLE_TH_ERRORS
}

PyObject* get_saved_tensors(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  FlashAttentionBackward* n = node_of(self);
  const Tensor saved[] = {n->q_.unpack(), n->k_.unpack(), n->v_.unpack(), n->o_.unpack(n->shared_from_this()), n->lse_.unpack()};
  THPObjectPtr out(PyTuple_New(5));
  if (!out) return nullptr;
  for (int i = 0; i < 5; i++) {
    PyObject* w = THPVariable_Wrap(saved[i]);
    if (!w) return nullptr;
    PyTuple_SET_ITEM(out.get(), i, w);
  }
  return out.release();
  END_HANDLE_TH_ERRORS
}

using torch::autograd::THPCppFunction_input_metadata;
using torch::autograd::THPCppFunction_metadata;
using torch::autograd::THPCppFunction_next_functions;
using torch::autograd::THPCppFunction_requires_grad;
PyGetSetDef g_node_properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                   {"params", get_params, nullptr, nullptr, nullptr},
                                   {"drop_bits", get_drop_bits, nullptr, nullptr, nullptr},
                                   {"saved_tensors", get_saved_tensors, nullptr, nullptr, nullptr},
                                   {nullptr}};
PyTypeObject g_node_type;

// a tensor argument, or an undefined tensor for None; false for anything else
bool tensor_arg(PyObject* a, Tensor& t) {
  if (a == Py_None) return true;
  if (!THPVariable_CheckExact(a)) return false;
  t = THPVariable_Unpack(a);
  return true;
}

// Shapes, dtypes and layouts that the library's Python binding accepts; false leaves the call to it.
bool describe(Problem& c, const Tensor& q, const Tensor& k, const Tensor& v) {
  acct_fa_params& p = c.p;
  const auto dt = q.scalar_type();
  if (dt != at::kHalf && dt != at::kBFloat16) return false;
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || k.scalar_type() != dt || v.scalar_type() != dt) return false;
  const int64_t B = q.size(0), N = q.size(1), Sq = q.size(2), D = q.size(3), Sk = k.size(2);
  for (int64_t x : {B, N, Sq, Sk, D})
    if (x > INT32_MAX) return false;
  for (const Tensor* t : {&q, &k, &v})
    if (t->size(2) > 1 && t->stride(0) == 0 && t->stride(1) == 0 && t->stride(2) == 0) return false;    // (refused there)
  if (k.size(0) != B || k.size(1) != N || k.size(3) != D || v.sizes() != k.sizes()) return false;
  const Tensor* all[] = {&q, &k, &v, &c.mask, &c.drop, &c.alibi, &c.mask_bits};
  for (const Tensor* t : all)
    if (t->defined() && (!t->device().is_cuda() || t->device() != q.device() || t->layout() != at::kStrided)) return false;
  p.dtype = dt == at::kHalf ? ACCT_F16 : ACCT_BF16;
  p.B = (int)B; p.N = (int)N; p.Sq = (int)Sq; p.Sk = (int)Sk; p.D = (int)D;
  const bool dense = p.mask_kind == ACCT_MASK_DENSE_U8 || p.mask_kind == ACCT_MASK_DENSE_F16;
  const bool tile = p.mask_kind == ACCT_MASK_TILE_U8 || p.mask_kind == ACCT_MASK_TILE_F16;
  if ((dense || tile) != c.mask.defined()) return false;
  if (dense || tile) {
    const auto want = p.mask_kind == ACCT_MASK_DENSE_U8 || p.mask_kind == ACCT_MASK_TILE_U8 ? at::kByte : dt;
    if (c.mask.scalar_type() != want || !c.mask.is_contiguous()) return false;
    if (dense) {
      if (c.mask.dim() != 3 || c.mask.size(1) != Sq || c.mask.size(2) != Sk || (c.mask.size(0) != 1 && c.mask.size(0) != B)) return false;
      p.mask_stride_b = c.mask.size(0) == 1 ? 0 : Sq * Sk;
    } else if (c.mask.numel() != 128 * 128) {
      return false;
    }
  }
  if (c.drop.defined()) {
    if (p.drop_philox || (c.drop.scalar_type() != at::kByte && c.drop.scalar_type() != dt) || !c.drop.is_contiguous() || c.drop.dim() != 4 ||
        c.drop.size(0) != B || c.drop.size(1) != N || c.drop.size(2) != Sq || c.drop.size(3) != Sk)
      return false;
    p.drop_mask_kind = c.drop.scalar_type() == at::kByte ? ACCT_DROP_U8 : ACCT_DROP_F16;
  }
  if (c.alibi.defined()) {
    const Tensor& a = c.alibi;
    if (a.scalar_type() != dt || a.dim() != 4 || a.size(3) != Sk || a.stride(3) != 1) return false;
    if ((a.size(0) != 1 && a.size(0) != B) || (a.size(1) != 1 && a.size(1) != N) || (a.size(2) != 1 && a.size(2) != Sq)) return false;
    p.alibi_stride_b = a.size(0) == 1 ? 0 : a.stride(0);
    p.alibi_stride_h = a.size(1) == 1 ? 0 : a.stride(1);
    p.alibi_stride_q = a.size(2) == 1 ? 0 : a.stride(2);
  }
  return true;
}

// forward(record, q, k, v, mask_kind, mask, mask_bits, mask_bits_filled, entry, drop, seed, offset, philox, alibi, prev, next,
// scale, keep_prob, row_prefix) -> (O, LSE), or None for a call that the Python side has to look at
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 19) {
    PyErr_SetString(PyExc_TypeError, "forward takes 19 arguments");
    return nullptr;
  }
  const bool record = *a++ == Py_True;
  Tensor q, k, v;
  Problem c;
  if (!tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !q.defined() || !k.defined() || !v.defined()) Py_RETURN_NONE;
  if (!tensor_arg(a[4], c.mask) || !tensor_arg(a[5], c.mask_bits) || !tensor_arg(a[8], c.drop) || !tensor_arg(a[12], c.alibi)) Py_RETURN_NONE;
  acct_fa_params& p = c.p;
  p.mask_kind = (int)PyLong_AsLong(a[3]);
  p.mask_bits_filled = PyObject_IsTrue(a[6]);
  p.drop_seed = PyLong_AsUnsignedLongLong(a[9]);
  p.drop_offset = (uint32_t)PyLong_AsUnsignedLong(a[10]);
  p.drop_philox = PyObject_IsTrue(a[11]);
  auto block = [](PyObject* x) {
    int over = 0;
    const long long b = PyLong_AsLongLongAndOverflow(x, &over);
    return (int)(over > 0 || b > ACCT_BLOCK_UNBOUNDED ? ACCT_BLOCK_UNBOUNDED : over < 0 || b < INT32_MIN ? INT32_MIN : b);
  };
  p.prev_block_num = block(a[13]);
  p.next_block_num = block(a[14]);
  p.scale = (float)PyFloat_AsDouble(a[15]);
  p.keep_prob = (float)PyFloat_AsDouble(a[16]);
  const long prefix = PyLong_AsLong(a[17]);
  if (PyErr_Occurred()) return nullptr;
  if (prefix > INT32_MAX || prefix < INT32_MIN) Py_RETURN_NONE;
  p.row_block_prefix = (int)prefix;
  if (!q.device().is_cuda() || !k.device().is_cuda() || !v.device().is_cuda() || q.dim() != 4 || k.dim() != 4 || v.dim() != 4) Py_RETURN_NONE;

  Tensor o, lse;
  std::shared_ptr<FlashAttentionBackward> node;
  int rc = ACCT_OK;
  bool known = true;
  {
    pybind11::gil_scoped_release free_python;
    if (record) {
      node = std::shared_ptr<FlashAttentionBackward>(new FlashAttentionBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
    }
    {
      c10::DeviceGuard device(q.device());
      at::AutoDispatchBelowADInplaceOrView below;
      auto rows = [](Tensor& t) { if (t.stride(3) != 1 || (t.stride(2) >= kFwdRowStrideEnd && t.size(2) >= 64)) t = t.contiguous(); };
      rows(q); rows(k); rows(v);
      known = describe(c, q, k, v) && (q.stride(3) == 1 || q.size(3) == 1);
      if (known) {
        o = at::empty_like(q);
        lse = at::empty({p.B, p.N, p.Sq}, q.options().dtype(at::kFloat));
        c.point(q, k, v);
        take_strides(o, p.o_stride);
        if (record) {
          // with dropout, the keep bits the forward packs (or draws) are kept for the backward of this step
          c.drop_bits = bytes_like(q, g_lib.drop_bits_bytes(&p));
          if (c.drop_bits.defined()) {
            p.drop_bits = c.drop_bits.data_ptr();
            p.drop_mask_kind |= ACCT_DROP_BITS_ONE_BAND;     // (the backward runs on these very parameters)
          }
        }
        const size_t bytes = g_lib.fwd_workspace_bytes(&p);
        const Tensor ws = bytes_like(q, bytes);
        rc = g_lib.fwd(&p, o.data_ptr(), lse.data_ptr<float>(), bytes ? ws.data_ptr() : nullptr, bytes, stream_of(q));
      }
    }
    if (known && rc == ACCT_OK && record) {
      p.mask_bits_filled = p.mask_bits != nullptr;
      p.drop_bits_filled = p.drop_bits != nullptr;
      node->problem = c;
      torch::autograd::set_history(o, node);
      node->q_ = torch::autograd::SavedVariable(q, false);
      node->k_ = torch::autograd::SavedVariable(k, false);
      node->v_ = torch::autograd::SavedVariable(v, false);
      node->o_ = torch::autograd::SavedVariable(o, true);
      node->lse_ = torch::autograd::SavedVariable(lse, false);
    }
  }
  if (!known) Py_RETURN_NONE;
  if (rc != ACCT_OK) {
    set_error(rc);
    return nullptr;
  }
  if (node && a[7] != Py_None) {
    Py_INCREF(a[7]);
    node->entry = std::make_shared<c10::SafePyObject>(a[7], getPyInterpreter());
  }
  THPObjectPtr out(PyTuple_New(2));
  if (!out) return nullptr;
  PyObject* w = THPVariable_Wrap(o);
  if (!w) return nullptr;
  PyTuple_SET_ITEM(out.get(), 0, w);
  w = THPVariable_Wrap(lse);
  if (!w) return nullptr;
  PyTuple_SET_ITEM(out.get(), 1, w);
  return out.release();
  END_HANDLE_TH_ERRORS
}

// setup(AcctError, view of the parameters, address of each entry point in the order of `Library`)
PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "setup takes 8 arguments");
    return nullptr;
  }
  void* at[6];
  for (int i = 0; i < 6; i++) {
    at[i] = PyLong_AsVoidPtr(a[2 + i]);
    if (PyErr_Occurred()) return nullptr;
  }
  auto take = [](auto& f, void* p) { f = reinterpret_cast<std::decay_t<decltype(f)>>(p); };
  take(g_lib.fwd, at[0]); take(g_lib.bwd, at[1]); take(g_lib.fwd_workspace_bytes, at[2]);
  take(g_lib.bwd_workspace_bytes, at[3]); take(g_lib.drop_bits_bytes, at[4]); take(g_lib.last_error, at[5]);
  Py_INCREF(a[0]); Py_INCREF(a[1]);
  g_error = a[0];
  g_params_view = a[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {{"forward", (PyCFunction)(void (*)())forward, METH_FASTCALL, "one call of the operator"},
                           {"setup", (PyCFunction)(void (*)())setup, METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  // torch's classes are compiled in: another version has other layouts, which a symbol that still resolves does not show
  THPObjectPtr torch(PyImport_ImportModule("torch"));
  THPObjectPtr version(torch ? PyObject_GetAttrString(torch.get(), "__version__") : nullptr);
  if (!version) return nullptr;
  THPObjectPtr text(PyObject_Str(version.get()));
  const char* now = text ? PyUnicode_AsUTF8(text.get()) : nullptr;
  if (!now) return nullptr;
  if (strcmp(now, ACCT_TORCH)) return PyErr_Format(PyExc_ImportError, "built for torch %s, this is torch %s", ACCT_TORCH, now);
  torch::autograd::_initFunctionPyTypeObject(g_node_type, "acctransformer_amd._FlashAttentionFnBackward", g_node_properties, nullptr);
  torch::autograd::registerCppFunction(typeid(FlashAttentionBackward), &g_node_type);
  return PyModule_Create(&g_module);
}
