// came8_host: descriptors of a param group's tensors for came8_step, filled natively.
//
// gather() does what the optimizers' Python does for every parameter of a group before a step (the checks of
// _prepare_param and _check_state, the fields of _descriptors and _fill_desc, the step counts) for the plain case:
// contiguous strided parameters and gradients on one GPU whose states exist in the optimizer's own layout.  It checks
// all of them anew on every call, changes nothing unless all pass, and returns None otherwise, upon which the Python
// takes the group from the start: it creates states, copies what is not contiguous and raises the errors.
// 192 adapters of 10 to 130 KB: 64 us of host time a step instead of 940; 292 tensors of a 24-layer model: 196 us
// instead of 1380.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>

#include <cstdint>
#include <vector>

#include "../../include/came8.h"

namespace {

PyObject* key(const char* name) { return PyUnicode_InternFromString(name); }

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return CAME8_F32;
    case at::kBFloat16: return CAME8_BF16;
    case at::kHalf: return CAME8_F16;
    default: return -1;
  }
}

// the tensor under `name` in a state, or null (borrowed)
const at::Tensor* tensor_of(PyObject* st, PyObject* name) {
  PyObject* o = PyDict_GetItemWithError(st, name);
  return o != nullptr && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool flag_off(PyObject* st, PyObject* name) {
  PyObject* o = PyDict_GetItemWithError(st, name);
  return o == nullptr || o == Py_False;
}

int64_t num_blocks(int64_t n, int64_t block) { return n <= 0 ? 1 : (n + block - 1) / block; }

template <typename T>
void put(T*& field, const at::Tensor* t) {
  field = static_cast<T*>(t->data_ptr());
}

// What the plain case asks of the parameter and gradient themselves.  The whole group is looked over before the first
// state is: a group that the Python takes after all (a transposed gradient at the end of 290 tensors) has then lost 8 us of
// its 1200, not 52.
bool plain(const at::Tensor& p, const at::Tensor& g) {
  return p.is_cuda() && p.layout() == at::kStrided && g.layout() == at::kStrided && g.device() == p.device() &&
         p.is_contiguous() && g.is_contiguous() && p.numel() != 0 && p.sizes() == g.sizes() && dtype_code(p) >= 0 &&
         dtype_code(g) >= 0;
}

// One parameter's descriptor; false: not the plain case.  *step: its state's step count.
bool describe(const at::Tensor& p, const at::Tensor& g, PyObject* st, int kind, int64_t block, came8_tensor& d,
              long* step) {
  static PyObject *k_mode = key("_mode"), *k_nd = key("_cuda_factored_nd_ext_path"),
                  *k_ndc = key("_cuda_factored_nd_chunked_ext_path"), *k_fact = key("factored"), *k_step = key("step"),
                  *k_mq = key("exp_avg_q"), *k_ma = key("exp_avg_absmax"), *k_rq = key("factored_row_q"),
                  *k_ra = key("factored_row_absmax"), *k_cq = key("factored_col_q"),
                  *k_ca = key("factored_col_absmax"), *k_vq = key("exp_avg_sq_q"), *k_va = key("exp_avg_sq_absmax"),
                  *k_m = key("exp_avg"), *k_v = key("exp_avg_sq"), *k_sr = key("exp_avg_sq_row"),
                  *k_sc = key("exp_avg_sq_col"), *k_rr = key("exp_avg_res_row"), *k_rc = key("exp_avg_res_col");
  PyObject* mode = PyDict_GetItemWithError(st, k_mode);
  if (mode == nullptr || !PyUnicode_Check(mode) ||
      PyUnicode_CompareWithASCIIString(mode, kind == CAME8_STATE_FP32 ? "cudafp" : "full8bit") != 0)
    return false;
  PyObject* fo = PyDict_GetItemWithError(st, k_fact);
  if (fo != Py_True && fo != Py_False) return false;
  const bool fact = fo == Py_True;
  const int64_t nd = p.dim(), n = p.numel();
  if (fact != (nd >= 2)) return false;
  PyObject* so = PyDict_GetItemWithError(st, k_step);
  if (so == nullptr || !PyLong_CheckExact(so)) return false;
  int over = 0;
  *step = PyLong_AsLongAndOverflow(so, &over);
  if (over != 0) return false;
  const int64_t C = nd > 0 ? p.size(nd - 1) : 1, R = fact ? p.size(nd - 2) : 1, P = fact ? n / (R * C) : 1;
  d = came8_tensor{};
  d.param = p.data_ptr();
  d.grad = g.data_ptr();
  d.param_dtype = dtype_code(p);
  d.grad_dtype = dtype_code(g);
  d.state_kind = kind;
  d.factored = fact ? 1 : 0;
  d.prefix = P;
  d.rows = R;
  d.cols = fact ? C : n;
  if (kind == CAME8_STATE_FP32) {
    const at::Tensor* m = tensor_of(st, k_m);
    if (m == nullptr || m->sizes() != p.sizes()) return false;
    const at::Tensor* s[5] = {m, fact ? tensor_of(st, k_sr) : tensor_of(st, k_v), fact ? tensor_of(st, k_rr) : m,
                              fact ? tensor_of(st, k_sc) : m, fact ? tensor_of(st, k_rc) : m};
    for (const at::Tensor* t : s)
      if (t == nullptr || t->device() != p.device() || t->scalar_type() != at::kFloat || !t->is_contiguous()) return false;
    put(d.exp_avg_q, s[0]);
    put(d.row_q, s[1]);
    if (fact) {
      put(d.row_absmax, s[2]);
      put(d.col_q, s[3]);
      put(d.col_absmax, s[4]);
    }
    return true;
  }
  if (!flag_off(st, k_nd) || !flag_off(st, k_ndc)) return false;  // per-matrix blocks
  const at::Tensor *mq = tensor_of(st, k_mq), *ma = tensor_of(st, k_ma);
  if (mq == nullptr || ma == nullptr || mq->sizes() != p.sizes() || mq->device() != p.device() ||
      ma->numel() != num_blocks(n, block))
    return false;
  put(d.exp_avg_q, mq);
  put(d.exp_avg_absmax, ma);
  const at::Tensor *rq = tensor_of(st, fact ? k_rq : k_vq), *ra = tensor_of(st, fact ? k_ra : k_va);
  if (rq == nullptr || ra == nullptr) return false;
  put(d.row_q, rq);
  put(d.row_absmax, ra);
  if (fact) {
    const at::Tensor *cq = tensor_of(st, k_cq), *ca = tensor_of(st, k_ca);
    if (cq == nullptr || ca == nullptr || rq->numel() != 2 * P * R || ra->numel() != 2 * num_blocks(P * R, block) ||
        cq->numel() != 2 * P * C || ca->numel() != 2 * num_blocks(P * C, block))
      return false;
    put(d.col_q, cq);
    put(d.col_absmax, ca);
  }
  return true;
}

// gather(params: list, state: dict, address: int, capacity: int, state_kind: int, block_size: int)
//   -> list of the parameters with a gradient, whose came8_tensor descriptors now lie at `address` in that order and
//      whose step counts are advanced; None: not the plain case, nothing changed.
PyObject* gather(PyObject*, PyObject* args) {
  PyObject *params, *state;
  unsigned long long addr;
  long long cap, block;
  int kind;
  if (!PyArg_ParseTuple(args, "O!O!KLiL", &PyList_Type, &params, &PyDict_Type, &state, &addr, &cap, &kind, &block))
    return nullptr;
  if (block < 1) Py_RETURN_NONE;  // the blocks are counted by a division; the Python raises the error
  try {
    came8_tensor* out = reinterpret_cast<came8_tensor*>(static_cast<uintptr_t>(addr));
    const Py_ssize_t n = PyList_GET_SIZE(params);
    std::vector<PyObject*> used;                     // the parameters with a gradient
    std::vector<std::pair<PyObject*, long>> counts;  // their states and step counts (the dicts outlive this call)
    std::vector<at::Tensor> grads;                   // and those (a key's hash may run Python, which may replace one)
    used.reserve(size_t(n));
    grads.reserve(size_t(n));
    const at::Tensor* first = nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* po = PyList_GET_ITEM(params, i);
      if (!THPVariable_CheckExact(po)) Py_RETURN_NONE;  // subclasses may keep their data elsewhere
      const at::Tensor& p = THPVariable_Unpack(po);
      const at::Tensor& g = p.grad();
      if (!g.defined()) continue;
      if (first == nullptr) first = &p;
      if (g.key_set().has(c10::DispatchKey::Python) || int64_t(used.size()) >= cap || p.device() != first->device() ||
          !plain(p, g))
        Py_RETURN_NONE;
      used.push_back(po);
      grads.push_back(g);
    }
    counts.reserve(used.size());
    for (size_t i = 0; i < used.size(); ++i) {
      const at::Tensor& p = THPVariable_Unpack(used[i]);
      PyObject* st = PyDict_GetItemWithError(state, used[i]);
      long step = 0;
      if (st == nullptr || !PyDict_Check(st) || !describe(p, grads[i], st, kind, block, out[i], &step)) {
        PyErr_Clear();
        Py_RETURN_NONE;
      }
      counts.emplace_back(st, step);
    }
    static PyObject* k_step = key("step");
    PyObject* res = PyList_New(Py_ssize_t(used.size()));
    if (res == nullptr) return nullptr;
    for (size_t i = 0; i < used.size(); ++i) {
      Py_INCREF(used[i]);
      PyList_SET_ITEM(res, Py_ssize_t(i), used[i]);
      PyObject* v = PyLong_FromLong(counts[i].second + 1);
      if (v == nullptr || PyDict_SetItem(counts[i].first, k_step, v) != 0) {
        Py_XDECREF(v);
        Py_DECREF(res);
        return nullptr;
      }
      Py_DECREF(v);
    }
    return res;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

PyMethodDef methods[] = {{"gather", gather, METH_VARARGS, "descriptors of a param group's tensors"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "came8_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_came8_host(void) { return PyModule_Create(&module); }
