// Host side of the optimizer steps as a CPython module (dion_amd._host): gathers the tensors of a parameter group, buckets
// them and calls the library.  The step of a small model is bound by what the host does per tensor and per launch; walking
// the parameters here instead of in Python costs 0.2 us per parameter instead of 4-6.
//
// Nothing is kept between calls: tensors, states and hyper-parameters are read anew every time.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <cmath>
#include <vector>
#include "../../include/dion_amd.h"

namespace {

// entry points of the library that _lib.py loaded
struct Api {
  decltype(&dion_amd_muon_buckets_workspace_bytes) muon_bytes;
  decltype(&dion_amd_muon_step_buckets) muon_step;
  decltype(&dion_amd_lion_step) lion_step;
  decltype(&dion_amd_adamw_step) adamw_step;
  decltype(&dion_amd_dion_buckets_workspace_bytes) dion_bytes;
  decltype(&dion_amd_dion_step_buckets) dion_step;
} api;
PyObject* g_error = nullptr;    // _lib.DionAmdError
PyObject* g_check = nullptr;    // _lib.check(rc, what)
PyObject *s_momentum, *s_variance, *s_q, *s_get, *s_buf;

struct Failed {};   // a Python exception is set

[[noreturn]] void fail(const char* fmt, const char* what = "") {
  PyErr_Format(g_error, fmt, what);
  throw Failed();
}

int dtype_code(at::ScalarType t) {
  if (t == at::kBFloat16) return DION_AMD_BF16;
  if (t == at::kFloat) return DION_AMD_F32;
  if (t == at::kDouble) return DION_AMD_F64;
  fail("unsupported dtype torch.%s", c10::toString(t));
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  PyObject* r = PyObject_CallFunction(g_check, "is", rc, what);
  Py_XDECREF(r);
  throw Failed();
}

// The interpreter lock is released while the library is called (argument checks, pointer tables and launches, 5 to 50 us):
// other threads of the program run meanwhile.  Whatever the call is handed is held by references of the caller's own.
struct Unlocked {
  PyThreadState* saved = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(saved); }
};

// One parameter with its gradient and its states.
struct Entry {
  at::Tensor p, g;
  at::Tensor s[2];
};

// A reference of our own; null: a Python exception is set.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) { if (!p) throw Failed(); }
  Ref(Ref&& o) : p(o.p) { o.p = nullptr; }
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

// map[key] for a dict or any other mapping; `none` (borrowed) where there is no such key.
Ref lookup(PyObject* map, PyObject* key, PyObject* none) {
  PyObject* v;
  if (PyDict_Check(map)) {
    v = PyDict_GetItemWithError(map, key);
    Py_XINCREF(v);
    if (!v && PyErr_Occurred()) throw Failed();
  } else {
    v = PyObject_GetItem(map, key);
    if (!v) {
      if (!PyErr_ExceptionMatches(PyExc_KeyError)) throw Failed();
      PyErr_Clear();
    }
  }
  if (!v) {
    v = none;
    Py_INCREF(v);
  }
  return Ref(v);
}

// The parameters of `params` (a tuple) that have a gradient, with the state tensors named `keys`.  Appends the parameters
// without state to `missing` (a Python list) instead.
void gather(PyObject* params, PyObject* state, PyObject* const* keys, int nkeys, std::vector<Entry>& out, PyObject* missing,
            std::vector<PyObject*>* objects = nullptr) {
  const Py_ssize_t n = PyTuple_GET_SIZE(params);
  out.reserve((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyTuple_GET_ITEM(params, i);
    if (!THPVariable_Check(o)) {
      PyErr_SetString(PyExc_TypeError, "parameters must be tensors");
      throw Failed();
    }
    const at::Tensor& p = THPVariable_Unpack(o);
    const at::Tensor& g = p.grad();
    if (!g.defined()) continue;
    const Ref st = lookup(state, o, Py_None);
    const int there = PyObject_IsTrue(st.p);   // (an empty state, as `Optimizer.state` makes them, is to be filled)
    if (there < 0) throw Failed();
    if (!there) {
      if (PyList_Append(missing, o)) throw Failed();
      continue;
    }
    out.emplace_back();
    if (objects) objects->push_back(o);
    Entry& e = out.back();
    e.p = p;
    e.g = g;
    for (int k = 0; k < nkeys; ++k) {
      const Ref t = lookup(st.p, keys[k], Py_None);
      if (!THPVariable_Check(t.p)) {
        PyErr_SetObject(PyExc_KeyError, keys[k]);
        throw Failed();
      }
      e.s[k] = THPVariable_Unpack(t.p);
    }
  }
}

// `nbytes` of workspace on `dev` from a _lib.Workspace
at::Tensor workspace(PyObject* ws, size_t nbytes, c10::Device dev) {
  {
    const Ref buf(PyObject_GetAttr(ws, s_buf));
    if (THPVariable_Check(buf.p)) {
      const at::Tensor& t = THPVariable_Unpack(buf.p);
      if ((size_t)t.numel() >= nbytes && t.device() == dev) return t;
    }
  }
  const Ref d(THPDevice_New(dev)), n(PyLong_FromSize_t(nbytes));
  const Ref t(PyObject_CallMethodObjArgs(ws, s_get, n.p, d.p, nullptr));
  return THPVariable_Unpack(t.p);
}

void* stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// ---- Muon

struct MuonBucket {
  at::Tensor p0;                 // shape, dtypes and device of the bucket
  at::ScalarType gtype;
  std::vector<void*> X, M;
  std::vector<const void*> G;
  long long m, n;
  float adjusted;
};

// adjust_lr of dion_amd.muon: 0 none, 1 spectral_norm, 2 rms_norm, 3 keller_muon; evaluated like a 0-dim fp32 tensor times
// a Python number
float adjusted_lr(float lr, int adjust, double rows, double cols) {
  switch (adjust) {
    case 1: return lr * (float)std::sqrt(rows / cols);
    case 2: return lr * (float)(0.2 * std::sqrt(rows > cols ? rows : cols));
    case 3: { const double q = rows / cols; return lr * (float)std::pow(q > 1.0 ? q : 1.0, 0.5); }
    default: return lr;
  }
}

// muon_group(params, state, lr, mu, weight_decay, epsilon, nesterov, adjust, flatten, coeffs address, steps, workspace)
// -> None, or the list of parameters whose state has to be created first (nothing was done then)
PyObject* muon_group(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 12) { PyErr_SetString(PyExc_TypeError, "muon_group: 12 arguments"); return nullptr; }
  PyObject* missing = nullptr;
  try {
    const float lr = (float)PyFloat_AsDouble(a[2]), mu = (float)PyFloat_AsDouble(a[3]), wd = (float)PyFloat_AsDouble(a[4]),
                eps = (float)PyFloat_AsDouble(a[5]);
    const int nesterov = PyObject_IsTrue(a[6]), adjust = (int)PyLong_AsLong(a[7]), flatten = PyObject_IsTrue(a[8]);
    const float* coeffs = static_cast<const float*>(PyLong_AsVoidPtr(a[9]));
    const int steps = (int)PyLong_AsLong(a[10]);
    if (PyErr_Occurred()) return nullptr;
    at::NoGradGuard no_grad;
    const Ref params(PySequence_Tuple(a[0]));   // (any collection; it keeps them while this call lasts)
    missing = PyList_New(0);
    if (!missing) return nullptr;
    std::vector<Entry> all;
    gather(params.p, a[1], &s_momentum, 1, all, missing);
    if (PyList_GET_SIZE(missing)) return missing;
    Py_CLEAR(missing);

    std::vector<MuonBucket> buckets;
    for (Entry& e : all) {
      // (the library reads as many elements of the gradient and the momentum as the parameter has, the momentum in its dtype)
      if (e.s[0].numel() != e.p.numel() || e.s[0].scalar_type() != e.p.scalar_type() || e.s[0].device() != e.p.device() ||
          e.g.numel() != e.p.numel() || e.g.device() != e.p.device())
        fail("Muon.step: gradient and momentum do not fit their parameter");
      MuonBucket* b = nullptr;
      for (MuonBucket& c : buckets)
        if (c.p0.sizes().equals(e.p.sizes()) && c.p0.scalar_type() == e.p.scalar_type() && c.gtype == e.g.scalar_type() &&
            c.p0.device() == e.p.device()) { b = &c; break; }
      const auto sizes = e.p.sizes();
      const long long rows = sizes[sizes.size() - 2], cols = sizes[sizes.size() - 1];
      if (!b) {
        if (!e.p.is_cuda()) {
          PyErr_Format(g_error, "Muon.step: tensor is on %s; the MI355X kernels need a GPU tensor (no CPU fallback)",
                       e.p.device().str().c_str());
          throw Failed();
        }
        buckets.emplace_back();
        b = &buckets.back();
        b->p0 = e.p;
        b->gtype = e.g.scalar_type();
        b->m = sizes.size() == 2 ? rows : (flatten ? sizes[0] : rows);
        b->n = sizes.size() == 2 ? cols : (flatten ? (sizes[0] ? e.p.numel() / sizes[0] : 0) : cols);
        b->adjusted = adjusted_lr(lr, adjust, (double)rows, (double)cols);
        const size_t count = all.size();
        b->X.reserve(count); b->G.reserve(count); b->M.reserve(count);
      }
      if (!e.p.is_contiguous() || !e.s[0].is_contiguous()) fail("Muon.step: parameters and momentum buffers must be contiguous");
      if (!e.g.is_contiguous()) e.g = e.g.contiguous();
      char *x = static_cast<char*>(e.p.data_ptr()), *g = static_cast<char*>(e.g.data_ptr()), *m = static_cast<char*>(e.s[0].data_ptr());
      const long long per = b->m * b->n, count = per ? e.p.numel() / per : 0;
      const long long xs = per * (long long)e.p.element_size(), gs = per * (long long)e.g.element_size(),
                      ms = per * (long long)e.s[0].element_size();
      for (long long i = 0; i < count; ++i) {
        b->X.push_back(x + i * xs);
        b->G.push_back(g + i * gs);
        b->M.push_back(m + i * ms);
      }
    }

    // buckets of one (dtype, gradient dtype, device) go to the library together
    const float decay = 1.f - lr * wd;
    std::vector<char> done(buckets.size(), 0);
    std::vector<dion_amd_muon_bucket> call;
    for (size_t i = 0; i < buckets.size(); ++i) {
      if (done[i]) continue;
      const MuonBucket& f = buckets[i];
      call.clear();
      for (size_t j = i; j < buckets.size(); ++j) {
        MuonBucket& b = buckets[j];
        if (done[j] || b.p0.scalar_type() != f.p0.scalar_type() || b.gtype != f.gtype || b.p0.device() != f.p0.device()) continue;
        done[j] = 1;
        if (!b.X.empty())
          call.push_back({b.X.data(), b.G.data(), b.M.data(), (int)b.X.size(), (int)b.m, (int)b.n, decay, b.adjusted});
      }
      if (call.empty()) continue;
      const c10::Device dev = f.p0.device();
      const int xc = dtype_code(f.p0.scalar_type()), gc = dtype_code(f.gtype);
      const size_t need = api.muon_bytes(call.data(), (int)call.size());
      const at::Tensor ws = workspace(a[11], need, dev);
      const c10::DeviceGuard guard(dev);
      int rc;
      {
        const Unlocked unlocked;
        rc = api.muon_step(call.data(), (int)call.size(), xc, gc, mu, nesterov, coeffs, steps, eps, 1, ws.data_ptr(), need,
                           stream_of(dev));
      }
      check(rc, "dion_amd_muon_step_buckets");
    }
    Py_RETURN_NONE;
  } catch (const Failed&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  Py_XDECREF(missing);
  return nullptr;
}

// ---- Dion

struct DionBucket {
  Entry first;                   // shape, dtypes and device of the bucket
  PyObject* p0;                  // its first parameter (borrowed)
  std::vector<void*> X, M, Q;
  std::vector<const void*> G;
  std::vector<PyObject*> params; // borrowed
  long long m, n, r;
};

// dion_group(params, state, lr, mu, weight_decay, epsilon, workspace, info) -> None when the step is done; a list: parameters
// whose state has to be created first (nothing was done then); a tuple: parameters of the buckets that the one-launch entry
// point does not take, which are left to the caller.  info(parameter, count): the status words of a bucket (int32 tensor).
PyObject* dion_group(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 8) { PyErr_SetString(PyExc_TypeError, "dion_group: 8 arguments"); return nullptr; }
  PyObject* missing = nullptr;
  try {
    const float lr = (float)PyFloat_AsDouble(a[2]), mu = (float)PyFloat_AsDouble(a[3]), wd = (float)PyFloat_AsDouble(a[4]),
                eps = (float)PyFloat_AsDouble(a[5]);
    if (PyErr_Occurred()) return nullptr;
    at::NoGradGuard no_grad;
    const Ref params(PySequence_Tuple(a[0]));
    missing = PyList_New(0);
    if (!missing) return nullptr;
    std::vector<Entry> all;
    std::vector<PyObject*> objects;
    PyObject* const keys[2] = {s_momentum, s_q};
    gather(params.p, a[1], keys, 2, all, missing, &objects);
    if (PyList_GET_SIZE(missing)) return missing;
    Py_CLEAR(missing);

    std::vector<DionBucket> buckets;
    for (size_t k = 0; k < all.size(); ++k) {
      Entry& e = all[k];
      DionBucket* b = nullptr;
      for (DionBucket& c : buckets)
        if (c.first.p.sizes().equals(e.p.sizes()) && c.first.p.scalar_type() == e.p.scalar_type() &&
            c.first.g.scalar_type() == e.g.scalar_type() && c.first.p.device() == e.p.device()) { b = &c; break; }
      if (!b) {
        if (!e.p.is_cuda()) {
          PyErr_Format(g_error, "Dion.step: tensor is on %s; the MI355X kernels need a GPU tensor (no CPU fallback)",
                       e.p.device().str().c_str());
          throw Failed();
        }
        buckets.emplace_back();
        b = &buckets.back();
        b->first = e;
        b->p0 = objects[k];
        b->m = e.p.size(0); b->n = e.p.size(1); b->r = e.s[1].size(1);
      }
      if (!e.p.is_contiguous() || !e.s[0].is_contiguous() || !e.s[1].is_contiguous())
        fail("Dion.step: parameters and optimizer states must be contiguous");
      if (!e.s[0].sizes().equals(e.p.sizes()) || e.s[1].size(0) != std::min(b->m, b->n) || e.s[1].size(1) != b->r)
        fail("Dion.step: optimizer states do not fit their parameter");
      if (!e.g.is_contiguous()) e.g = e.g.contiguous();
      b->X.push_back(e.p.data_ptr());
      b->G.push_back(e.g.data_ptr());
      b->M.push_back(e.s[0].data_ptr());
      b->Q.push_back(e.s[1].data_ptr());
      b->params.push_back(objects[k]);
    }

    // buckets of one set of dtypes and device go to the library together
    const float decay = 1.f - lr * wd, ef_alpha = -(1.f - mu);
    std::vector<char> done(buckets.size(), 0);
    std::vector<dion_amd_dion_bucket> call;
    std::vector<DionBucket*> members;
    std::vector<at::Tensor> infos;
    std::vector<PyObject*> left;
    for (size_t i = 0; i < buckets.size(); ++i) {
      if (done[i]) continue;
      const Entry f = buckets[i].first;
      call.clear();
      members.clear();
      for (size_t j = i; j < buckets.size(); ++j) {
        DionBucket& b = buckets[j];
        if (done[j] || b.first.p.scalar_type() != f.p.scalar_type() || b.first.g.scalar_type() != f.g.scalar_type() ||
            b.first.s[0].scalar_type() != f.s[0].scalar_type() || b.first.s[1].scalar_type() != f.s[1].scalar_type() ||
            b.first.p.device() != f.p.device())
          continue;
        done[j] = 1;
        members.push_back(&b);
        const float scale = (float)std::pow((double)b.m / (double)b.n, 0.5);
        call.push_back({b.X.data(), b.G.data(), b.M.data(), b.Q.data(), (int)b.X.size(), (int)b.m, (int)b.n, (int)b.r, scale * lr, nullptr});
      }
      const c10::Device dev = f.p.device();
      const int xc = dtype_code(f.p.scalar_type()), gc = dtype_code(f.g.scalar_type()), mc = dtype_code(f.s[0].scalar_type()),
                qc = dtype_code(f.s[1].scalar_type());
      const size_t need = api.dion_bytes(call.data(), (int)call.size(), xc, gc, mc, qc);
      if (need == 0) {
        for (DionBucket* b : members) left.insert(left.end(), b->params.begin(), b->params.end());
        continue;
      }
      infos.clear();
      for (size_t j = 0; j < members.size(); ++j) {
        const Ref cnt(PyLong_FromSize_t(members[j]->X.size()));
        const Ref t(PyObject_CallFunctionObjArgs(a[7], members[j]->p0, cnt.p, nullptr));
        infos.push_back(THPVariable_Unpack(t.p));
        call[j].info = static_cast<int*>(infos.back().data_ptr());
      }
      const at::Tensor ws = workspace(a[6], need, dev);
      const c10::DeviceGuard guard(dev);
      int rc;
      {
        const Unlocked unlocked;
        rc = api.dion_step(call.data(), (int)call.size(), xc, gc, mc, qc, ef_alpha, decay, eps, ws.data_ptr(), need, stream_of(dev));
      }
      check(rc, "dion_amd_dion_step_buckets");
    }
    if (left.empty()) Py_RETURN_NONE;
    PyObject* rest = PyTuple_New((Py_ssize_t)left.size());
    if (!rest) return nullptr;
    for (size_t i = 0; i < left.size(); ++i) {
      Py_INCREF(left[i]);
      PyTuple_SET_ITEM(rest, (Py_ssize_t)i, left[i]);
    }
    return rest;
  } catch (const Failed&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  Py_XDECREF(missing);
  return nullptr;
}

// ---- Lion / AdamW

// (hyper-parameters are evaluated like 0-dim fp32 tensors, reference dion/scalar_opts.py:89-187)
void elementwise_run(bool adamw, std::vector<Entry>& all, const char* what, float lr, float beta1, float beta2, float wd,
                     double step, float eps) {
  const int ns = adamw ? 2 : 1;
  for (const Entry& e : all) {
    const at::Tensor* ts[4] = {&e.p, &e.g, &e.s[0], &e.s[1]};
    for (int k = 0; k < 2 + ns; ++k) {
      if (!ts[k]->is_cuda()) {
        PyErr_Format(g_error, "%s: tensor is on %s; the MI355X kernels need a GPU tensor (no CPU fallback)", what,
                     ts[k]->device().str().c_str());
        throw Failed();
      }
      if (!ts[k]->is_contiguous()) fail("%s: parameters, gradients and optimizer states must be contiguous", what);
      if (k && !ts[k]->sizes().equals(e.p.sizes())) fail("%s: shapes of a parameter and its gradient / states differ", what);
    }
  }
  float adjusted = lr, bc2 = 0.f;
  if (adamw && !all.empty()) {
    // (torch's own power and square root: their fp32 results are not the C library's in the last bit)
    const at::Tensor st = at::scalar_tensor(step, at::TensorOptions().dtype(step == std::floor(step) ? at::kLong : at::kFloat));
    const float p1 = at::pow(at::scalar_tensor(beta1, at::kFloat), st).item<float>();
    const float p2 = at::pow(at::scalar_tensor(beta2, at::kFloat), st).item<float>();
    adjusted = lr / (1.f - p1);
    bc2 = at::sqrt(at::scalar_tensor(1.f - p2, at::kFloat)).item<float>();
  }
  const float decay = 1.f - lr * wd;
  std::vector<char> done(all.size(), 0);
  std::vector<void*> X, M, V;
  std::vector<const void*> G;
  std::vector<long long> numel;
  for (size_t i = 0; i < all.size(); ++i) {
    if (done[i] || all[i].p.numel() == 0) continue;
    const Entry& f = all[i];
    X.clear(); G.clear(); M.clear(); V.clear(); numel.clear();
    for (size_t j = i; j < all.size(); ++j) {
      const Entry& e = all[j];
      if (done[j] || e.p.numel() == 0 || e.p.device() != f.p.device() || e.p.scalar_type() != f.p.scalar_type() ||
          e.g.scalar_type() != f.g.scalar_type() || e.s[0].scalar_type() != f.s[0].scalar_type() ||
          (adamw && e.s[1].scalar_type() != f.s[1].scalar_type()))
        continue;
      done[j] = 1;
      X.push_back(e.p.data_ptr());
      G.push_back(e.g.data_ptr());
      M.push_back(e.s[0].data_ptr());
      if (adamw) V.push_back(e.s[1].data_ptr());
      numel.push_back(e.p.numel());
    }
    const c10::Device dev = f.p.device();
    const int xc = dtype_code(f.p.scalar_type()), gc = dtype_code(f.g.scalar_type()), mc = dtype_code(f.s[0].scalar_type());
    const c10::DeviceGuard guard(dev);
    const int vc = adamw ? dtype_code(f.s[1].scalar_type()) : 0;
    int rc;
    {
      const Unlocked unlocked;
      rc = adamw ? api.adamw_step(X.data(), G.data(), M.data(), V.data(), numel.data(), (int)X.size(), xc, gc, mc, vc, adjusted,
                                  1.f - beta1, 1.f - beta2, decay, bc2, eps, stream_of(dev))
                 : api.lion_step(X.data(), G.data(), M.data(), numel.data(), (int)X.size(), xc, gc, mc, lr, 1.f - beta1,
                                 1.f - beta2, decay, stream_of(dev));
    }
    check(rc, adamw ? "dion_amd_adamw_step" : "dion_amd_lion_step");
  }
}

struct Scalars { float lr, b1, b2, wd, eps; double step; };
bool scalars(PyObject* const* a, Scalars& s) {   // lr, beta1, beta2, weight_decay, step, epsilon
  s.lr = (float)PyFloat_AsDouble(a[0]);
  s.b1 = (float)PyFloat_AsDouble(a[1]);
  s.b2 = (float)PyFloat_AsDouble(a[2]);
  s.wd = (float)PyFloat_AsDouble(a[3]);
  s.step = PyFloat_AsDouble(a[4]);
  s.eps = (float)PyFloat_AsDouble(a[5]);
  return !PyErr_Occurred();
}

// element_group(adamw, params, state, lr, beta1, beta2, weight_decay, step, epsilon) -> None or the parameters without state
PyObject* element_group(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 9) { PyErr_SetString(PyExc_TypeError, "element_group: 9 arguments"); return nullptr; }
  PyObject* missing = nullptr;
  try {
    const bool adamw = PyObject_IsTrue(a[0]) == 1;
    Scalars s;
    if (!scalars(a + 3, s)) return nullptr;
    at::NoGradGuard no_grad;
    const Ref params(PySequence_Tuple(a[1]));
    missing = PyList_New(0);
    if (!missing) return nullptr;
    std::vector<Entry> all;
    PyObject* const keys[2] = {s_momentum, s_variance};
    gather(params.p, a[2], keys, adamw ? 2 : 1, all, missing);
    if (PyList_GET_SIZE(missing)) return missing;
    Py_CLEAR(missing);
    elementwise_run(adamw, all, adamw ? "adamw_update_foreach" : "lion_update_foreach", s.lr, s.b1, s.b2, s.wd, s.step, s.eps);
    Py_RETURN_NONE;
  } catch (const Failed&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  Py_XDECREF(missing);
  return nullptr;
}

// element_lists(adamw, X, G, M, V, lr, beta1, beta2, weight_decay, step, epsilon): the same for lists of tensors (V is not
// read for Lion)
PyObject* element_lists(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 11) { PyErr_SetString(PyExc_TypeError, "element_lists: 11 arguments"); return nullptr; }
  try {
    const bool adamw = PyObject_IsTrue(a[0]) == 1;
    Scalars s;
    if (!scalars(a + 5, s)) return nullptr;
    at::NoGradGuard no_grad;
    for (int k = 0; k < (adamw ? 4 : 3); ++k)
      if (!PyList_Check(a[1 + k]) || PyList_GET_SIZE(a[1 + k]) != PyList_GET_SIZE(a[1])) {
        PyErr_SetString(PyExc_TypeError, "expected lists of equal length");
        return nullptr;
      }
    const Py_ssize_t n = PyList_GET_SIZE(a[1]);
    std::vector<Entry> all((size_t)n);
    for (Py_ssize_t i = 0; i < n; ++i) {
      at::Tensor* to[4] = {&all[i].p, &all[i].g, &all[i].s[0], &all[i].s[1]};
      for (int k = 0; k < (adamw ? 4 : 3); ++k) {
        PyObject* o = PyList_GET_ITEM(a[1 + k], i);
        if (!THPVariable_Check(o)) {
          PyErr_SetString(PyExc_TypeError, "expected lists of tensors");
          return nullptr;
        }
        *to[k] = THPVariable_Unpack(o);
      }
    }
    elementwise_run(adamw, all, adamw ? "adamw_update_foreach" : "lion_update_foreach", s.lr, s.b1, s.b2, s.wd, s.step, s.eps);
    Py_RETURN_NONE;
  } catch (const Failed&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// ---- module

// bind(DionAmdError, check, addresses of the entry points in the order of Api)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *err, *chk;
  unsigned long long f[6];
  if (!PyArg_ParseTuple(args, "OOKKKKKK", &err, &chk, f, f + 1, f + 2, f + 3, f + 4, f + 5)) return nullptr;
  Py_INCREF(err);
  Py_INCREF(chk);
  g_error = err;
  g_check = chk;
  api.muon_bytes = reinterpret_cast<decltype(api.muon_bytes)>(f[0]);
  api.muon_step = reinterpret_cast<decltype(api.muon_step)>(f[1]);
  api.lion_step = reinterpret_cast<decltype(api.lion_step)>(f[2]);
  api.adamw_step = reinterpret_cast<decltype(api.adamw_step)>(f[3]);
  api.dion_bytes = reinterpret_cast<decltype(api.dion_bytes)>(f[4]);
  api.dion_step = reinterpret_cast<decltype(api.dion_step)>(f[5]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "Entry points of the loaded library."},
    {"muon_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(muon_group)), METH_FASTCALL, "Muon step of a group."},
    {"dion_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dion_group)), METH_FASTCALL, "Dion step of a group."},
    {"element_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(element_group)), METH_FASTCALL,
     "Lion / AdamW step of a group."},
    {"element_lists", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(element_lists)), METH_FASTCALL,
     "Lion / AdamW step of lists of tensors."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of the optimizer steps.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  s_momentum = PyUnicode_InternFromString("momentum");
  s_variance = PyUnicode_InternFromString("variance");
  s_q = PyUnicode_InternFromString("Q");
  s_get = PyUnicode_InternFromString("get");
  s_buf = PyUnicode_InternFromString("_buf");
  return PyModule_Create(&module);
}
