// The host side of a step in native code: a CPython module that checks tensors, refreshes a plan's descriptors and
// makes the calls of the C ABI (include/q4adamw.h).
//
// What it replaces is interpreter work, about 0.1 us per attribute of a tensor, and ctypes' conversion of a call's
// arguments.  It only ever takes the common case: wherever an argument, a tensor's type, device, layout or size is not
// what the fast path is for, a function here says so (None, or False) before it has changed anything, and the
// Python code beside it, which words the refusals, takes the call.  us, before / with it, one machine: a direct call on
// one small tensor 8.4 / 4.7 (2.6 of it the launch); a step of six small tensors 21.5 / 12.9 (6 of it torch's wrapper
// around Optimizer.step), of two launches 31.1 / 17.3; the first pass of a clipped step over 148 tensors 722 / 413.
#include <Python.h>

#include <stdint.h>

#include <exception>
#include <memory>
#include <vector>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/q4adamw.h"

// What the module was built for: torch's and the interpreter's builds, in words that the loader compares with the running
// ones (the code below has torch's inline accessors of a tensor's fields in it, and a module of another build would
// read them at that build's offsets).
#ifndef Q4HOST_BUILT_FOR
#error "define Q4HOST_BUILT_FOR: see compile_host_module in build.py"
#endif

namespace {

// ---------------------------------------------------------------------------
// the library and what torch knows about the current device
// ---------------------------------------------------------------------------
struct Library {
  decltype(&q4adamw_fused_4bit) fused_4bit;
  decltype(&q4adamw_fused_single_tensor) fused_single_tensor;
  decltype(&q4adamw_fused_4bit_multi_ex) multi;
  decltype(&q4adamw_fused_4bit_multi_sr) multi_sr;
  decltype(&q4adamw_fused_4bit_rank1_multi) rank1;
  decltype(&q4adamw_fused_4bit_rank1_multi_sr) rank1_sr;
  decltype(&q4adamw_fused_single_tensor_multi_ex) small;
  decltype(&q4adamw_fused_step_multi) both;
};
Library lib;
PyObject *raw_stream_of = nullptr;     // torch._C._cuda_getCurrentRawStream
PyObject *current_device = nullptr;    // torch._C._cuda_getDevice

// bind(addresses of the eight functions above, in order, raw_stream_of, current_device)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 10) {
    PyErr_SetString(PyExc_TypeError, "bind takes eight addresses and two functions");
    return nullptr;
  }
  void *f[8];
  for (int i = 0; i < 8; ++i) {
    f[i] = PyLong_AsVoidPtr(args[i]);
    if (!f[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  lib.fused_4bit = reinterpret_cast<decltype(lib.fused_4bit)>(f[0]);
  lib.fused_single_tensor = reinterpret_cast<decltype(lib.fused_single_tensor)>(f[1]);
  lib.multi = reinterpret_cast<decltype(lib.multi)>(f[2]);
  lib.multi_sr = reinterpret_cast<decltype(lib.multi_sr)>(f[3]);
  lib.rank1 = reinterpret_cast<decltype(lib.rank1)>(f[4]);
  lib.rank1_sr = reinterpret_cast<decltype(lib.rank1_sr)>(f[5]);
  lib.small = reinterpret_cast<decltype(lib.small)>(f[6]);
  lib.both = reinterpret_cast<decltype(lib.both)>(f[7]);
  Py_INCREF(args[8]);
  Py_INCREF(args[9]);
  Py_XSETREF(raw_stream_of, args[8]);
  Py_XSETREF(current_device, args[9]);
  Py_RETURN_NONE;
}

// The current stream of a device if that device is the current one; false: neither known nor an error set.
bool stream_of(int64_t device, void **stream) {
  if (!raw_stream_of || !current_device) return false;
  PyObject *d = PyObject_CallNoArgs(current_device);
  if (!d) {
    PyErr_Clear();
    return false;
  }
  const long current = PyLong_AsLong(d);
  PyObject *s = current == device ? PyObject_CallOneArg(raw_stream_of, d) : nullptr;
  Py_DECREF(d);
  if (!s) {
    PyErr_Clear();
    return false;
  }
  *stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// ---------------------------------------------------------------------------
// tensors
// ---------------------------------------------------------------------------
int tag_of(c10::ScalarType t) {
  return t == c10::ScalarType::Float ? Q4ADAMW_FP32 : t == c10::ScalarType::BFloat16 ? Q4ADAMW_BF16 : t == c10::ScalarType::Half ? Q4ADAMW_FP16 : -1;
}

// A dense tensor of torch's own, on a GPU: its pointer and what else the checks need.
struct Dense {
  void *ptr;
  int64_t numel;
  int64_t device;
  c10::ScalarType type;
};

bool dense(const at::Tensor &t, Dense *out) {
  if (!t.defined() || t.layout() != c10::kStrided || !t.is_cuda() || t.unsafeGetTensorImpl()->is_python_dispatch() || !t.is_contiguous()) return false;
  out->ptr = t.data_ptr();
  out->numel = t.numel();
  out->device = t.device().index();
  out->type = t.scalar_type();
  return true;
}

bool dense(PyObject *o, Dense *out) { return THPVariable_CheckExact(o) && dense(THPVariable_Unpack(o), out); }

bool numbers(PyObject *const *args, int n, float *out) {
  for (int i = 0; i < n; ++i) {
    if (!PyFloat_CheckExact(args[i]) && !PyLong_CheckExact(args[i])) return false;
    const double x = PyFloat_AsDouble(args[i]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    out[i] = (float)x;
  }
  return true;
}

// fused_4bit(p, g, exp_avg, exp_avg_sq, exp_avg_scale, exp_avg_sq_scale, beta1, beta2, lr, weight_decay, eps, step):
// the call's status, or None where the call is not for the fast path
PyObject *fused_4bit(PyObject *, PyObject *const *args, Py_ssize_t n) {
  Dense t[6];
  float x[6];
  void *stream = nullptr;
  if (n != 12 || !lib.fused_4bit) Py_RETURN_NONE;
  try {
    for (int i = 0; i < 6; ++i)
      if (!dense(args[i], &t[i]) || t[i].device != t[0].device) Py_RETURN_NONE;
  } catch (const std::exception &) {
    Py_RETURN_NONE;
  }
  const int64_t bytes = (t[0].numel + 1) / 2, blocks = (t[0].numel + Q4ADAMW_BLOCK - 1) / Q4ADAMW_BLOCK;
  const int p_tag = tag_of(t[0].type), g_tag = tag_of(t[1].type);
  if (p_tag < 0 || g_tag < 0 || t[1].numel != t[0].numel || t[2].numel != bytes || t[3].numel != bytes || t[4].numel != blocks ||
      t[5].numel != blocks || t[2].type != c10::ScalarType::Byte || t[3].type != c10::ScalarType::Byte ||
      t[4].type != c10::ScalarType::Float || t[5].type != c10::ScalarType::Float || !numbers(args + 6, 6, x) || !stream_of(t[0].device, &stream))
    Py_RETURN_NONE;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = lib.fused_4bit(t[0].ptr, t[1].ptr, static_cast<uint8_t *>(t[2].ptr), static_cast<uint8_t *>(t[3].ptr), static_cast<float *>(t[4].ptr),
                      static_cast<float *>(t[5].ptr), t[0].numel, p_tag, g_tag, x[0], x[1], x[2], x[3], x[4], x[5], stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// fused_single_tensor(p, g, exp_avg, exp_avg_sq, beta1, beta2, lr, weight_decay, eps, step): likewise
PyObject *fused_single_tensor(PyObject *, PyObject *const *args, Py_ssize_t n) {
  Dense t[4];
  float x[6];
  void *stream = nullptr;
  if (n != 10 || !lib.fused_single_tensor) Py_RETURN_NONE;
  try {
    for (int i = 0; i < 4; ++i)
      if (!dense(args[i], &t[i]) || t[i].device != t[0].device || t[i].numel != t[0].numel) Py_RETURN_NONE;
  } catch (const std::exception &) {
    Py_RETURN_NONE;
  }
  const int p_tag = tag_of(t[0].type), g_tag = tag_of(t[1].type);
  if (p_tag < 0 || g_tag < 0 || t[2].type != c10::ScalarType::Float || t[3].type != c10::ScalarType::Float || !numbers(args + 4, 6, x) ||
      !stream_of(t[0].device, &stream))
    Py_RETURN_NONE;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = lib.fused_single_tensor(t[0].ptr, t[1].ptr, static_cast<float *>(t[2].ptr), static_cast<float *>(t[3].ptr), t[0].numel, p_tag, g_tag, x[0],
                               x[1], x[2], x[3], x[4], x[5], stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// gradients(parameter lists, descriptor array's address, its capacity): writes the gradients there are, in order, as
// q4adamw_grad and returns (their number, dtype tag, device index) -- or None: none there, more than fit, or not all
// dense and of one dtype on one device
PyObject *gradients(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3 || !PyTuple_CheckExact(args[0])) Py_RETURN_NONE;
  q4adamw_grad *out = static_cast<q4adamw_grad *>(PyLong_AsVoidPtr(args[1]));
  const Py_ssize_t capacity = PyLong_AsSsize_t(args[2]);
  if (PyErr_Occurred()) return nullptr;
  Py_ssize_t count = 0;
  Dense first = {}, d;
  try {
    for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(args[0]); ++k) {
      PyObject *params = PyTuple_GET_ITEM(args[0], k);
      if (!PyList_CheckExact(params)) Py_RETURN_NONE;
      for (Py_ssize_t i = 0; i < PyList_GET_SIZE(params); ++i) {
        PyObject *p = PyList_GET_ITEM(params, i);
        if (!THPVariable_CheckExact(p)) Py_RETURN_NONE;
        const at::Tensor &g = THPVariable_Unpack(p).grad();
        if (!g.defined()) continue;
        if (count == capacity || !dense(g, &d) || tag_of(d.type) < 0) Py_RETURN_NONE;
        if (count == 0) first = d;
        if (d.type != first.type || d.device != first.device) Py_RETURN_NONE;
        out[count].g = d.ptr;
        out[count].numel = d.numel;
        ++count;
      }
    }
  } catch (const std::exception &) {
    Py_RETURN_NONE;
  }
  if (count == 0) Py_RETURN_NONE;
  return Py_BuildValue("niL", count, tag_of(first.type), (long long)first.device);
}

// ---------------------------------------------------------------------------
// an optimizer's plan
// ---------------------------------------------------------------------------
struct Bucket {
  int kind;                    // 0 small, 1 block-scaled, 2 stochastic, 3 rank-1, 4 rank-1 and stochastic
  std::vector<int32_t> idx;    // into the parameters with a gradient
  char *arr;                   // descriptors; the second 8-byte field of each is the gradient
  size_t stride;
  int p_tag, g_tag;
  const uint32_t *salts;
  int with = -1;               // kinds 1 and 2: a bucket of kind 0 of the same types that goes in the same call
  bool taken = false;          // kind 0: goes in another one's call
};

// One param group's launches.  Every object here is borrowed: the Python plan that owns this one holds them.
struct Plan {
  struct Param {
    PyObject *object;
    void *ptr;
    int64_t numel;
    c10::ScalarType grad_type;
    bool has_grad;
  };
  struct Held {
    PyObject *holder, *key, *value;
  };
  std::vector<Param> params;         // all of the group's
  std::vector<Held> held;
  std::vector<Bucket> buckets;
  std::vector<void *> fresh;         // refresh: the gradients' addresses
  PyObject *step_buffer;
  float *steps;                      // of the parameters with a gradient
  int64_t device, with_grad;
};

PyObject *state_keys[3];      // "step", "exp_avg", "exp_avg_sq"

const char kPlanName[] = "quantfour_adamw_cuda_amd.plan";
void drop_plan(PyObject *capsule) { delete static_cast<Plan *>(PyCapsule_GetPointer(capsule, kPlanName)); }
Plan *plan_of(PyObject *o) { return static_cast<Plan *>(PyCapsule_GetPointer(o, kPlanName)); }

// plan(parameters, step buffer, held [(state, step, exp_avg, exp_avg_sq)] and [(dict, key, value)], buckets [(kind, [indices], address, stride, p tag, g tag, salts'
// address or 0)]): a capsule, or None if the group is not for the fast path.  All arguments are kept by the caller.
// May throw (torch's checks, or memory that is not there): make_plan takes that for None.
PyObject *new_plan(PyObject *const *args, Py_ssize_t n) {
  if (n != 5 || !PyTuple_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !PyList_CheckExact(args[2]) || !PyList_CheckExact(args[3]) ||
      !PyList_CheckExact(args[4]))
    Py_RETURN_NONE;
  auto plan = std::make_unique<Plan>();
  plan->device = -1;
  plan->with_grad = 0;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[0]); ++i) {
    PyObject *o = PyTuple_GET_ITEM(args[0], i);
    Dense d, g;
    if (!dense(o, &d)) Py_RETURN_NONE;
    const at::Tensor &grad = THPVariable_Unpack(o).grad();
    if (grad.defined() && !dense(grad, &g)) Py_RETURN_NONE;
    if (plan->device == -1) plan->device = d.device;
    if (d.device != plan->device) Py_RETURN_NONE;
    plan->params.push_back({o, d.ptr, d.numel, grad.defined() ? g.type : d.type, grad.defined()});
    plan->with_grad += grad.defined();
  }
  const at::Tensor &steps = THPVariable_Unpack(args[1]);
  if (!steps.is_cpu() || steps.scalar_type() != c10::ScalarType::Float || !steps.is_contiguous() || steps.numel() != plan->with_grad) Py_RETURN_NONE;
  plan->step_buffer = args[1];
  plan->steps = static_cast<float *>(steps.data_ptr());
  for (int list = 2; list < 4; ++list)
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[list]); ++i) {
      PyObject *t = PyList_GET_ITEM(args[list], i);
      if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != (list == 2 ? 4 : 3) || !PyDict_Check(PyTuple_GET_ITEM(t, 0))) Py_RETURN_NONE;
      if (list == 3) plan->held.push_back({PyTuple_GET_ITEM(t, 0), PyTuple_GET_ITEM(t, 1), PyTuple_GET_ITEM(t, 2)});
      else
        for (int k = 0; k < 3; ++k) plan->held.push_back({PyTuple_GET_ITEM(t, 0), state_keys[k], PyTuple_GET_ITEM(t, k + 1)});
    }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[4]); ++i) {
    Bucket b;
    PyObject *idx;
    unsigned long long arr, stride, salts;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(args[4], i), "iO!KKiiK", &b.kind, &PyList_Type, &idx, &arr, &stride, &b.p_tag, &b.g_tag, &salts)) return nullptr;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(idx); ++k) {
      const long x = PyLong_AsLong(PyList_GET_ITEM(idx, k));
      if (x < 0 || x >= plan->with_grad) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "index out of range");
        return nullptr;
      }
      b.idx.push_back((int32_t)x);
    }
    if (b.idx.empty() || b.kind < 0 || b.kind > 4) Py_RETURN_NONE;
    b.arr = reinterpret_cast<char *>((uintptr_t)arr);
    b.stride = (size_t)stride;
    b.salts = reinterpret_cast<const uint32_t *>((uintptr_t)salts);
    plan->buckets.push_back(std::move(b));
  }
  // small tensors go with quantized ones of their types; refresh sees to it that a bucket has one step number,
  // run that the two have the same one
  for (Bucket &b : plan->buckets)
    for (size_t k = 0; k < plan->buckets.size() && b.with < 0 && (b.kind == 1 || b.kind == 2); ++k) {
      Bucket &o = plan->buckets[k];
      if (o.kind == 0 && !o.taken && o.p_tag == b.p_tag && o.g_tag == b.g_tag) {
        o.taken = true;
        b.with = (int)k;
      }
    }
  plan->fresh.resize((size_t)plan->with_grad);
  PyObject *capsule = PyCapsule_New(plan.get(), kPlanName, drop_plan);
  if (capsule) plan.release();
  return capsule;
}

PyObject *make_plan(PyObject *, PyObject *const *args, Py_ssize_t n) {
  try {
    return new_plan(args, n);
  } catch (const std::exception &) {
    Py_RETURN_NONE;
  }
}

// refresh(plan, the group's parameters, step buffer): True if the plan still describes the group -- the same parameters at
// the same addresses, the same ones with a gradient, the same state, dense gradients of the same dtypes and sizes -- after
// pointing its descriptors at the gradients
PyObject *refresh(PyObject *, PyObject *const *args, Py_ssize_t n) {
  Plan *plan = n == 3 ? plan_of(args[0]) : nullptr;
  if (!plan) return n == 3 ? nullptr : (PyErr_SetString(PyExc_TypeError, "refresh takes three arguments"), nullptr);
  PyObject *params = args[1];
  if (!PyList_CheckExact(params) || (size_t)PyList_GET_SIZE(params) != plan->params.size() || args[2] != plan->step_buffer) Py_RETURN_FALSE;
  for (const Plan::Held &h : plan->held) {
    PyObject *now = PyDict_GetItemWithError(h.holder, h.key);
    if (now != h.value) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  }
  try {
    size_t k = 0;
    for (size_t i = 0; i < plan->params.size(); ++i) {
      const Plan::Param &p = plan->params[i];
      if (PyList_GET_ITEM(params, (Py_ssize_t)i) != p.object) Py_RETURN_FALSE;
      const at::Tensor &t = THPVariable_Unpack(p.object);
      const at::Tensor &grad = t.grad();
      if (grad.defined() != p.has_grad) Py_RETURN_FALSE;
      if (!p.has_grad) continue;
      Dense d;
      if (t.data_ptr() != p.ptr || !dense(grad, &d) || d.type != p.grad_type || d.numel != p.numel || t.numel() != p.numel || d.device != plan->device)
        Py_RETURN_FALSE;
      plan->fresh[k++] = d.ptr;
    }
    if (THPVariable_Unpack(plan->step_buffer).data_ptr() != plan->steps) Py_RETURN_FALSE;
  } catch (const std::exception &) {
    Py_RETURN_FALSE;
  }
  for (const Bucket &b : plan->buckets)
    for (int32_t i : b.idx)
      if (plan->steps[i] != plan->steps[b.idx[0]]) Py_RETURN_FALSE;
  for (const Bucket &b : plan->buckets)
    for (size_t k = 0; k < b.idx.size(); ++k) reinterpret_cast<void **>(b.arr + k * b.stride)[1] = plan->fresh[(size_t)b.idx[k]];
  Py_RETURN_TRUE;
}

// whether a bucket of small tensors is at the step of the bucket in whose call it goes
bool together(const Plan &plan, const Bucket &small) {
  for (const Bucket &b : plan.buckets)
    if (b.with >= 0 && &plan.buckets[(size_t)b.with] == &small) return plan.steps[b.idx[0]] == plan.steps[small.idx[0]];
  return false;
}

// run(plan, beta1, beta2, lr, weight_decay, eps, options' address or 0, seed): advances the step counters and makes the
// launches; the first status that is not 0 and its bucket's number, or (0, number of buckets), or None with nothing done
PyObject *run(PyObject *, PyObject *const *args, Py_ssize_t n) {
  Plan *plan = n == 8 ? plan_of(args[0]) : nullptr;
  if (!plan) return n == 8 ? nullptr : (PyErr_SetString(PyExc_TypeError, "run takes eight arguments"), nullptr);
  float x[5];
  void *stream = nullptr;
  if (!numbers(args + 1, 5, x)) Py_RETURN_NONE;
  const q4adamw_grad_options *options = static_cast<const q4adamw_grad_options *>(PyLong_AsVoidPtr(args[6]));
  const uint64_t seed = PyLong_AsUnsignedLongLongMask(args[7]);
  if (PyErr_Occurred()) return nullptr;
  if (!stream_of(plan->device, &stream)) Py_RETURN_NONE;
  for (int64_t i = 0; i < plan->with_grad; ++i) plan->steps[i] += 1.0f;
  int rc = 0;
  size_t k = 0;
  Py_BEGIN_ALLOW_THREADS
  for (; k < plan->buckets.size(); ++k) {
    const Bucket &b = plan->buckets[k];
    const float step = plan->steps[b.idx[0]];
    const int count = (int)b.idx.size();
    if (b.taken && together(*plan, b)) continue;
    if (b.with >= 0 && together(*plan, plan->buckets[(size_t)b.with])) {
      const Bucket &o = plan->buckets[(size_t)b.with];
      rc = lib.both(reinterpret_cast<const q4adamw_tensor *>(b.arr), count, reinterpret_cast<const q4adamw_small_tensor *>(o.arr), (int)o.idx.size(),
                    b.kind == 2, b.salts, seed, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4], step, options, stream);
      if (rc != 0) break;
      continue;
    }
    switch (b.kind) {
      case 0:
        rc = lib.small(reinterpret_cast<const q4adamw_small_tensor *>(b.arr), count, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4], step, options, stream);
        break;
      case 1:
        rc = lib.multi(reinterpret_cast<const q4adamw_tensor *>(b.arr), count, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4], step, options, stream);
        break;
      case 2:
        rc = lib.multi_sr(reinterpret_cast<const q4adamw_tensor *>(b.arr), count, b.salts, seed, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4], step,
                          options, stream);
        break;
      case 3:
        rc = lib.rank1(reinterpret_cast<const q4adamw_rank1_tensor *>(b.arr), count, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4], step, options, stream);
        break;
      default:
        rc = lib.rank1_sr(reinterpret_cast<const q4adamw_rank1_tensor *>(b.arr), count, b.salts, seed, b.p_tag, b.g_tag, x[0], x[1], x[2], x[3], x[4],
                          step, options, stream);
    }
    if (rc != 0) break;
  }
  Py_END_ALLOW_THREADS
  return Py_BuildValue("in", rc, (Py_ssize_t)k);
}

PyMethodDef kMethods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(bind)), METH_FASTCALL, nullptr},
    {"fused_4bit", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(fused_4bit)), METH_FASTCALL, nullptr},
    {"fused_single_tensor", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(fused_single_tensor)), METH_FASTCALL, nullptr},
    {"gradients", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(gradients)), METH_FASTCALL, nullptr},
    {"plan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(make_plan)), METH_FASTCALL, nullptr},
    {"refresh", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(refresh)), METH_FASTCALL, nullptr},
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(run)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_q4host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__q4host(void) {
  const char *const names[3] = {"step", "exp_avg", "exp_avg_sq"};
  for (int k = 0; k < 3; ++k)
    if (!(state_keys[k] = PyUnicode_InternFromString(names[k]))) return nullptr;
  PyObject *module = PyModule_Create(&kModule);
  if (module && (PyModule_AddStringConstant(module, "built_for", Q4HOST_BUILT_FOR) < 0 ||
                 PyModule_AddIntConstant(module, "library_version", Q4ADAMW_VERSION) < 0))
    Py_CLEAR(module);
  return module;
}
