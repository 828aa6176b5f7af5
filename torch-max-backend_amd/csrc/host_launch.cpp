// Host side of a launch, native: the launchers in Python (eager_kernels/hip_ops.py) validate an operand layout once and
// leave a plan of its launch here; a later call with the same layout is one lookup, its allocations and the launch. And
// the step loop of a compiled graph (torch_compile_backend/compiler.py).
//
// What bounds a launch of a few microseconds of work is this path. Microseconds a call, in Python and here, with HIP's own
// 3.0 .. 3.5 in both: addmm of 128 x 768 x 768 8.9 -> 5.1, layer norm with statistics 12.4 -> 6.6, softmax 8.1 -> 4.3, a sum of
// rows 9.5 -> 5.0, argmax 9.0 -> 4.1. The step loop adds 0.2 a step (0.6 in Python): a GPT-2 forward of 1 x 128, some
// 380 steps and 100 launches, 1354 -> 890, a decode step of 32 x 499 1627 -> 1158.
//
// A plan's key is everything the launcher looks at: per tensor type, device, sizes, strides and the address modulo 16,
// and the call's other arguments. Addresses are not part of it: every call passes those of its own tensors, and
// allocates results and scratch of its own on PyTorch's allocator. Calls this file does not take (a subclass, a tensor without
// plain storage, an argument that is no constant, an unknown layout) return None and run in Python. All state is guarded by
// the interpreter lock, which is given up during the launch, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <deque>
#include <memory>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

#include "../../include/tmb_hip.h"

namespace {

// ---- calling an entry point with arguments put together at run time, through its own type ------------------------
struct Slot {
  int64_t i = 0;
  double d = 0.0;
};
template <typename A>
A slot_as(const Slot& s) {
  if constexpr (std::is_pointer_v<A>) return reinterpret_cast<A>(s.i);
  else if constexpr (std::is_floating_point_v<A>) return static_cast<A>(s.d);
  else return static_cast<A>(s.i);
}
template <typename F>
struct Thunk;
template <typename... A>
struct Thunk<int (*)(A...)> {
  static constexpr size_t count = sizeof...(A);
  template <size_t... I>
  static int spread(int (*f)(A...), const Slot* s, std::index_sequence<I...>) {
    return f(slot_as<A>(s[I])...);
  }
  static int call(void* f, const Slot* s) {
    return spread(reinterpret_cast<int (*)(A...)>(f), s, std::index_sequence_for<A...>{});
  }
};
struct Entry {
  const char* name;
  size_t args;
  int (*call)(void*, const Slot*);
};
#define TMB_ENTRY(f) {#f, Thunk<decltype(&f)>::count, &Thunk<decltype(&f)>::call}
const Entry kEntries[] = {
    TMB_ENTRY(tmb_softmax_rows), TMB_ENTRY(tmb_softmax_rows_scaled), TMB_ENTRY(tmb_layer_norm_rows),
    TMB_ENTRY(tmb_reduce_rows), TMB_ENTRY(tmb_reduce_cols), TMB_ENTRY(tmb_argmax_rows), TMB_ENTRY(tmb_gemm_ws),
    TMB_ENTRY(tmb_gemm_residual_ws), TMB_ENTRY(tmb_attention_fwd), TMB_ENTRY(tmb_attention_bwd),
    TMB_ENTRY(tmb_attention_f32_fwd), TMB_ENTRY(tmb_attention_f32_bwd), TMB_ENTRY(tmb_attention_decode),
    TMB_ENTRY(tmb_attention_decode_append), TMB_ENTRY(tmb_gelu), TMB_ENTRY(tmb_gather_rows),
    TMB_ENTRY(tmb_gelu_backward), TMB_ENTRY(tmb_softmax_backward_rows), TMB_ENTRY(tmb_layer_norm_backward_rows),
    TMB_ENTRY(tmb_layer_norm_backward_add_rows)};
#undef TMB_ENTRY
constexpr size_t kMostArgs = 32;

// ---- plans ----------------------------------------------------------------------------------------------------
enum Source : char { kConst, kTensor, kOutput, kScratch, kStream, kBlob };
struct Argument {
  Source source;
  int index = 0;
  Slot value;
};
struct Output {
  std::vector<int64_t> sizes, strides;  // (no strides: contiguous)
  bool strided = false;
  at::ScalarType type = at::kFloat;
};
struct Plan {
  std::vector<int64_t> key;
  std::vector<PyObject*> extras;  // owned
  const Entry* entry = nullptr;
  void* function = nullptr;
  std::vector<Argument> arguments;
  std::vector<std::vector<int64_t>> blobs;
  std::vector<Output> outputs;
  int64_t scratch = 0;
  bool single = true;
  std::vector<int> results;  // output numbers; -1: None
  uint64_t hash = 0;
  bool used = false;  // since it last stood in front of g_order
  ~Plan() {
    for (PyObject* o : extras) Py_DECREF(o);
  }
};
// (never destroyed: at the end of the process the interpreter that owns the plans' objects is gone)
std::unordered_map<uint64_t, std::vector<std::shared_ptr<Plan>>>& g_plans =
    *new std::unordered_map<uint64_t, std::vector<std::shared_ptr<Plan>>>;
// The plans in the order in which they may go once there are kMostPlans: from the front, and one that has been used since
// it last stood there goes to the back instead. A generation loop leaves a plan for every length of its cache; those of
// its other launches stay. (Some 2 KB each.)
std::deque<std::shared_ptr<Plan>>& g_order = *new std::deque<std::shared_ptr<Plan>>;
constexpr size_t kMostPlans = 8192;
PyObject* g_check = nullptr;  // check(name, status): raises

// Plain strided HIP tensors only; anything that a transform or a mode has wrapped runs in Python.
bool usable(const at::Tensor& t) {
  constexpr c10::DispatchKeySet odd(
      {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
       c10::DispatchKey::Functionalize, c10::DispatchKey::Batched, c10::DispatchKey::ZeroTensor,
       c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd) && t.has_storage();
}

// What a plan may hold on to of a call's other arguments: values that nobody can change. (A 0-dimensional tensor given for a
// number equals itself whatever it holds by then.)
bool constant(PyObject* o, int depth = 0) {
  if (o == Py_None || PyBool_Check(o) || PyLong_CheckExact(o) || PyFloat_CheckExact(o) || PyUnicode_CheckExact(o) ||
      THPDtype_Check(o))
    return true;
  if (!PyTuple_CheckExact(o) || depth > 1) return false;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(o); ++i)
    if (!constant(PyTuple_GET_ITEM(o, i), depth + 1)) return false;
  return true;
}

struct Call {
  std::vector<int64_t> key;
  std::vector<Py_hash_t> hashes;
  const at::Tensor* tensors[8];
  int count = 0;
  PyObject* const* extras = nullptr;
  Py_ssize_t extra_count = 0;
  uint64_t hash = 0;
};

// args: operation number, number of tensors, the tensors (None where absent), the other arguments. False: not a call for
// this file (no Python error is set).
bool read_call(PyObject* const* args, Py_ssize_t nargs, Call& c) {
  if (nargs < 3) return false;
  const long op = PyLong_AsLong(args[0]), n = PyLong_AsLong(args[1]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  if (n < 1 || n > 8 || nargs < 2 + n) return false;
  c.key.clear();
  c.key.push_back(op * 16 + n);
  c.count = static_cast<int>(n);
  for (long i = 0; i < n; ++i) {
    PyObject* o = args[2 + i];
    if (o == Py_None) {
      c.tensors[i] = nullptr;
      c.key.push_back(-1);
      continue;
    }
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!usable(t)) return false;
    c.tensors[i] = &t;
    const auto sizes = t.sizes();
    const auto strides = t.strides();
    c.key.push_back(static_cast<int64_t>(t.scalar_type()) | static_cast<int64_t>(t.get_device()) << 8 |
                    static_cast<int64_t>(sizes.size()) << 24 |
                    static_cast<int64_t>(reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) << 40);
    c.key.insert(c.key.end(), sizes.begin(), sizes.end());
    c.key.insert(c.key.end(), strides.begin(), strides.end());
  }
  if (c.tensors[0] == nullptr) return false;
  c.extras = args + 2 + n;
  c.extra_count = nargs - 2 - n;
  uint64_t h = 1469598103934665603ull;
  auto mix = [&](uint64_t v) { h = (h ^ v) * 1099511628211ull, h ^= h >> 29; };
  for (const int64_t v : c.key) mix(static_cast<uint64_t>(v));
  for (Py_ssize_t i = 0; i < c.extra_count; ++i) {
    if (!constant(c.extras[i])) return false;
    const Py_hash_t v = PyObject_Hash(c.extras[i]);
    if (v == -1) {
      PyErr_Clear();
      return false;
    }
    mix(static_cast<uint64_t>(v));
  }
  c.hash = h;
  return true;
}

std::shared_ptr<Plan> find(const Call& c) {
  const auto at = g_plans.find(c.hash);
  if (at == g_plans.end()) return nullptr;
  for (const auto& plan : at->second) {
    if (plan->key != c.key || static_cast<Py_ssize_t>(plan->extras.size()) != c.extra_count) continue;
    bool same = true;
    for (Py_ssize_t i = 0; same && i < c.extra_count; ++i) {
      PyObject *mine = plan->extras[i], *asked = c.extras[i];
      if (mine == asked) continue;
      // (1, True and 1.0 are equal, but not the same argument to every launcher)
      const int equal = Py_TYPE(mine) == Py_TYPE(asked) ? PyObject_RichCompareBool(mine, asked, Py_EQ) : 0;
      if (equal < 0) PyErr_Clear();
      same = equal == 1;
    }
    if (same) {
      plan->used = true;
      return plan;
    }
  }
  return nullptr;
}

void drop_one() {
  while (g_order.front()->used) {  // (ends: each one passed is marked unused)
    g_order.front()->used = false;
    g_order.push_back(std::move(g_order.front()));
    g_order.pop_front();
  }
  const std::shared_ptr<Plan> plan = std::move(g_order.front());
  g_order.pop_front();
  const auto at = g_plans.find(plan->hash);
  auto& same_hash = at->second;
  same_hash.erase(std::find(same_hash.begin(), same_hash.end(), plan));
  if (same_hash.empty()) g_plans.erase(at);
}

PyObject* launch(const Plan& plan, const Call& c) {
  at::Tensor outputs[8], scratch;
  const auto device = c.tensors[0]->device();
  for (size_t i = 0; i < plan.outputs.size(); ++i) {
    const Output& o = plan.outputs[i];
    const auto options = at::TensorOptions().dtype(o.type).device(device);
    outputs[i] = o.strided ? at::empty_strided(o.sizes, o.strides, options) : at::empty(o.sizes, options);
  }
  if (plan.scratch > 0) scratch = at::empty({plan.scratch}, at::TensorOptions().dtype(at::kByte).device(device));
  Slot slots[kMostArgs];
  for (size_t i = 0; i < plan.arguments.size(); ++i) {
    const Argument& a = plan.arguments[i];
    const void* p = nullptr;
    switch (a.source) {
      case kConst: slots[i] = a.value; continue;
      case kTensor: p = c.tensors[a.index] ? c.tensors[a.index]->const_data_ptr() : nullptr; break;
      case kOutput: p = outputs[a.index].data_ptr(); break;
      case kScratch: p = plan.scratch > 0 ? scratch.data_ptr() : nullptr; break;
      case kStream: p = c10::hip::getCurrentHIPStream().stream(); break;
      case kBlob: p = plan.blobs[a.index].data(); break;
    }
    slots[i].i = static_cast<int64_t>(reinterpret_cast<intptr_t>(p));
  }
  int status;
  Py_BEGIN_ALLOW_THREADS;
  status = plan.entry->call(plan.function, slots);
  Py_END_ALLOW_THREADS;
  if (status != 0) {
    PyObject* r = PyObject_CallFunction(g_check, "si", plan.entry->name, status);
    if (r != nullptr) {
      Py_DECREF(r);
      PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", plan.entry->name, status);
    }
    return nullptr;
  }
  if (plan.single) return THPVariable_Wrap(outputs[plan.results[0]]);
  PyObject* result = PyTuple_New(static_cast<Py_ssize_t>(plan.results.size()));
  if (result == nullptr) return nullptr;
  for (size_t i = 0; i < plan.results.size(); ++i) {
    PyObject* item = Py_None;
    if (plan.results[i] >= 0) {
      item = THPVariable_Wrap(outputs[plan.results[i]]);
      if (item == nullptr) {
        Py_DECREF(result);
        return nullptr;
      }
    } else {
      Py_INCREF(item);
    }
    PyTuple_SET_ITEM(result, static_cast<Py_ssize_t>(i), item);
  }
  return result;
}

PyObject* planned(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Call c;  // (its vectors: one allocation a call)
  c.key.reserve(96);
  if (!read_call(args, nargs, c)) Py_RETURN_NONE;
  const std::shared_ptr<Plan> plan = find(c);
  if (plan == nullptr) Py_RETURN_NONE;
  return launch(*plan, c);
  END_HANDLE_TH_ERRORS
}

bool read_ints(PyObject* o, std::vector<int64_t>& out) {
  PyObject* seq = PySequence_Fast(o, "plan: a sequence of numbers");
  if (seq == nullptr) return false;
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); ++i)
    out.push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i)));
  Py_DECREF(seq);
  return !PyErr_Occurred();
}

// keep(spec, operation, number of tensors, tensors.., other arguments..). spec = (name, address, arguments, outputs,
// scratch bytes, result): an argument is a number, ("t", tensor number), ("o", output number), "scratch", "stream" or a
// tuple of numbers (passed as a pointer to them); an output (sizes, strides or None, dtype); the result an output
// number or a tuple of them and None.
PyObject* keep(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Call c;
  if (nargs < 4 || !read_call(args + 1, nargs - 1, c)) Py_RETURN_FALSE;
  auto plan = std::make_shared<Plan>();
  const char* name;
  unsigned long long address;
  PyObject *arguments, *outputs, *result;
  long long scratch;
  if (!PyArg_ParseTuple(args[0], "sKO!O!LO", &name, &address, &PyTuple_Type, &arguments, &PyTuple_Type, &outputs, &scratch,
                        &result))
    return nullptr;
  for (const Entry& e : kEntries)
    if (std::string(e.name) == name) plan->entry = &e;
  if (plan->entry == nullptr || plan->entry->args != static_cast<size_t>(PyTuple_GET_SIZE(arguments)) ||
      plan->entry->args > kMostArgs || PyTuple_GET_SIZE(outputs) > 8) {
    PyErr_Format(PyExc_ValueError, "plan: %s does not take %zd arguments", name, PyTuple_GET_SIZE(arguments));
    return nullptr;
  }
  plan->function = reinterpret_cast<void*>(address);
  plan->scratch = scratch;
  plan->key = c.key;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(arguments); ++i) {
    PyObject* o = PyTuple_GET_ITEM(arguments, i);
    Argument a{kConst};
    if (o == Py_None) {
    } else if (PyUnicode_Check(o)) {
      a.source = PyUnicode_CompareWithASCIIString(o, "stream") == 0 ? kStream : kScratch;
    } else if (PyTuple_Check(o) && PyTuple_GET_SIZE(o) == 2 && PyUnicode_Check(PyTuple_GET_ITEM(o, 0))) {
      a.source = PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(o, 0), "t") == 0 ? kTensor : kOutput;
      a.index = static_cast<int>(PyLong_AsLong(PyTuple_GET_ITEM(o, 1)));
      if (a.index < 0 || a.index >= (a.source == kTensor ? c.count : static_cast<int>(PyTuple_GET_SIZE(outputs)))) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_IndexError, "plan: no such tensor");
        return nullptr;
      }
    } else if (PyTuple_Check(o)) {
      a.source = kBlob;
      a.index = static_cast<int>(plan->blobs.size());
      plan->blobs.emplace_back();
      if (!read_ints(o, plan->blobs.back())) return nullptr;
    } else if (PyFloat_Check(o)) {
      a.value.d = PyFloat_AS_DOUBLE(o);
    } else {
      a.value.i = PyLong_AsLongLong(o);
    }
    if (PyErr_Occurred()) return nullptr;
    plan->arguments.push_back(a);
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(outputs); ++i) {
    PyObject *sizes, *strides, *dtype;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(outputs, i), "OOO", &sizes, &strides, &dtype)) return nullptr;
    Output o;
    if (!THPDtype_Check(dtype) || !read_ints(sizes, o.sizes)) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "plan: an output has sizes, strides and a dtype");
      return nullptr;
    }
    o.type = reinterpret_cast<THPDtype*>(dtype)->scalar_type;
    o.strided = strides != Py_None;
    if (o.strided && !read_ints(strides, o.strides)) return nullptr;
    plan->outputs.push_back(std::move(o));
  }
  plan->single = !PyTuple_Check(result);
  for (Py_ssize_t i = 0; i < (plan->single ? 1 : PyTuple_GET_SIZE(result)); ++i) {
    PyObject* o = plan->single ? result : PyTuple_GET_ITEM(result, i);
    const long at = o == Py_None ? -1 : PyLong_AsLong(o);
    if (PyErr_Occurred()) return nullptr;
    if (at >= static_cast<long>(plan->outputs.size()) || (at < 0 && plan->single)) {
      PyErr_SetString(PyExc_IndexError, "plan: no such output");
      return nullptr;
    }
    plan->results.push_back(static_cast<int>(at));
  }
  for (Py_ssize_t i = 0; i < c.extra_count; ++i) {
    Py_INCREF(c.extras[i]);
    plan->extras.push_back(c.extras[i]);
  }
  if (find(c) != nullptr) Py_RETURN_FALSE;
  if (g_order.size() >= kMostPlans) drop_one();
  plan->hash = c.hash;
  g_order.push_back(plan);
  g_plans[c.hash].push_back(std::move(plan));
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* forget(PyObject*, PyObject*) {
  g_plans.clear();
  g_order.clear();
  Py_RETURN_NONE;
}

PyObject* set_check(PyObject*, PyObject* check) {
  Py_INCREF(check);
  Py_XSETREF(g_check, check);
  Py_RETURN_NONE;
}

// ---- the step loop of a compiled graph ---------------------------------------------------------------------------
// A step: (function, argument template, ((position, slot), ..) or None, keyword names, keyword values, node, out slot,
// slots released after it). Without positions the step's arguments are put together by `materialize(step number, env)`, which
// returns (arguments, keywords).
struct Step {
  PyObject* function;
  std::vector<PyObject*> arguments;  // positional ones, then the keywords' values; owned
  std::vector<std::pair<int, int>> from_slots;
  PyObject* names;  // keyword names or nullptr
  PyObject* node;
  bool flat;
  int positional;
  int out;
  std::vector<int> release;
};
struct Program {
  std::vector<Step> steps;
  size_t most_arguments = 0;  // of one step
  PyObject* materialize = nullptr;
  PyObject* current_node = nullptr;  // the context variable that names the running step's node
  ~Program() {
    for (Step& s : steps) {
      Py_DECREF(s.function);
      Py_XDECREF(s.names);
      Py_DECREF(s.node);
      for (PyObject* o : s.arguments) Py_DECREF(o);
    }
    Py_XDECREF(materialize);
    Py_XDECREF(current_node);
  }
};
constexpr const char* kProgram = "tmb_program";
void free_program(PyObject* capsule) { delete static_cast<Program*>(PyCapsule_GetPointer(capsule, kProgram)); }

PyObject* program(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *steps, *materialize, *current_node;
  if (!PyArg_ParseTuple(args, "O!OO", &PyList_Type, &steps, &materialize, &current_node)) return nullptr;
  auto p = std::make_unique<Program>();
  Py_INCREF(materialize);
  p->materialize = materialize;
  Py_INCREF(current_node);
  p->current_node = current_node;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(steps); ++i) {
    PyObject *function, *arguments, *from, *names, *values, *node, *release;
    int out;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(steps, i), "OO!OOO!OiO!", &function, &PyTuple_Type, &arguments, &from, &names,
                          &PyTuple_Type, &values, &node, &out, &PyTuple_Type, &release))
      return nullptr;
    p->steps.emplace_back();
    Step& s = p->steps.back();
    Py_INCREF(function);
    s.function = function;
    Py_INCREF(node);
    s.node = node;
    s.names = nullptr;
    if (names != Py_None) {
      Py_INCREF(names);
      s.names = names;
    }
    s.positional = static_cast<int>(PyTuple_GET_SIZE(arguments));
    for (PyObject* part : {arguments, values})
      for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(part); ++j) {
        Py_INCREF(PyTuple_GET_ITEM(part, j));
        s.arguments.push_back(PyTuple_GET_ITEM(part, j));
      }
    p->most_arguments = std::max(p->most_arguments, s.arguments.size());
    s.flat = from != Py_None;
    if (s.flat) {
      if (!PyTuple_Check(from)) {
        PyErr_SetString(PyExc_TypeError, "program: positions of slots");
        return nullptr;
      }
      for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(from); ++j) {
        int position, slot;
        if (!PyArg_ParseTuple(PyTuple_GET_ITEM(from, j), "ii", &position, &slot)) return nullptr;
        if (position < 0 || position >= s.positional || slot < 0) {
          PyErr_SetString(PyExc_IndexError, "program: position of a slot");
          return nullptr;
        }
        s.from_slots.emplace_back(position, slot);
      }
    }
    s.out = out;
    for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(release); ++j) {
      s.release.push_back(static_cast<int>(PyLong_AsLong(PyTuple_GET_ITEM(release, j))));
      if (PyErr_Occurred()) return nullptr;
    }
  }
  PyObject* capsule = PyCapsule_New(p.get(), kProgram, free_program);
  if (capsule != nullptr) p.release();
  return capsule;
  END_HANDLE_TH_ERRORS
}

// run(program, env, failed): the steps in order, results into the list `env`. A step that raises leaves its number in
// `failed`.
PyObject* run(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *capsule, *env, *failed;
  if (!PyArg_ParseTuple(args, "OO!O!", &capsule, &PyList_Type, &env, &PyList_Type, &failed)) return nullptr;
  auto* p = static_cast<Program*>(PyCapsule_GetPointer(capsule, kProgram));
  if (p == nullptr) return nullptr;
  const Py_ssize_t slots = PyList_GET_SIZE(env);
  auto put = [&](int slot, PyObject* value) {  // takes the reference
    if (slot < 0 || slot >= slots || PyList_GET_SIZE(env) != slots) {
      Py_DECREF(value);
      PyErr_SetString(PyExc_IndexError, "program: no such slot");
      return false;
    }
    return PyList_SetItem(env, slot, value) == 0;
  };
  std::vector<PyObject*> stack;
  stack.reserve(p->most_arguments + 1);  // (no allocation, and so nothing that throws, between a step's own actions)
  for (size_t i = 0; i < p->steps.size(); ++i) {
    const Step& s = p->steps[i];
    PyObject* token = PyContextVar_Set(p->current_node, s.node);
    if (token == nullptr) return nullptr;
    PyObject* result = nullptr;
    if (s.flat) {
      stack.assign(s.arguments.size() + 1, nullptr);  // (one in front, which a bound method may use)
      std::copy(s.arguments.begin(), s.arguments.end(), stack.begin() + 1);
      bool there = true;
      for (const auto& [position, slot] : s.from_slots) {
        there = there && slot < PyList_GET_SIZE(env);
        if (there) stack[position + 1] = PyList_GET_ITEM(env, slot);
      }
      if (there) {
        for (PyObject* o : stack) Py_XINCREF(o);  // (a step may drop its arguments from env by itself)
        result = PyObject_Vectorcall(s.function, stack.data() + 1,
                                     static_cast<size_t>(s.positional) | PY_VECTORCALL_ARGUMENTS_OFFSET, s.names);
        for (size_t j = 1; j < stack.size(); ++j) Py_XDECREF(stack[j]);
      } else {
        PyErr_SetString(PyExc_IndexError, "program: no such slot");
      }
    } else {
      PyObject* both = PyObject_CallFunction(p->materialize, "nO", static_cast<Py_ssize_t>(i), env);
      if (both != nullptr) {
        PyObject *a, *kw;
        if (PyArg_ParseTuple(both, "O!O!", &PyTuple_Type, &a, &PyDict_Type, &kw)) result = PyObject_Call(s.function, a, kw);
        Py_DECREF(both);
      }
    }
    if (result == nullptr) {
      PyObject *type, *value, *trace;
      PyErr_Fetch(&type, &value, &trace);
      if (PyContextVar_Reset(p->current_node, token) < 0) PyErr_Clear();
      Py_DECREF(token);
      PyObject* number = PyLong_FromSize_t(i);
      if (number == nullptr || PyList_Append(failed, number) < 0) PyErr_Clear();
      Py_XDECREF(number);
      PyErr_Restore(type, value, trace);
      return nullptr;
    }
    const int reset = PyContextVar_Reset(p->current_node, token);
    Py_DECREF(token);
    if (reset < 0) {
      Py_DECREF(result);
      return nullptr;
    }
    if (!put(s.out, result)) return nullptr;
    for (const int slot : s.release) {
      Py_INCREF(Py_None);
      if (!put(slot, Py_None)) return nullptr;
    }
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"planned", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(planned)), METH_FASTCALL,
     "planned(operation, n, tensors.., arguments..): the results of a launch whose layout has a plan, or None"},
    {"keep", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(keep)), METH_FASTCALL,
     "keep(spec, operation, n, tensors.., arguments..): leaves the plan of a launch"},
    {"forget", forget, METH_NOARGS, "forget(): drops all plans"},
    {"set_check", set_check, METH_O, "set_check(f): f(name, status) raises for a status that is not 0"},
    {"program", program, METH_VARARGS, "program(steps, materialize, current_node): the steps of a graph"},
    {"run", run, METH_VARARGS, "run(program, env, failed): runs them"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "tmb_host", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit_tmb_host() { return PyModule_Create(&kModule); }
