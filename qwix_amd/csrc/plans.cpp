// Launch plans: what an operator call does on the device, kept per operand metadata and replayed without Python.
//
// An operator (quantize, dot_general, ...) decides from shapes, strides, dtypes and options which buffers to allocate and
// which entry points of libqwix_hip.so to call with which constants; that costs tens of microseconds of Python, more than
// most of the kernels.  None of it depends on the data or on where it lies.  qwix_amd/plans.py writes the decision down
// once -- allocations, calls, results -- and this module finds it again by the operands' metadata and carries it out:
// nothing here is keyed by the address or the identity of an operand, and nothing outlives a call but the plan.
//   run(fixed, *operands): the signature is the fixed part (a hashable Python object with the options) and, per
// operand, dtype, device, shape, strides and the alignment of its memory.
//   Thread safety: the table is only touched under the interpreter lock; allocations and launches run without it, on a plan
// that the call holds a reference to.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <memory>
#include <string>
#include <tuple>
#include <unordered_map>
#include <utility>
#include <vector>

#include "../../include/qwix_hip.h"

namespace {

// ---------------------------------------------------------------------------------------------- typed calls
// One machine word per argument, converted to the entry point's own parameter types.
union Slot {
  int64_t i;
  double f;
  void* p;
};
template <typename T>
T as(const Slot& s) {
  if constexpr (std::is_pointer_v<T>) return static_cast<T>(s.p);
  else if constexpr (std::is_floating_point_v<T>) return static_cast<T>(s.f);
  else return static_cast<T>(s.i);
}
template <typename... A, size_t... I>
int call_with(int (*fn)(A...), const Slot* s, std::index_sequence<I...>) {
  return fn(as<A>(s[I])...);
}
template <auto Fn>
struct Entry;
template <typename... A, int (*Fn)(A...)>
struct Entry<Fn> {
  static constexpr int arity = sizeof...(A);
  static int call(const Slot* s) { return call_with(Fn, s, std::index_sequence_for<A...>{}); }
};
struct EntryPoint {
  const char* name;
  int arity;
  int (*call)(const Slot*);
};
#define QWIX_ENTRY(fn) EntryPoint{#fn, Entry<&fn>::arity, &Entry<&fn>::call}
const EntryPoint kEntries[] = {
    QWIX_ENTRY(qwix_hip_quantize),          QWIX_ENTRY(qwix_hip_quantize_with_scale), QWIX_ENTRY(qwix_hip_dequantize),
    QWIX_ENTRY(qwix_hip_dequantize_rm),     QWIX_ENTRY(qwix_hip_transpose_q),         QWIX_ENTRY(qwix_hip_qgemm),
    QWIX_ENTRY(qwix_hip_qgemm_ws),          QWIX_ENTRY(qwix_hip_qgemm_zp),            QWIX_ENTRY(qwix_hip_qgemm_ragged),
    QWIX_ENTRY(qwix_hip_qgemm_batched),     QWIX_ENTRY(qwix_hip_qgemm_dynamic_act),   QWIX_ENTRY(qwix_hip_qgemm_hadamard_act),
    QWIX_ENTRY(qwix_hip_ksum_i8),           QWIX_ENTRY(qwix_hip_ksum_groups),         QWIX_ENTRY(qwix_hip_qgemm_grouped_ws),
    QWIX_ENTRY(qwix_hip_qgemm_grouped_zp),  QWIX_ENTRY(qwix_hip_gemm_bf16),           QWIX_ENTRY(qwix_hip_gemm_bf16_wq_ws),
    QWIX_ENTRY(qwix_hip_gemv_wq),           QWIX_ENTRY(qwix_hip_gemv_wq_zp),          QWIX_ENTRY(qwix_hip_gemv_wq_groups),
    QWIX_ENTRY(qwix_hip_gemm_wq_groups),    QWIX_ENTRY(qwix_hip_qgemm_zp_i8),
    QWIX_ENTRY(qwix_hip_qgemm_batched_act),  QWIX_ENTRY(qwix_hip_qgemm_batched_act_kn),  QWIX_ENTRY(qwix_hip_qgemm_dynamic_relu),  QWIX_ENTRY(qwix_hip_fwht),              QWIX_ENTRY(qwix_hip_fwht_quantize),
};
constexpr int kMaxArgs = 32;

// ---------------------------------------------------------------------------------------------- plans
enum ArgKind { kConst, kConstFloat, kOperand, kBuffer, kStream };
struct Arg {
  ArgKind kind;
  int index;    // operand or buffer
  Slot value;   // constant, or byte offset
};
struct Call {
  const EntryPoint* entry;
  std::vector<Arg> args;
};
struct Buffer {
  std::vector<int64_t> sizes, strides;
  at::TensorOptions options;
  bool contiguous;
};
struct Result {
  int buffer;
  bool whole;  // the buffer as it was allocated
  std::vector<int64_t> sizes, strides;
  int64_t offset;
};
struct Plan {
  std::vector<Buffer> buffers;
  std::vector<Call> calls;
  std::vector<Result> results;
  PyObject* rebuild = nullptr;  // rebuild(*results) is what the call returns; null: the only result
  int device = 0;
  ~Plan() { Py_XDECREF(rebuild); }
};
struct Seen {
  PyObject* fixed;
  std::string signature;
  std::shared_ptr<const Plan> plan;  // a call holds its own reference: `rebuild` is Python, other threads run meanwhile
  int times = 0;
};
struct Cache {
  std::unordered_map<uint64_t, std::vector<Seen>> seen;
  size_t count = 0;
  void clear() {
    for (auto& [h, v] : seen)
      for (Seen& s : v) Py_DECREF(s.fixed);
    seen.clear();
    count = 0;
  }
};
constexpr size_t kMaxSeen = 8192;  // signatures remembered; beyond it a cache starts anew

PyObject *g_qarray = nullptr, *g_int4 = nullptr, *g_stream = nullptr, *g_fail = nullptr;
int g_record_at = 0;
PyObject *s_qvalue, *s_scale, *s_zero_point, *s_qtype, *s_data, *s_packed_axis;

struct Operands {
  std::string signature;
  std::vector<const at::Tensor*> tensors;
  std::vector<PyObject*> keep;  // attributes read on the way
  ~Operands() {
    for (PyObject* o : keep) Py_DECREF(o);
  }
  void put(int64_t v) { signature.append(reinterpret_cast<const char*>(&v), sizeof v); }
  bool tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.layout() != at::kStrided || t.is_neg()) return false;
    put(static_cast<int64_t>(t.scalar_type()) | static_cast<int64_t>(t.device().index()) << 8 | t.dim() << 16 |
        static_cast<int64_t>(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) << 32);
    const auto sizes = t.sizes(), strides = t.strides();
    signature.append(reinterpret_cast<const char*>(sizes.data()), sizes.size() * 8);
    signature.append(reinterpret_cast<const char*>(strides.data()), strides.size() * 8);
    tensors.push_back(&t);
    return true;
  }
  PyObject* attribute(PyObject* o, PyObject* name) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (a != nullptr) keep.push_back(a);
    return a;
  }
  bool values(PyObject* o) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) == g_int4) {
      PyObject* axis = attribute(o, s_packed_axis);
      if (axis == nullptr) return false;
      put(-4 - PyLong_AsLongLong(axis));
      PyObject* data = attribute(o, s_data);
      return data != nullptr && tensor(data);
    }
    return tensor(o);
  }
  // False: not a kind of operand that plans are kept for (a Python error may be set; the caller clears it).
  bool add(PyObject* o) {
    if (o == Py_None) {
      put(-1);
      return true;
    }
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) == g_qarray) {
      PyObject *q = attribute(o, s_qvalue), *s = attribute(o, s_scale), *z = attribute(o, s_zero_point), *t = attribute(o, s_qtype);
      if (!q || !s || !z || !t || !PyUnicode_Check(t)) return false;
      Py_ssize_t n = 0;
      const char* name = PyUnicode_AsUTF8AndSize(t, &n);
      if (name == nullptr) return false;
      put(-2);
      signature.append(name, static_cast<size_t>(n) + 1);
      if (!values(q) || !tensor(s)) return false;
      if (z == Py_None) {
        put(-3);
        return true;
      }
      return tensor(z);
    }
    return values(o);
  }
};

uint64_t hash_of(PyObject* fixed, const std::string& signature, bool* ok) {
  const Py_hash_t h = PyObject_Hash(fixed);
  *ok = h != -1;
  return std::hash<std::string>()(signature) * 0x9E3779B97F4A7C15ull + static_cast<uint64_t>(h);
}

Seen* lookup(Cache& c, PyObject* fixed, const std::string& signature, uint64_t h) {
  auto it = c.seen.find(h);
  if (it == c.seen.end()) return nullptr;
  for (Seen& s : it->second) {
    if (s.signature != signature) continue;
    const int eq = PyObject_RichCompareBool(s.fixed, fixed, Py_EQ);
    if (eq < 0) PyErr_Clear();
    if (eq > 0) return &s;
  }
  return nullptr;
}

// The interpreter lock let go for a scope: allocations can wait for the device and launches for room in its queue, and other
// threads (a host callback that a stream waits for among them) must be able to run meanwhile.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// Allocates and launches; no Python inside.  Returns a refused call's entry point and status, or {nullptr, 0}.
std::pair<const EntryPoint*, int> carry_out(const Plan& p, void* const* operands, void* stream, at::Tensor* buffers) {
  const Unlocked unlocked;
  for (size_t k = 0; k < p.buffers.size(); ++k) {
    const Buffer& b = p.buffers[k];
    buffers[k] = b.contiguous ? at::empty(b.sizes, b.options) : at::empty_strided(b.sizes, b.strides, b.options);
  }
  for (const Call& c : p.calls) {
    Slot slots[kMaxArgs];
    for (size_t k = 0; k < c.args.size(); ++k) {
      const Arg& a = c.args[k];
      switch (a.kind) {
        case kOperand: slots[k].p = static_cast<char*>(operands[a.index]) + a.value.i; break;
        case kBuffer: slots[k].p = static_cast<char*>(buffers[a.index].data_ptr()) + a.value.i; break;
        case kStream: slots[k].p = stream; break;
        default: slots[k] = a.value;
      }
    }
    if (const int status = c.entry->call(slots)) return {c.entry, status};
  }
  return {nullptr, 0};
}

PyObject* run_plan(const Plan& p, const Operands& ops) {
  PyObject* index = PyLong_FromLong(p.device);
  PyObject* handle = PyObject_CallOneArg(g_stream, index);
  Py_DECREF(index);
  if (handle == nullptr) return nullptr;
  void* stream = reinterpret_cast<void*>(static_cast<intptr_t>(PyLong_AsLongLong(handle)));
  Py_DECREF(handle);
  // (the operands' objects are held by the caller and by `ops`; their addresses are read under the lock)
  std::vector<void*> operands;
  for (const at::Tensor* t : ops.tensors) operands.push_back(t->data_ptr());
  at::Tensor buffers[16];
  const auto [refused, status] = carry_out(p, operands.data(), stream, buffers);
  if (refused != nullptr) {
    PyObject* r = PyObject_CallFunction(g_fail, "si", refused->name, status);  // raises
    Py_XDECREF(r);
    return nullptr;
  }
  auto result = [&](const Result& r) -> PyObject* {
    at::Tensor& b = buffers[r.buffer];
    return THPVariable_Wrap(r.whole ? b : b.as_strided(r.sizes, r.strides, r.offset));
  };
  if (p.rebuild == nullptr) return result(p.results[0]);
  PyObject* out[8];
  const size_t nr = p.results.size();
  for (size_t k = 0; k < nr; ++k) out[k] = result(p.results[k]);
  PyObject* r = PyObject_Vectorcall(p.rebuild, out, nr, nullptr);
  for (size_t k = 0; k < nr; ++k) Py_DECREF(out[k]);
  return r;
}

Cache& cache() {
  static Cache* c = new Cache;  // not destroyed: its Python objects must not be released behind the interpreter
  return *c;
}
thread_local int t_recording = 0;  // a plan is being recorded on this thread: nested operators take their ordinary path

// recording(+1 / -1)
PyObject* recording(PyObject*, PyObject* by) {
  t_recording += static_cast<int>(PyLong_AsLong(by));
  Py_RETURN_NONE;
}

// run(fixed, *operands): the result of a kept plan; None: none is kept; True: none is kept, and this kind of call has come
// up so often (the number setup was given) that it is worth recording.
PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) try {
  if (t_recording) Py_RETURN_NONE;
  Cache* const c = &cache();
  Operands ops;
  for (Py_ssize_t k = 1; k < n; ++k)
    if (!ops.add(args[k])) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
  bool ok;
  const uint64_t h = hash_of(args[0], ops.signature, &ok);
  if (!ok) {  // options that cannot be hashed (lists)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  Seen* s = lookup(*c, args[0], ops.signature, h);
  if (s == nullptr) {
    if (c->count >= kMaxSeen) c->clear();
    Py_INCREF(args[0]);
    c->seen[h].push_back(Seen{args[0], std::move(ops.signature), {}, 1});
    ++c->count;
    Py_RETURN_NONE;
  }
  if (const std::shared_ptr<const Plan> p = s->plan) return run_plan(*p, ops);
  if (++s->times == g_record_at) Py_RETURN_TRUE;
  Py_RETURN_NONE;
} catch (const std::exception&) {  // out of memory and the like: the ordinary path meets it again and raises as torch does
  PyErr_Clear();
  Py_RETURN_NONE;
}

bool int_list(PyObject* o, std::vector<int64_t>* out) {
  PyObject* f = PySequence_Fast(o, "a sequence of integers");
  if (f == nullptr) return false;
  for (Py_ssize_t k = 0; k < PySequence_Fast_GET_SIZE(f); ++k) out->push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(f, k)));
  Py_DECREF(f);
  return !PyErr_Occurred();
}

// keep(fixed, operands, buffers, calls, results, rebuild)
//   buffers: [(sizes, strides, a tensor of the dtype and device)], calls: [(name, [(kind, index, value)])],
//   results: [(buffer, sizes, strides, offset)], rebuild: callable or None
PyObject* keep(PyObject*, PyObject* args) {
  PyObject *fixed, *operands, *buffers, *calls, *results, *rebuild;
  if (!PyArg_ParseTuple(args, "OO!O!O!O!O", &fixed, &PyTuple_Type, &operands, &PyList_Type, &buffers, &PyList_Type,
                        &calls, &PyList_Type, &results, &rebuild))
    return nullptr;
  Cache* const c = &cache();
  Operands ops;
  for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(operands); ++k)
    if (!ops.add(PyTuple_GET_ITEM(operands, k))) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  bool ok;
  const uint64_t h = hash_of(fixed, ops.signature, &ok);
  if (!ok) return nullptr;
  Seen* s = lookup(*c, fixed, ops.signature, h);
  if (s == nullptr || s->plan != nullptr || PyList_GET_SIZE(buffers) > 16 || PyList_GET_SIZE(results) > 8) Py_RETURN_FALSE;
  auto p = std::make_shared<Plan>();
  for (Py_ssize_t k = 0; k < PyList_GET_SIZE(buffers); ++k) {
    PyObject *sizes, *strides, *like;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(buffers, k), "OOO", &sizes, &strides, &like)) return nullptr;
    Buffer b;
    if (!int_list(sizes, &b.sizes) || !int_list(strides, &b.strides)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(like);
    b.options = at::TensorOptions().dtype(t.scalar_type()).device(t.device());
    p->device = t.device().index();
    b.contiguous = true;
    int64_t want = 1;
    for (size_t d = b.sizes.size(); d-- > 0;) {
      if (b.sizes[d] != 1 && b.strides[d] != want) b.contiguous = false;
      want *= b.sizes[d];
    }
    p->buffers.push_back(std::move(b));
  }
  for (Py_ssize_t k = 0; k < PyList_GET_SIZE(calls); ++k) {
    const char* name;
    PyObject* list;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(calls, k), "sO!", &name, &PyList_Type, &list)) return nullptr;
    Call call{nullptr, {}};
    for (const EntryPoint& e : kEntries)
      if (std::strcmp(e.name, name) == 0) call.entry = &e;
    if (call.entry == nullptr || call.entry->arity != PyList_GET_SIZE(list) || call.entry->arity > kMaxArgs) Py_RETURN_FALSE;
    for (Py_ssize_t a = 0; a < PyList_GET_SIZE(list); ++a) {
      int kind, index;
      PyObject* value;
      if (!PyArg_ParseTuple(PyList_GET_ITEM(list, a), "iiO", &kind, &index, &value)) return nullptr;
      Arg arg{static_cast<ArgKind>(kind), index, {}};
      if (kind == kConstFloat) arg.value.f = PyFloat_AsDouble(value);
      else arg.value.i = PyLong_AsLongLong(value);
      if (PyErr_Occurred()) return nullptr;
      if ((kind == kOperand && index >= static_cast<int>(ops.tensors.size())) ||
          (kind == kBuffer && index >= static_cast<int>(p->buffers.size())))
        Py_RETURN_FALSE;
      call.args.push_back(arg);
    }
    p->calls.push_back(std::move(call));
  }
  for (Py_ssize_t k = 0; k < PyList_GET_SIZE(results); ++k) {
    Result r{};
    PyObject *sizes, *strides;
    long long offset;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(results, k), "iOOL", &r.buffer, &sizes, &strides, &offset)) return nullptr;
    if (!int_list(sizes, &r.sizes) || !int_list(strides, &r.strides) || r.buffer >= static_cast<int>(p->buffers.size())) return nullptr;
    r.offset = offset;
    const Buffer& b = p->buffers[r.buffer];
    r.whole = offset == 0 && r.sizes == b.sizes && r.strides == b.strides;
    p->results.push_back(std::move(r));
  }
  if (rebuild != Py_None) {
    Py_INCREF(rebuild);
    p->rebuild = rebuild;
  } else if (p->results.size() != 1) {
    Py_RETURN_FALSE;
  }
  s->plan = std::move(p);
  Py_RETURN_TRUE;
}

// tensors(*operands): the tensors that plans see in the operands, in their order, or None.
PyObject* tensors(PyObject*, PyObject* const* args, Py_ssize_t n) try {
  Operands ops;
  for (Py_ssize_t k = 0; k < n; ++k)
    if (!ops.add(args[k])) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
  PyObject* out = PyTuple_New(static_cast<Py_ssize_t>(ops.tensors.size()));
  for (size_t k = 0; k < ops.tensors.size(); ++k) PyTuple_SET_ITEM(out, static_cast<Py_ssize_t>(k), THPVariable_Wrap(*ops.tensors[k]));
  return out;
} catch (const std::exception&) {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// setup(QArray, Int4Tensor, current raw stream function, failure function, calls up to the recorded one)
PyObject* setup(PyObject*, PyObject* args) {
  if (!PyArg_ParseTuple(args, "OOOOi", &g_qarray, &g_int4, &g_stream, &g_fail, &g_record_at)) return nullptr;
  for (PyObject* o : {g_qarray, g_int4, g_stream, g_fail}) Py_INCREF(o);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"recording", recording, METH_O, nullptr},
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(run)), METH_FASTCALL, nullptr},
    {"keep", keep, METH_VARARGS, nullptr},
    {"tensors", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(tensors)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_plans", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__plans() {
  s_qvalue = PyUnicode_InternFromString("qvalue");
  s_scale = PyUnicode_InternFromString("scale");
  s_zero_point = PyUnicode_InternFromString("zero_point");
  s_qtype = PyUnicode_InternFromString("qtype");
  s_data = PyUnicode_InternFromString("data");
  s_packed_axis = PyUnicode_InternFromString("packed_axis");
  return PyModule_Create(&kModule);
}
