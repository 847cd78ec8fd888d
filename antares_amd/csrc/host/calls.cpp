// The call path of the operators in native code: a CPython extension on torch's C++ tensors.
//
// An operator call from Python used to cost 9 to 10 us of host time (argument checks, shape look-ups, output
// allocation through torch.empty, ctypes conversions), more than most of the kernels it launches.  What a call does
// depends only on the dtypes, shapes, devices, contiguity and 16-byte alignment of its tensors, on which of them share
// memory and on which arguments are given, so the Python side works it out once per such signature - a recipe: outputs and
// intermediates to allocate, kernels and library entry points to call, and where each argument comes from - and this file
// replays it: signature, look-up, allocation, launches.  Anything unusual (an argument that is no plain tensor, a new
// signature) goes to the operator's Python method, which checks everything and raises the errors; a recipe holds no data
// and no result, only how to compute it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cstddef>
#include <memory>
#include <string>
#include <string_view>
#include <unordered_map>
#include <vector>

namespace {

constexpr int kMaxSlots = 24;            // flattened arguments of a call
constexpr int kMaxInts = 20;             // integer and pointer arguments of a library entry point
constexpr int kMaxFloats = 4;
// A recipe costs as much to make as a call without one (attention over a cache that grows: 9 us of host time a call, 17 with a
// recipe made each time, 4 replayed).  An operator whose last kCredit recipes have not been used is called with another
// signature every time: it gets one only when a signature is met again.  The table holds the positions of a long sequence;
// it is emptied when it is full.
constexpr int kCredit = 8;
constexpr size_t kMaxRecipes = 8192;     // per operator
constexpr size_t kMet = 8192;            // signatures that are remembered, by a part of their hash

PyObject* g_error = nullptr;             // ArtError
PyObject* g_parameter = nullptr;         // torch.nn.Parameter
const char* (*g_last_error)() = nullptr;
int (*g_launch)(void*, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, void*, const uint64_t*, int) = nullptr;
unsigned long long g_generation = 0;     // recipes of an older generation are worked out again

struct Arg {
  enum Kind { kPointer, kInt, kFloat, kStream, kSlotInt, kSlotFloat } kind;
  int index;
  uint64_t i;
  float f;
};
struct Launch {
  void* fn;
  bool kernel;
  unsigned grid[3], block[3];
  std::vector<Arg> args;
};
struct Alloc {
  at::ScalarType dtype;
  std::vector<int64_t> sizes;
};
struct Recipe {
  unsigned long long generation;
  uint64_t tuned_version, config_version;
  int device;
  bool device_stream;                                    // the stream of the tensors' device, or of the current device
  int slots;
  std::vector<Alloc> allocs;
  std::vector<Launch> launches;
  std::vector<std::pair<int, bool>> numbers;             // slots whose numbers are passed on; true: as a float
  std::vector<int> results;
  bool uses_stream, used;
};

struct Operator {
  PyObject_HEAD
  PyObject *tuned, *config, *fast_path;                  // attributes a recipe depends on: setting one empties the table
  std::vector<PyObject*>* params;                        // interned names of the parameters
  std::vector<char>* dynamic;                            // list parameter whose numbers are not part of the signature
  std::unordered_map<std::string, std::shared_ptr<Recipe>>* table;
  int credit;                                            // recipes that may still be made on first sight: one less each, one more with its use
  std::vector<uint32_t>* met;
  std::string* last_key;
  std::shared_ptr<Recipe>* last;
};

// What changes with every change of a dict; an object whose changes cannot be told never has the version it had.
uint64_t version_of(PyObject* dict) {
  static uint64_t never = 0;
  if (!dict || dict == Py_None) return 0;
  return PyDict_CheckExact(dict) ? ((PyDictObject*)dict)->ma_version_tag : --never;
}

bool current(const Operator* op, const Recipe& r) {
  return r.generation == g_generation && r.tuned_version == version_of(op->tuned) && r.config_version == version_of(op->config);
}

// Whether this signature has been met before (now it has); two may be taken for one another, which only costs time.
bool met_before(Operator* op, const char* bytes, size_t size) {
  const uint64_t h = std::hash<std::string_view>{}(std::string_view(bytes, size));
  if (op->met->empty()) op->met->resize(kMet);
  uint32_t& place = (*op->met)[h % kMet];
  const uint32_t mark = (uint32_t)(h >> 32) | 1;
  if (place == mark) return true;
  place = mark;
  return false;
}

void renew(Operator* op) {                               // nothing is known about the operator's calls
  op->table->clear();
  op->last->reset();
  op->met->clear();
  op->credit = kCredit;
}

struct Slots {
  PyObject* obj[kMaxSlots];
  int n = 0;
  int device = -1;
  struct Range { uintptr_t from, to; int slot; } memory[kMaxSlots];      // of the tensors that have elements
  int tensors = 0;
};

struct Key {
  int64_t word[160];
  int n = 0;
  bool put(int64_t v) {
    if (n == 160) return false;
    word[n++] = v;
    return true;
  }
};

bool is_tensor(PyObject* o) { return (PyObject*)Py_TYPE(o) == THPVariableClass || (PyObject*)Py_TYPE(o) == g_parameter; }

bool describe_tensor(PyObject* o, Key& key, Slots& s) {
  const at::Tensor& t = THPVariable_Unpack(o);
  // wrappers of torch.func are plain tensors to Python and have no storage (vmap, grad, jvp) or no memory (functionalize)
  if (t.layout() != at::kStrided || !t.is_cuda() || !t.has_storage() || !t.is_contiguous()) return false;
  const uintptr_t address = (uintptr_t)t.mutable_data_ptr();     // the call may write: a lazy copy gets its memory here
  if (address == 0 && t.numel() != 0) return false;
  const int device = t.device().index();
  if (s.device < 0) s.device = device;
  const auto sizes = t.sizes();
  int first = 0;                                         // one tensor in two places: which place it had first
  while (s.obj[first] != o) ++first;
  if (!key.put(1 | (int64_t)t.scalar_type() << 8 | (int64_t)device << 16 | (int64_t)sizes.size() << 24 |
               (int64_t)(address & 15) << 32 | (int64_t)first << 40))
    return false;
  for (int64_t v : sizes)
    if (!key.put(v)) return false;
  if (t.numel() != 0) s.memory[s.tensors++] = {address, address + (uintptr_t)t.nbytes(), s.n - 1};
  return true;
}

// Which tensors share memory: a kernel may be the right one only where its result is not over an operand.  One word per
// tensor that overlaps earlier ones (behind everything else, so that the rest of the key says whether there can be any).
bool describe_overlaps(Key& key, const Slots& s) {
  for (int i = 1; i < s.tensors; ++i) {
    int64_t with = 0;
    for (int j = 0; j < i; ++j)
      if (s.memory[i].from < s.memory[j].to && s.memory[j].from < s.memory[i].to) with |= (int64_t)1 << s.memory[j].slot;
    if (with && !key.put((int64_t)s.memory[i].slot << 32 | with)) return false;
  }
  return true;
}

// One argument's part of the signature; false: not something a recipe can be kept for.
bool describe(PyObject* o, bool dynamic, bool nested, Key& key, Slots& s) {
  if (s.n == kMaxSlots) return false;
  s.obj[s.n++] = o;
  if (o == nullptr) return key.put(0);                   // not given: another call than with None, maybe one argument short
  if (o == Py_None) return key.put(8);
  if (is_tensor(o)) return describe_tensor(o, key, s);
  if (PyBool_Check(o)) return key.put(dynamic ? 2 : 2 | (int64_t)(o == Py_True) << 8);
  if (PyLong_CheckExact(o)) {
    if (dynamic) return key.put(3);
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow && key.put(4) && key.put(v);
  }
  if (PyFloat_CheckExact(o)) {
    if (dynamic) return key.put(5);
    const double v = PyFloat_AS_DOUBLE(o);
    return key.put(6) && key.put(*reinterpret_cast<const int64_t*>(&v));
  }
  if (!nested && (PyList_CheckExact(o) || PyTuple_CheckExact(o))) {
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    if (!key.put(7 | (int64_t)n << 8)) return false;
    for (Py_ssize_t i = 0; i < n; ++i)
      if (!describe(PySequence_Fast_GET_ITEM(o, i), dynamic, true, key, s)) return false;
    return true;
  }
  return false;
}

// Signature of a call: every parameter in order, list arguments flattened behind their own slot.
bool signature(Operator* op, PyObject* args, PyObject* kwargs, Key& key, Slots& s) {
  const Py_ssize_t given = PyTuple_GET_SIZE(args);
  const Py_ssize_t count = (Py_ssize_t)op->params->size();
  if (given > count || count > kMaxSlots) return false;
  PyObject* value[kMaxSlots];
  for (Py_ssize_t i = 0; i < count; ++i) value[i] = i < given ? PyTuple_GET_ITEM(args, i) : nullptr;
  if (kwargs && PyDict_GET_SIZE(kwargs)) {
    PyObject *name, *v;
    Py_ssize_t pos = 0;
    while (PyDict_Next(kwargs, &pos, &name, &v)) {
      Py_ssize_t i = 0;
      while (i < count && (*op->params)[i] != name) ++i;          // interned on both sides as a rule
      if (i == count) {
        for (i = 0; i < count; ++i)
          if (PyUnicode_Compare((*op->params)[i], name) == 0) break;
      }
      if (i == count || i < given) return false;                  // unknown or given twice: the Python method says so
      value[i] = v;
    }
  }
  // the parameters take the first slots, elements of lists the ones behind them
  PyObject* lists[kMaxSlots];
  char list_dynamic[kMaxSlots];
  int nlists = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* o = value[i];
    if (o && (PyList_CheckExact(o) || PyTuple_CheckExact(o))) {
      s.obj[s.n++] = o;
      if (!key.put(7 | (int64_t)PySequence_Fast_GET_SIZE(o) << 8)) return false;
      lists[nlists] = o;
      list_dynamic[nlists++] = (*op->dynamic)[i];
    } else if (!describe(o, false, false, key, s)) {
      return false;
    }
  }
  for (int l = 0; l < nlists; ++l)
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(lists[l]); ++i)
      if (!describe(PySequence_Fast_GET_ITEM(lists[l], i), list_dynamic[l], true, key, s)) return false;
  return describe_overlaps(key, s);
}

// A library entry point with any mix of up to kMaxInts integer / pointer and kMaxFloats float arguments: the x86-64
// calling convention numbers the two classes independently, so one prototype with all integers first reaches them all,
// and a callee does not look at arguments it does not have.
int call_library(void* fn, const uint64_t* a, const float* f) {
  typedef int (*F)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                   uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, float, float, float, float);
  return ((F)fn)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15], a[16], a[17],
                 a[18], a[19], f[0], f[1], f[2], f[3]);
}

// A number of the call as an entry point takes it: what the Python method's int() or float() of it and ctypes' c_int or
// c_float make of that, errors included - whatever kind of number the call that left the recipe had there.
bool pass_number(PyObject* o, bool as_float, uint64_t& i, float& f) {
  if (as_float) {
    f = (float)PyFloat_AsDouble(o);
  } else if (PyLong_Check(o)) {
    i = (uint64_t)PyLong_AsUnsignedLongLongMask(o);
  } else if (PyObject* whole = PyNumber_Long(o)) {
    i = (uint64_t)PyLong_AsUnsignedLongLongMask(whole);
    Py_DECREF(whole);
  }
  return !PyErr_Occurred();
}

// The arguments of a call stay alive until it is over: while other threads run, one of them may empty a list argument.
struct Held {
  const Slots& s;
  explicit Held(const Slots& slots) : s(slots) {
    for (int i = 0; i < s.n; ++i) Py_XINCREF(s.obj[i]);
  }
  ~Held() {
    for (int i = 0; i < s.n; ++i) Py_XDECREF(s.obj[i]);
  }
};

struct Unlocked {                                        // other threads run meanwhile, whichever way this scope is left
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

int launch_all(const Recipe& r, const uint64_t* pointer, const uint64_t* slot_int, const float* slot_float, uint64_t stream) {
  Unlocked unlocked;
  for (const Launch& l : r.launches) {
    int rc;
    uint64_t a[64];
    float f[kMaxFloats] = {0.f, 0.f, 0.f, 0.f};
    int na = 0, nf = 0;
    for (const Arg& g : l.args) {
      switch (g.kind) {
        case Arg::kPointer: a[na++] = pointer[g.index]; break;
        case Arg::kInt: a[na++] = g.i; break;
        case Arg::kFloat: f[nf++] = g.f; break;
        case Arg::kStream: a[na++] = stream; break;
        case Arg::kSlotInt: a[na++] = slot_int[g.index]; break;
        case Arg::kSlotFloat: f[nf++] = slot_float[g.index]; break;
      }
    }
    if (l.kernel) {
      rc = g_launch(l.fn, l.grid[0], l.grid[1], l.grid[2], l.block[0], l.block[1], l.block[2], 0, (void*)(uintptr_t)stream, a, na);
    } else {
      while (na < kMaxInts) a[na++] = 0;
      rc = call_library(l.fn, a, f);
    }
    if (rc) return rc;
  }
  return 0;
}

// `no_room`: nothing was launched, there was no memory for what the recipe allocates (nullptr, no error set).
PyObject* execute(const std::shared_ptr<Recipe>& keep, const Slots& s, bool& no_room) {
  const Recipe& r = *keep;
  const Held held(s);
  at::Tensor fresh[kMaxSlots];
  uint64_t pointer[2 * kMaxSlots];
  uint64_t slot_int[kMaxSlots];
  float slot_float[kMaxSlots];
  for (int i = 0; i < s.n; ++i) {
    pointer[i] = 0;
    PyObject* o = s.obj[i];
    if (o && is_tensor(o)) pointer[i] = (uint64_t)(uintptr_t)THPVariable_Unpack(o).mutable_data_ptr();
  }
  for (const auto& n : r.numbers)
    if (!pass_number(s.obj[n.first], n.second, slot_int[n.first], slot_float[n.first])) return nullptr;
  try {
    for (size_t i = 0; i < r.allocs.size(); ++i) {
      fresh[i] = at::Tensor(at::detail::empty_cuda(r.allocs[i].sizes, r.allocs[i].dtype, at::Device(at::kCUDA, (c10::DeviceIndex)r.device), std::nullopt));
      pointer[s.n + i] = (uint64_t)(uintptr_t)fresh[i].const_data_ptr();
    }
  } catch (const c10::OutOfMemoryError&) {
    no_room = true;
    return nullptr;
  }
  const uint64_t stream = !r.uses_stream ? 0 : (uint64_t)(uintptr_t)c10::hip::getCurrentHIPStream(r.device_stream ? (c10::DeviceIndex)r.device : (c10::DeviceIndex)-1).stream();
  const int rc = launch_all(r, pointer, slot_int, slot_float, stream);
  if (rc) {
    PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, g_last_error());
    return nullptr;
  }
  auto result = [&](int i) -> PyObject* {
    if (i < 0) Py_RETURN_NONE;
    if (i >= s.n) return THPVariable_Wrap(fresh[i - s.n]);
    Py_INCREF(s.obj[i]);
    return s.obj[i];
  };
  if (r.results.size() == 1) return result(r.results[0]);
  PyObject* out = PyTuple_New((Py_ssize_t)r.results.size());
  if (!out) return nullptr;
  for (size_t i = 0; i < r.results.size(); ++i) {
    PyObject* v = result(r.results[i]);
    if (!v) { Py_DECREF(out); return nullptr; }
    PyTuple_SET_ITEM(out, (Py_ssize_t)i, v);
  }
  return out;
}

// Where torch.empty is more than memory - a dispatch mode sees it, deterministic algorithms have it filled - results are made
// by it, in the Python method.
bool plain_allocations() {
  const at::Context& context = at::globalContext();
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !(context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory());
}

void use(Operator* op, Recipe& r) {
  if (!r.used && op->credit < kCredit) ++op->credit;
  r.used = true;
}

// C++ exceptions of torch (no storage, out of memory, no device) leave as the Python exceptions that torch makes of them.
PyObject* operator_call(PyObject* self, PyObject* args, PyObject* kwargs) {
  HANDLE_TH_ERRORS
  Operator* op = (Operator*)self;
  Key key;
  Slots s;
  bool known = plain_allocations() && signature(op, args, kwargs, key, s), no_room = false;
  if (known) {
    const char* bytes = (const char*)key.word;
    const size_t size = (size_t)key.n * sizeof(int64_t);
    if (*op->last && op->last_key->size() == size && memcmp(op->last_key->data(), bytes, size) == 0 && current(op, **op->last)) {
      std::shared_ptr<Recipe> r = *op->last;
      use(op, *r);
      PyObject* result = execute(r, s, no_room);
      if (!no_room) return result;
    }
    auto it = op->table->find(std::string(bytes, size));
    if (!no_room && it != op->table->end() && current(op, *it->second)) {
      std::shared_ptr<Recipe> r = it->second;
      *op->last_key = it->first;
      *op->last = r;
      use(op, *r);
      PyObject* result = execute(r, s, no_room);
      if (!no_room) return result;
    }
    if (no_room) {
      known = false;                                     // this call is run another way, or raises; the recipe stays for the next one
    } else if (it == op->table->end() && !met_before(op, bytes, size)) {
      known = op->credit > 0;
      if (known) --op->credit;
    }
  }
  // no recipe: the Python method runs the call and, where it can and is asked to (`known`), leaves one (commit)
  static PyObject* name = PyUnicode_InternFromString("_call");
  PyObject* pending;
  if (known) {
    PyObject* slots = PyTuple_New(s.n);
    if (!slots) return nullptr;
    for (int i = 0; i < s.n; ++i) {
      PyObject* o = s.obj[i] ? s.obj[i] : Py_None;
      Py_INCREF(o);
      PyTuple_SET_ITEM(slots, i, o);
    }
    pending = Py_BuildValue("(y#Ni)", (const char*)key.word, (Py_ssize_t)(key.n * sizeof(int64_t)), slots, s.device);
    if (!pending) return nullptr;
  } else {
    pending = Py_None;
    Py_INCREF(pending);
  }
  PyObject* method = PyObject_GetAttr(self, name);
  if (!method) { Py_DECREF(pending); return nullptr; }
  const Py_ssize_t n = PyTuple_GET_SIZE(args);
  PyObject* full = PyTuple_New(n + 1);
  if (!full) { Py_DECREF(method); Py_DECREF(pending); return nullptr; }
  PyTuple_SET_ITEM(full, 0, pending);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyTuple_GET_ITEM(args, i);
    Py_INCREF(o);
    PyTuple_SET_ITEM(full, i + 1, o);
  }
  PyObject* out = PyObject_Call(method, full, kwargs);
  Py_DECREF(full);
  Py_DECREF(method);
  return out;
  END_HANDLE_TH_ERRORS
}

// commit(key, slots, device, device_stream, allocs, launches, results)
//   allocs:   [(dtype code of torch, (sizes...))]
//   launches: [(address, grid or None, block, args)], an argument being ('p', index) | ('i', int) | ('f', float) | ('s',) | ('I', slot) | ('F', slot)
PyObject* operator_commit(PyObject* self, PyObject* args) {
  Operator* op = (Operator*)self;
  const char* key;
  Py_ssize_t key_size;
  int slots, device, device_stream;
  PyObject *allocs, *launches, *results;
  if (!PyArg_ParseTuple(args, "y#iiiOOO", &key, &key_size, &slots, &device, &device_stream, &allocs, &launches, &results)) return nullptr;
  auto r = std::make_shared<Recipe>();
  r->generation = g_generation;
  r->tuned_version = version_of(op->tuned);
  r->config_version = version_of(op->config);
  r->device = device;
  r->device_stream = device_stream != 0;
  r->uses_stream = r->used = false;
  r->slots = slots;
  if (!PyList_Check(allocs) || !PyList_Check(launches) || !PyList_Check(results) || PyList_GET_SIZE(allocs) > kMaxSlots) {
    PyErr_SetString(PyExc_TypeError, "commit: allocs (at most 24), launches and results are lists");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(allocs); ++i) {
    PyObject *dtype, *sizes;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(allocs, i), "OO!", &dtype, &PyTuple_Type, &sizes)) return nullptr;
    if (!THPDtype_Check(dtype)) { PyErr_SetString(PyExc_TypeError, "commit: an allocation needs a dtype"); return nullptr; }
    Alloc a;
    a.dtype = ((THPDtype*)dtype)->scalar_type;
    for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(sizes); ++d) a.sizes.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(sizes, d)));
    if (PyErr_Occurred()) return nullptr;
    r->allocs.push_back(std::move(a));
  }
  const int tensors = slots + (int)r->allocs.size();
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(launches); ++i) {
    unsigned long long fn;
    PyObject *grid, *block, *list;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(launches, i), "KOOO!", &fn, &grid, &block, &PyList_Type, &list)) return nullptr;
    Launch l;
    l.fn = (void*)(uintptr_t)fn;
    l.kernel = grid != Py_None;
    r->uses_stream |= l.kernel;
    if (l.kernel && (!PyArg_ParseTuple(grid, "III", &l.grid[0], &l.grid[1], &l.grid[2]) || !PyArg_ParseTuple(block, "III", &l.block[0], &l.block[1], &l.block[2])))
      return nullptr;
    int ints = 0, floats = 0;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(list); ++k) {
      int kind;
      PyObject* v = nullptr;
      if (!PyArg_ParseTuple(PyList_GET_ITEM(list, k), "C|O", &kind, &v)) return nullptr;
      Arg g{};
      if (kind == 's') { g.kind = Arg::kStream; r->uses_stream = true; }
      else if (kind == 'i') { g.kind = Arg::kInt; g.i = (uint64_t)PyLong_AsUnsignedLongLongMask(v); }
      else if (kind == 'f') { g.kind = Arg::kFloat; g.f = (float)PyFloat_AsDouble(v); }
      else {
        g.kind = kind == 'p' ? Arg::kPointer : kind == 'I' ? Arg::kSlotInt : Arg::kSlotFloat;
        g.index = (int)PyLong_AsLong(v);
        if (!PyErr_Occurred() && (g.index < 0 || g.index >= (kind == 'p' ? tensors : slots)))
          PyErr_SetString(PyExc_IndexError, "commit: an argument refers to a slot that does not exist");
        else if (kind != 'p') r->numbers.emplace_back(g.index, g.kind == Arg::kSlotFloat);
      }
      if (PyErr_Occurred()) return nullptr;
      (g.kind == Arg::kFloat || g.kind == Arg::kSlotFloat ? floats : ints)++;
      l.args.push_back(g);
    }
    if (ints > (l.kernel ? 64 : kMaxInts) || floats > (l.kernel ? 0 : kMaxFloats)) {
      PyErr_SetString(PyExc_ValueError, "commit: too many arguments");
      return nullptr;
    }
    r->launches.push_back(std::move(l));
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(results); ++i) {
    const int v = (int)PyLong_AsLong(PyList_GET_ITEM(results, i));
    if (PyErr_Occurred()) return nullptr;
    if (v >= tensors) { PyErr_SetString(PyExc_IndexError, "commit: a result that does not exist"); return nullptr; }
    r->results.push_back(v);
  }
  if (op->table->size() >= kMaxRecipes) renew(op);
  std::string k(key, (size_t)key_size);
  (*op->table)[k] = r;
  *op->last_key = std::move(k);
  *op->last = std::move(r);
  Py_RETURN_NONE;
}

// bind(names, dynamic): the parameters of _call in order, and for which of them the numbers in a list argument are not
// part of the signature (they are passed on as they are)
PyObject* operator_bind(PyObject* self, PyObject* args) {
  Operator* op = (Operator*)self;
  PyObject *names, *dynamic;
  if (!PyArg_ParseTuple(args, "O!O!", &PyTuple_Type, &names, &PyTuple_Type, &dynamic)) return nullptr;
  for (PyObject* p : *op->params) Py_DECREF(p);
  op->params->clear();
  op->dynamic->clear();
  renew(op);
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); ++i) {
    PyObject* n = PyTuple_GET_ITEM(names, i);
    if (!PyUnicode_Check(n)) { PyErr_SetString(PyExc_TypeError, "bind: names are strings"); return nullptr; }
    Py_INCREF(n);
    PyUnicode_InternInPlace(&n);
    op->params->push_back(n);
    const int is = PySequence_Contains(dynamic, n);
    if (is < 0) return nullptr;
    op->dynamic->push_back((char)is);
  }
  Py_RETURN_NONE;
}

PyObject* operator_new(PyTypeObject* type, PyObject*, PyObject*) {
  Operator* op = (Operator*)type->tp_alloc(type, 0);
  if (!op) return nullptr;
  op->params = new std::vector<PyObject*>();
  op->dynamic = new std::vector<char>();
  op->table = new std::unordered_map<std::string, std::shared_ptr<Recipe>>();
  op->met = new std::vector<uint32_t>();
  op->credit = kCredit;
  op->last_key = new std::string();
  op->last = new std::shared_ptr<Recipe>();
  return (PyObject*)op;
}

int operator_traverse(PyObject* self, visitproc visit, void* arg) {
  Operator* op = (Operator*)self;
  Py_VISIT(op->tuned);
  Py_VISIT(op->config);
  Py_VISIT(op->fast_path);
  return 0;
}

int operator_clear(PyObject* self) {
  Operator* op = (Operator*)self;
  Py_CLEAR(op->tuned);
  Py_CLEAR(op->config);
  Py_CLEAR(op->fast_path);
  return 0;
}

void operator_dealloc(PyObject* self) {
  Operator* op = (Operator*)self;
  PyObject_GC_UnTrack(self);
  operator_clear(self);
  for (PyObject* p : *op->params) Py_DECREF(p);
  delete op->params;
  delete op->dynamic;
  delete op->table;
  delete op->met;
  delete op->last_key;
  delete op->last;
  Py_TYPE(self)->tp_free(self);
}

PyObject* attribute_get(PyObject* self, void* offset) {
  PyObject* v = *(PyObject**)((char*)self + (size_t)offset);
  if (!v) v = Py_None;
  Py_INCREF(v);
  return v;
}

int attribute_set(PyObject* self, PyObject* value, void* offset) {
  Operator* op = (Operator*)self;
  renew(op);
  Py_XINCREF(value);
  PyObject** field = (PyObject**)((char*)self + (size_t)offset);
  PyObject* old = *field;
  *field = value;
  Py_XDECREF(old);
  return 0;
}

PyGetSetDef operator_attributes[] = {
    {"tuned", attribute_get, attribute_set, "choices of tuning runs", (void*)offsetof(Operator, tuned)},
    {"config", attribute_get, attribute_set, "parsed config", (void*)offsetof(Operator, config)},
    {"fast_path", attribute_get, attribute_set, "handler of a hand-written kernel, or None", (void*)offsetof(Operator, fast_path)},
    {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyMethodDef operator_methods[] = {
    {"_commit", operator_commit, METH_VARARGS, "keep how a call of this signature is run"},
    {"_bind", operator_bind, METH_VARARGS, "name the parameters"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject OperatorType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* module_setup(PyObject*, PyObject* args) {
  unsigned long long launch, last_error;
  PyObject *error, *parameter;
  if (!PyArg_ParseTuple(args, "KKOO", &launch, &last_error, &error, &parameter)) return nullptr;
  g_launch = (decltype(g_launch))(uintptr_t)launch;
  g_last_error = (decltype(g_last_error))(uintptr_t)last_error;
  Py_INCREF(error);
  Py_XSETREF(g_error, error);
  Py_INCREF(parameter);
  Py_XSETREF(g_parameter, parameter);
  Py_RETURN_NONE;
}

PyObject* module_forget(PyObject*, PyObject*) {
  ++g_generation;
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {{"setup", module_setup, METH_VARARGS, "addresses of art_launch and art_last_error, the error class, torch.nn.Parameter"},
                                {"forget", module_forget, METH_NOARGS, "every recipe is worked out again at its next call"},
                                {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_calls", "operator calls in native code", -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  OperatorType.tp_name = "antares_amd.runtime._calls.Operator";
  OperatorType.tp_basicsize = sizeof(Operator);
  OperatorType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  OperatorType.tp_doc = "an operator whose calls are replayed from recipes";
  OperatorType.tp_new = operator_new;
  OperatorType.tp_dealloc = operator_dealloc;
  OperatorType.tp_traverse = operator_traverse;
  OperatorType.tp_clear = operator_clear;
  OperatorType.tp_call = operator_call;
  OperatorType.tp_getset = operator_attributes;
  OperatorType.tp_methods = operator_methods;
  if (PyType_Ready(&OperatorType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&OperatorType);
  PyModule_AddObject(m, "Operator", (PyObject*)&OperatorType);
  return m;
}
