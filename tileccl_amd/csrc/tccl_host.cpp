// CPython extension `tileccl_amd._host`: the host side of a repeated call.
//
// A fused operation or a collective on small tensors takes as long as the host needs to issue it.  The checks of a
// call, the descriptors it builds and its launch options depend on the tensors' layouts only, so they are made once
// (in Python) and kept as a `Call`; what is left for every call is to see that the tensors still have those layouts,
// to write their addresses and the launch number into copies of the descriptors and to call the C entry point.  In
// Python that took 3 to 5 us (a key of shapes, strides and types per tensor alone takes 1 us), beside the 2.5 us of
// the launch itself; here it takes 0.3 us.
//
// `Table` holds the calls of one owner (a context, a heap, an operation), found by a hash of the key and the layouts, bounded, the
// one that has not been used for longest dropped first.  Everything runs under the interpreter lock except the C entry
// point; a Call does not change once it is built, and each launch works on copies of its descriptors, so threads may
// share both.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <list>
#include <unordered_map>
#include <vector>

#include "../../include/tileccl_hip.h"

namespace {

constexpr int kMaxArgs = 12;     // arguments of an entry point, the stream included
constexpr int kMaxTensors = 9;   // an operation's operands and output; one tensor per rank
constexpr unsigned long kCalls = 64;  // a table's bound unless it is given one

PyObject *kGemm, *kSync;                                       // stand for the descriptor copies in an argument list
PyObject *sEpoch, *sLockEpoch, *sClear, *sMaxTasks, *sSpin, *sNext, *sRevision;  // attributes of the signal words
PyObject *current_stream, *is_capturing, *report, *device0;

size_t mixed(size_t h, size_t v) { return (h ^ v) * 0x9e3779b97f4a7c15ull + (h >> 29); }

// Everything about a tensor that a descriptor depends on, except where it lies.
struct Layout {
  c10::ScalarType type;
  c10::Device device{c10::kCPU};
  int misaligned;  // address modulo 16
  std::vector<int64_t> sizes, strides;

  explicit Layout(const at::Tensor& t)
      : type(t.scalar_type()), device(t.device()), misaligned((int)((uintptr_t)t.data_ptr() & 15)),
        sizes(t.sizes().begin(), t.sizes().end()), strides(t.strides().begin(), t.strides().end()) {}
  static size_t hash(size_t h, const at::Tensor& t, uintptr_t at) {
    h = mixed(h, (size_t)t.scalar_type() * 16 + (at & 15));
    for (const int64_t n : t.sizes()) h = mixed(h, (size_t)n);
    for (const int64_t n : t.strides()) h = mixed(h, (size_t)n);
    return h;
  }
  bool matches(const at::Tensor& t, uintptr_t at) const {
    return type == t.scalar_type() && misaligned == (int)(at & 15) && device == t.device() && t.sizes().equals(sizes) &&
           t.strides().equals(strides);
  }
};

// One argument of an entry point: a value, a descriptor copy, or a tensor's address plus an offset.
struct Arg {
  enum Kind { kValue, kGemmCopy, kSyncCopy, kTensor } kind;
  int64_t value;
  int tensor;
};

struct Call {
  PyObject_HEAD
  // (constructed in place: Python allocates the object zeroed)
  std::vector<Layout>* layouts;
  std::vector<Arg>* args;
  int64_t (*entry)(int64_t, ...);
  tccl_gemm_desc gemm;
  tccl_sync_desc_arrivals sync;
  bool has_gemm, has_sync;
  int c_tensor;          // tensor whose address plus c_offset is the GEMM's C (< 0: C is fixed)
  int64_t c_offset;
  int64_t a_bytes, c_bytes;  // of an A that the GEMM reads by columns (0: it does not) and of its C: they must lie apart
  int64_t heap_lo, heap_size;  // the tensors in `on_heap` (a bit mask) must start in this range
  int64_t ranks_lo, ranks_size;  // all ranks' heaps: an A by columns lies in none but this rank's, where launches store to the peers'
  uint32_t on_heap;
  std::vector<int64_t>* bases;  // per tensor: all must lie at one offset from these
  int counted;           // 0: the launch is not numbered, 1: by `epoch`, 2: by `lock_epoch`
  long long revision;    // of the signal words when their descriptor was copied (< 0: they have none)
  size_t hash;           // of the key and the layouts
  PyObject *key, *tag, *what, *words, *prepare, *keep, *variant;
};

int call_traverse(Call* self, visitproc visit, void* arg) {
  Py_VISIT(self->key);
  Py_VISIT(self->tag);
  Py_VISIT(self->what);
  Py_VISIT(self->words);
  Py_VISIT(self->prepare);
  Py_VISIT(self->keep);
  Py_VISIT(self->variant);
  return 0;
}
int call_clear(Call* self) {
  Py_CLEAR(self->key);
  Py_CLEAR(self->tag);
  Py_CLEAR(self->what);
  Py_CLEAR(self->words);
  Py_CLEAR(self->prepare);
  Py_CLEAR(self->keep);
  Py_CLEAR(self->variant);
  return 0;
}
void call_dealloc(Call* self) {
  PyObject_GC_UnTrack(self);
  call_clear(self);
  delete self->layouts;
  delete self->args;
  delete self->bases;
  Py_TYPE(self)->tp_free((PyObject*)self);
}

// Tensors without memory of their own (sparse, nested, inside torch.vmap or torch.func.grad) throw when asked for an
// address or strides, and the interpreter's frames above an entry of this module are no place for a C++ exception: every
// entry that looks at tensors or allocates goes through here.
template <typename Result, typename Body>
Result guarded(Result failed, Body body) {
  try {
    return body();
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
  }
  return failed;
}

struct Reference {  // given up at the end of its scope
  PyObject* object = nullptr;
  ~Reference() { Py_XDECREF(object); }
};

PyObject* own(PyObject* o) {
  if (o == Py_None) return nullptr;
  Py_XINCREF(o);
  return o;
}

bool int_attr(PyObject* o, PyObject* name, long long& out) {
  PyObject** dict = _PyObject_GetDictPtr(o);  // signal words keep theirs there
  PyObject* kept = dict && *dict ? PyDict_GetItemWithError(*dict, name) : nullptr;
  if (kept) {
    out = PyLong_AsLongLong(kept);
    return !(out == -1 && PyErr_Occurred());
  }
  if (PyErr_Occurred()) return false;
  PyObject* v = PyObject_GetAttr(o, name);
  if (!v) return false;
  out = PyLong_AsLongLong(v);
  Py_DECREF(v);
  return !(out == -1 && PyErr_Occurred());
}

// Plain values of a key count by value, anything else (a context, signal words, a contract) by identity.
bool plain(PyObject* o) { return PyLong_CheckExact(o) || PyUnicode_CheckExact(o) || PyFloat_CheckExact(o) || PyBool_Check(o); }
bool same(PyObject* a, PyObject* b) {
  if (a == b) return true;
  if (Py_TYPE(a) != Py_TYPE(b) || !plain(a)) return false;
  const int r = PyObject_RichCompareBool(a, b, Py_EQ);
  if (r < 0) PyErr_Clear();
  return r == 1;
}
bool same_key(PyObject* a, PyObject* b) {
  if (a == b) return true;
  const Py_ssize_t n = PyTuple_GET_SIZE(a);
  if (n != PyTuple_GET_SIZE(b)) return false;
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!same(PyTuple_GET_ITEM(a, i), PyTuple_GET_ITEM(b, i))) return false;
  return true;
}
size_t key_hash(PyObject* key) {
  size_t h = (size_t)PyTuple_GET_SIZE(key);
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(key); ++i) {
    PyObject* o = PyTuple_GET_ITEM(key, i);
    Py_hash_t v = (Py_hash_t)((uintptr_t)o >> 4);
    if (plain(o) && (v = PyObject_Hash(o)) == -1) PyErr_Clear();
    h = mixed(h, (size_t)v);
  }
  return h;
}

// Call(entry, what, args, tensors, key, *, tag, gemm, c, sync, words, variant, on_heap, heap, bases, prepare, keep)
int call_init_checked(Call* self, PyObject* pos, PyObject* kw) {
  static const char* names[] = {"entry", "what", "args", "tensors", "key", "tag", "gemm", "c", "sync", "words", "variant",
                                "on_heap", "heap", "bases", "prepare", "keep", nullptr};
  unsigned long long entry = 0, gemm = 0, sync = 0;
  PyObject *what, *args, *tensors, *key, *tag = Py_None, *c = Py_None, *words = Py_None, *variant = Py_None, *on_heap = Py_None,
           *heap = Py_None, *bases = Py_None, *prepare = Py_None, *keep = Py_None;
  if (!PyArg_ParseTupleAndKeywords(pos, kw, "KOO!O!O!|$OKOKOOOOOOO", (char**)names, &entry, &what, &PyTuple_Type, &args, &PyTuple_Type,
                                   &tensors, &PyTuple_Type, &key, &tag, &gemm, &c, &sync, &words, &variant, &on_heap, &heap, &bases, &prepare,
                                   &keep))
    return -1;
  if (self->layouts) {
    PyErr_SetString(PyExc_RuntimeError, "a Call is built once");
    return -1;
  }
  self->entry = (int64_t(*)(int64_t, ...))(uintptr_t)entry;
  self->layouts = new std::vector<Layout>();
  self->args = new std::vector<Arg>();
  self->bases = new std::vector<int64_t>();
  const Py_ssize_t n = PyTuple_GET_SIZE(tensors);
  if (n < 1 || n > kMaxTensors || PyTuple_GET_SIZE(args) >= kMaxArgs || entry == 0) {
    PyErr_SetString(PyExc_ValueError, "a Call takes an entry point, 1 to 9 tensors and at most 11 arguments");
    return -1;
  }
  self->hash = key_hash(key);
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!THPVariable_Check(PyTuple_GET_ITEM(tensors, i))) {
      PyErr_SetString(PyExc_TypeError, "a Call is built for tensors");
      return -1;
    }
    const at::Tensor& t = THPVariable_Unpack(PyTuple_GET_ITEM(tensors, i));
    self->layouts->emplace_back(t);
    self->hash = Layout::hash(self->hash, t, (uintptr_t)t.data_ptr());
  }
  if (gemm) {
    self->has_gemm = true;
    memcpy(&self->gemm, (const void*)(uintptr_t)gemm, sizeof(self->gemm));
  }
  if (sync) {
    self->has_sync = true;
    memcpy(&self->sync, (const void*)(uintptr_t)sync, sizeof(self->sync));
  }
  auto tensor_index = [n](long long i) { return i >= 0 && i < n; };
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args); ++i) {
    PyObject* a = PyTuple_GET_ITEM(args, i);
    Arg arg{Arg::kValue, 0, 0};
    if (a == kGemm && gemm) {
      arg.kind = Arg::kGemmCopy;
    } else if (a == kSync && sync) {
      arg.kind = Arg::kSyncCopy;
    } else if (PyTuple_Check(a)) {
      long long offset = 0;
      arg.kind = Arg::kTensor;
      if (!PyArg_ParseTuple(a, "iL", &arg.tensor, &offset)) return -1;
      arg.value = offset;
      if (!tensor_index(arg.tensor)) {
        PyErr_SetString(PyExc_ValueError, "an argument names a tensor that the Call does not have");
        return -1;
      }
    } else if (a != Py_None) {
      arg.value = (int64_t)PyLong_AsUnsignedLongLongMask(a);
      if (PyErr_Occurred()) return -1;
    }
    self->args->push_back(arg);
  }
  self->c_tensor = -1;
  if (c != Py_None) {
    long long offset = 0;
    if (!PyArg_ParseTuple(c, "iL", &self->c_tensor, &offset)) return -1;
    self->c_offset = offset;
  }
  if ((gemm && n < 2) || (c != Py_None && !tensor_index(self->c_tensor))) {
    PyErr_SetString(PyExc_ValueError, "a GEMM's operands are the first two tensors of the Call");
    return -1;
  }
  if (gemm && (self->gemm.flags & TCCL_GEMM_A_COLUMNS)) {
    const tccl_gemm_desc& d = self->gemm;
    self->a_bytes = ((int64_t)(d.K - 1 - ((d.flags >> TCCL_GEMM_A_SHORT_SHIFT) & 15)) * d.lda + d.M) * 2;
    self->c_bytes = ((int64_t)(d.M - 1) * d.ldc + d.N) * (d.out_dtype == TCCL_F32 ? 4 : 2);
  }
  if (heap != Py_None) {
    long long lo = 0, size = 0, all_lo = 0, all_size = 0;
    if (!PyArg_ParseTuple(heap, "LL|LL", &lo, &size, &all_lo, &all_size)) return -1;
    self->heap_lo = lo;
    self->heap_size = size;
    self->ranks_lo = all_lo;
    self->ranks_size = all_size;
    self->on_heap = on_heap == Py_None ? ~0u : (uint32_t)PyLong_AsUnsignedLongMask(on_heap);
    if (PyErr_Occurred()) return -1;
  }
  if (bases != Py_None) {
    PyObject* seq = PySequence_Fast(bases, "bases must be a sequence");
    if (!seq) return -1;
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); ++i) self->bases->push_back((int64_t)PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i)));
    Py_DECREF(seq);
    if (PyErr_Occurred()) return -1;
    if ((Py_ssize_t)self->bases->size() != n) {
      PyErr_SetString(PyExc_ValueError, "one base per tensor");
      return -1;
    }
  }
  if (sync && words != Py_None && variant != Py_None) {
    const char* v = PyUnicode_AsUTF8(variant);
    if (!v) return -1;
    self->counted = !strcmp(v, "s2") ? 1 : !strcmp(v, "s1") ? 2 : 0;
  }
  self->revision = -1;
  if (sync && words != Py_None && PyObject_HasAttr(words, sRevision) && !int_attr(words, sRevision, self->revision)) return -1;
  Py_INCREF(key);
  self->key = key;
  self->tag = own(tag);
  self->what = own(what);
  self->words = own(words);
  self->variant = own(variant);
  self->prepare = own(prepare);
  self->keep = own(keep);
  return 0;
}

int call_init(Call* self, PyObject* pos, PyObject* kw) {
  return guarded(-1, [&] { return call_init_checked(self, pos, kw); });
}

PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// The launch's number: what SyncWords.next_epoch() gives.  The ordinary case (nothing to clear, no wrap-around near)
// is one increment; the others are left to that method.
bool next_number(const Call* c, int32_t& number) {
  long long epoch, lock_epoch, tasks, clear;
  if (!int_attr(c->words, sClear, clear) || !int_attr(c->words, sEpoch, epoch) || !int_attr(c->words, sLockEpoch, lock_epoch) ||
      !int_attr(c->words, sMaxTasks, tasks))
    return false;
  PyObject* capturing = PyObject_CallNoArgs(is_capturing);
  if (!capturing) return false;
  const bool recorded = capturing == Py_True;
  Py_DECREF(capturing);
  const long long last = epoch > lock_epoch ? epoch : lock_epoch;
  if (clear || recorded || tasks <= 0 || last >= (1ll << 30) / tasks) {
    PyObject* n = PyObject_CallMethodObjArgs(c->words, sNext, c->variant, nullptr);
    if (!n) return false;
    number = (int32_t)PyLong_AsLong(n);
    Py_DECREF(n);
    return !PyErr_Occurred();
  }
  const bool by_lock = c->counted == 2;
  number = (int32_t)((by_lock ? lock_epoch : epoch) + 1);
  PyObject* n = PyLong_FromLong(number);
  if (!n) return false;
  const int rc = PyObject_GenericSetAttr(c->words, by_lock ? sLockEpoch : sEpoch, n);  // (no part of the words' descriptor)
  Py_DECREF(n);
  return rc == 0;
}

// A launch that the entry point refused has signalled nothing: its number goes to the next one, or the words would be
// behind the numbers (and this rank's behind its peers') from here on.
bool number_back(const Call* c, int32_t number) {
  PyObject* name = c->counted == 2 ? sLockEpoch : sEpoch;
  long long now = 0;
  if (!int_attr(c->words, name, now)) return false;
  if (now != number) return true;  // another thread has numbered a launch since
  PyObject* n = PyLong_FromLong(number - 1);
  if (!n) return false;
  const int rc = PyObject_GenericSetAttr(c->words, name, n);
  Py_DECREF(n);
  return rc == 0;
}

// Issue the call on these tensors (of the layouts it was built for, at the addresses `at`).  Returns the tag, or null with an
// exception set.
PyObject* launch(Call* c, PyObject* const* tensors, int64_t* at, PyObject* alpha) {
  tccl_gemm_desc gemm;
  tccl_sync_desc_arrivals sync;
  Reference prepared;  // operands that had to be packed live until the launch is issued
  if (c->prepare) {
    PyObject* operands[2] = {tensors[0], tensors[1]};
    PyObject* pair = prepared.object = PyObject_Vectorcall(c->prepare, operands, 2, nullptr);
    if (!pair) return nullptr;
    if (!PyTuple_Check(pair) || PyTuple_GET_SIZE(pair) != 2 || !THPVariable_Check(PyTuple_GET_ITEM(pair, 0)) ||
        !THPVariable_Check(PyTuple_GET_ITEM(pair, 1))) {
      PyErr_SetString(PyExc_TypeError, "prepare must return the two operands");
      return nullptr;
    }
    for (int i = 0; i < 2; ++i) at[i] = (int64_t)(uintptr_t)THPVariable_Unpack(PyTuple_GET_ITEM(pair, i)).data_ptr();
  }
  bool ok = true;
  if (c->has_gemm) {
    gemm = c->gemm;
    gemm.A = (const void*)at[0];
    gemm.B = (const void*)at[1];
    if (c->c_tensor >= 0) gemm.C = (void*)(at[c->c_tensor] + c->c_offset);
    if (alpha != Py_None) {
      const double value = PyFloat_AsDouble(alpha);
      ok = !(value == -1.0 && PyErr_Occurred());
      gemm.alpha = (float)value;
    }
  }
  if (ok && c->has_sync) {
    sync = c->sync;
    if (c->words) {
      long long spin = 0;
      ok = int_attr(c->words, sSpin, spin);
      sync.sync.spin_limit_ns = spin;
      if (ok && c->counted) ok = next_number(c, sync.sync.epoch);
    }
  }
  int64_t v[kMaxArgs] = {0};
  if (ok) {
    PyObject* index[1] = {device0};
    PyObject* s = PyObject_Vectorcall(current_stream, index, 1, nullptr);
    ok = s != nullptr;
    if (ok) v[c->args->size()] = (int64_t)PyLong_AsUnsignedLongLongMask(s);
    Py_XDECREF(s);
    ok = ok && !PyErr_Occurred();
  }
  if (!ok) return nullptr;
  for (size_t i = 0; i < c->args->size(); ++i) {
    const Arg& a = (*c->args)[i];
    v[i] = a.kind == Arg::kGemmCopy ? (int64_t)(uintptr_t)&gemm : a.kind == Arg::kSyncCopy ? (int64_t)(uintptr_t)&sync
           : a.kind == Arg::kTensor ? at[a.tensor] + a.value : a.value;
  }
  // Every parameter of the entry points is an integer or a pointer.  Passed as 64-bit integers they land where the
  // x86-64 calling convention puts the declared types; arguments past an entry point's own are not looked at.
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = (int32_t)((int64_t(*)(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t))c->entry)(
      v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11]);
  Py_END_ALLOW_THREADS;
  if (rc != 0) {
    if (rc < 0 && c->has_sync && c->words && c->counted && !number_back(c, sync.sync.epoch)) return nullptr;
    PyObject* r = PyObject_CallFunction(report, "iO", (int)rc, c->what ? c->what : Py_None);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "error code %d", (int)rc);
    return nullptr;
  }
  PyObject* tag = c->tag ? c->tag : Py_True;
  Py_INCREF(tag);
  return tag;
}

// The tensors' addresses; false if one has none, or no sizes and strides, which no call is for.
bool addresses(PyObject* const* tensors, Py_ssize_t n, int64_t* at) {
  try {
    for (Py_ssize_t i = 0; i < n; ++i) {
      const at::Tensor& t = THPVariable_Unpack(tensors[i]);
      if (t.layout() != c10::kStrided || t.unsafeGetTensorImpl()->is_nested()) return false;
      at[i] = (int64_t)(uintptr_t)t.data_ptr();
      t.strides();
    }
  } catch (...) {
    return false;
  }
  return true;
}

bool fits(const Call* c, PyObject* const* tensors, const int64_t* at, Py_ssize_t n) {
  if ((Py_ssize_t)c->layouts->size() != n) return false;
  int64_t offset = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor& t = THPVariable_Unpack(tensors[i]);
    if (!(*c->layouts)[i].matches(t, (uintptr_t)at[i])) return false;
    if (c->heap_size && ((c->on_heap >> i) & 1u)) {
      const int64_t into = at[i] - c->heap_lo;
      if (!(into >= 0 && into < c->heap_size) && t.numel() != 0) return false;
    }
    if (!c->bases->empty()) {
      const int64_t from_base = at[i] - (*c->bases)[i];
      if (i == 0) offset = from_base;
      if (from_base != offset) return false;
    }
  }
  if (c->a_bytes) {
    const int64_t out = c->c_tensor >= 0 ? at[c->c_tensor] + c->c_offset : (int64_t)(uintptr_t)c->gemm.C;
    if (at[0] < out + c->c_bytes && out < at[0] + c->a_bytes) return false;
    auto starts_in = [at](int64_t lo, int64_t size) { return at[0] - lo >= 0 && at[0] - lo < size; };
    if (starts_in(c->ranks_lo, c->ranks_size) && !starts_in(c->heap_lo, c->heap_size)) return false;
  }
  return true;
}

struct Table {
  PyObject_HEAD
  std::list<Call*>* order;  // used last first
  std::unordered_multimap<size_t, std::list<Call*>::iterator>* by_hash;
  size_t limit;
};

// Table(limit=64)
PyObject* table_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  static const char* names[] = {"limit", nullptr};
  unsigned long limit = kCalls;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "|k", (char**)names, &limit)) return nullptr;
  if (limit < 1) {
    PyErr_SetString(PyExc_ValueError, "a Table holds at least one Call");
    return nullptr;
  }
  return guarded((PyObject*)nullptr, [&] {
    Table* t = (Table*)type->tp_alloc(type, 0);
    if (!t) return (PyObject*)nullptr;
    Reference held{(PyObject*)t};
    t->limit = limit;
    t->order = new std::list<Call*>();
    t->by_hash = new std::unordered_multimap<size_t, std::list<Call*>::iterator>();
    held.object = nullptr;
    return (PyObject*)t;
  });
}
int table_traverse(Table* self, visitproc visit, void* arg) {
  if (self->order)
    for (Call* c : *self->order) Py_VISIT((PyObject*)c);
  return 0;
}
int table_clear(Table* self) {
  if (self->by_hash) self->by_hash->clear();
  std::list<Call*> calls;
  if (self->order) calls.swap(*self->order);
  for (Call* c : calls) Py_DECREF(c);
  return 0;
}
void table_dealloc(Table* self) {
  PyObject_GC_UnTrack(self);
  table_clear(self);
  delete self->order;
  delete self->by_hash;
  Py_TYPE(self)->tp_free((PyObject*)self);
}

void drop(Table* self, Call* call) {
  const auto range = self->by_hash->equal_range(call->hash);
  for (auto i = range.first; i != range.second; ++i) {
    if (*i->second != call) continue;
    self->order->erase(i->second);
    self->by_hash->erase(i);
    Py_DECREF(call);  // (may run other code: the table is in order by now)
    return;
  }
}

PyObject* table_add(Table* self, PyObject* object) {
  if (!PyObject_TypeCheck(object, &CallType) || !((Call*)object)->layouts || !((Call*)object)->key) {
    PyErr_SetString(PyExc_TypeError, "Table.add expects a Call");
    return nullptr;
  }
  Call* call = (Call*)object;
  const bool added = guarded(false, [&] {
    self->order->push_front(call);
    try {
      self->by_hash->emplace(call->hash, self->order->begin());
    } catch (...) {
      self->order->pop_front();
      throw;
    }
    return true;
  });
  if (!added) return nullptr;
  Py_INCREF(call);
  if (self->order->size() > self->limit) drop(self, self->order->back());
  Py_RETURN_NONE;
}

// The call for these tensors, moved to the front; null if there is none.  A program that repeats one call finds it there.
Call* find(Table* self, PyObject* key, PyObject* const* tensors, const int64_t* at, Py_ssize_t n) {
  Call* first = self->order->front();
  if (fits(first, tensors, at, n) && same_key(first->key, key)) return first;
  size_t hash = key_hash(key);
  for (Py_ssize_t i = 0; i < n; ++i) hash = Layout::hash(hash, THPVariable_Unpack(tensors[i]), (uintptr_t)at[i]);
  const auto range = self->by_hash->equal_range(hash);
  for (auto i = range.first; i != range.second; ++i) {
    Call* c = *i->second;
    if (!fits(c, tensors, at, n) || !same_key(c->key, key)) continue;
    self->order->splice(self->order->begin(), *self->order, i->second);
    return c;
  }
  return nullptr;
}

// launch(key, alpha, *tensors): the tag of the call that was issued, or None if there is none for these tensors.
PyObject* table_launch(Table* self, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs < 3 || nargs > 2 + kMaxTensors || !PyTuple_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "launch(key, alpha, *tensors): a tuple, a number or None, 1 to 9 tensors");
    return nullptr;
  }
  for (Py_ssize_t i = 2; i < nargs; ++i)
    if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
  if (self->order->empty()) Py_RETURN_NONE;
  int64_t at[kMaxTensors];
  if (!addresses(args + 2, nargs - 2, at)) Py_RETURN_NONE;
  return guarded((PyObject*)nullptr, [&]() -> PyObject* {
    Call* c = find(self, args[0], args + 2, at, nargs - 2);
    if (!c) Py_RETURN_NONE;
    Reference held{(PyObject*)c};  // another thread may drop it from the table meanwhile
    Py_INCREF(c);
    if (c->revision >= 0) {
      long long now = 0;
      if (!int_attr(c->words, sRevision, now)) return nullptr;
      if (now != c->revision) {  // what the copied descriptor points at may be gone: the call is built again
        drop(self, c);
        Py_RETURN_NONE;
      }
    }
    return launch(c, args + 2, at, args[1]);
  });
}

Py_ssize_t table_len(Table* self) { return (Py_ssize_t)self->order->size(); }

PyMethodDef table_methods[] = {{"add", (PyCFunction)table_add, METH_O, "Keep a Call; past the limit the one unused for longest goes."},
                               {"launch", (PyCFunction)(void (*)())table_launch, METH_FASTCALL,
                                "launch(key, alpha, *tensors) -> the tag of the Call that was issued, or None."},
                               {nullptr, nullptr, 0, nullptr}};
PySequenceMethods table_sequence = {(lenfunc)table_len};
PyTypeObject TableType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// setup(current_stream, is_capturing, report): how the module asks for torch's stream and reports error codes.
PyObject* setup(PyObject*, PyObject* args) {
  PyObject *stream, *capturing, *rep;
  if (!PyArg_ParseTuple(args, "OOO", &stream, &capturing, &rep)) return nullptr;
  Py_INCREF(stream);
  Py_INCREF(capturing);
  Py_INCREF(rep);
  Py_XSETREF(current_stream, stream);
  Py_XSETREF(is_capturing, capturing);
  Py_XSETREF(report, rep);
  Py_RETURN_NONE;
}
PyMethodDef module_methods[] = {{"setup", setup, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  CallType.tp_name = "tileccl_amd._host.Call";
  CallType.tp_basicsize = sizeof(Call);
  CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  CallType.tp_new = PyType_GenericNew;
  CallType.tp_init = (initproc)call_init;
  CallType.tp_dealloc = (destructor)call_dealloc;
  CallType.tp_traverse = (traverseproc)call_traverse;
  CallType.tp_clear = (inquiry)call_clear;
  TableType.tp_name = "tileccl_amd._host.Table";
  TableType.tp_basicsize = sizeof(Table);
  TableType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  TableType.tp_new = table_new;
  TableType.tp_dealloc = (destructor)table_dealloc;
  TableType.tp_traverse = (traverseproc)table_traverse;
  TableType.tp_clear = (inquiry)table_clear;
  TableType.tp_methods = table_methods;
  TableType.tp_as_sequence = &table_sequence;
  if (PyType_Ready(&CallType) < 0 || PyType_Ready(&TableType) < 0) return nullptr;
  kGemm = PyUnicode_FromString("GEMM");
  kSync = PyUnicode_FromString("SYNC");
  sEpoch = PyUnicode_InternFromString("epoch");
  sLockEpoch = PyUnicode_InternFromString("lock_epoch");
  sClear = PyUnicode_InternFromString("clear_every_launch");
  sMaxTasks = PyUnicode_InternFromString("max_tasks_per_tile");
  sSpin = PyUnicode_InternFromString("spin_limit_ns");
  sNext = PyUnicode_InternFromString("next_epoch");
  sRevision = PyUnicode_InternFromString("revision");
  device0 = PyLong_FromLong(0);  // every rank lives on device 0
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&CallType);
  Py_INCREF(&TableType);
  Py_INCREF(kGemm);
  Py_INCREF(kSync);
  PyModule_AddObject(m, "Call", (PyObject*)&CallType);
  PyModule_AddObject(m, "Table", (PyObject*)&TableType);
  PyModule_AddObject(m, "GEMM", kGemm);
  PyModule_AddObject(m, "SYNC", kSync);
  return m;
}
