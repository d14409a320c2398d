// The way from Python to the kernels' C entries: the call itself without an argument object per parameter (ctypes took some 4 us a
// call), and the operand checks of what every layer runs without an interpreter's step per question (another 4 us a product). A
// step of a few short prompts (24 layers of 0.5B sizes, 172 calls) waited for the host: 2.21 ms with 1.27 ms of kernels, 1.47 so. The layers of a step that are alike make one layer's calls again
// (tape, play below; engine/tapes.py).
// A check here answers the sizes that the launch needs, or nothing: what it does not pass goes to the checks in Python, which take what is
// left to other kernels and say what is wrong with the rest. Nothing is remembered from call to call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <memory>
#include <utility>
#include <vector>

namespace {

using at::Tensor;

enum Code : int { kF32 = 0, kBF16 = 1, kI32 = 2, kI64 = 3, kOther = 9 };      // (the first two as the C entries take them)

int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return kF32;
    case at::kBFloat16: return kBF16;
    case at::kInt: return kI32;
    case at::kLong: return kI64;
    default: return kOther;
  }
}

// the tensor behind an argument, on the GPU and of that rank; null for anything else
const Tensor* gpu(PyObject* o, int64_t rank) {
  if (!THPVariable_Check(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.dim() == rank ? &t : nullptr;
}
const Tensor* dense(PyObject* o, int64_t rank, int code) {
  const Tensor* t = gpu(o, rank);
  return t && code_of(*t) == code && t->is_contiguous() ? t : nullptr;
}
// the leading dimension of a matrix with contiguous rows; -1 for anything else
int64_t leading(const Tensor& t) {
  const int64_t rows = t.size(0), columns = t.size(1);
  if (t.stride(1) != 1 && columns > 1) return -1;
  return rows > 1 ? t.stride(0) : std::max(t.stride(0), columns);
}
bool aligned(const Tensor& t, uintptr_t to) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % to == 0; }

#define NOT_HERE Py_RETURN_NONE

// product(out, a, w, w2 or None, bias or None) -> (M, N, K, ldo, lda, ldw, code of out): a bfloat16 product that the matrix-core kernels take
// (with w2, the up projection beside the gate's: out is bfloat16 too)
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) NOT_HERE;
  const Tensor *out = gpu(args[0], 2), *a = gpu(args[1], 2), *w = gpu(args[2], 2);
  if (!out || !a || !w || code_of(*a) != kBF16 || code_of(*w) != kBF16) NOT_HERE;
  const int oc = code_of(*out);
  const int64_t M = a->size(0), K = a->size(1), N = w->size(0);
  if ((oc != kF32 && oc != kBF16) || w->size(1) != K || out->size(0) != M || out->size(1) != N || K % 8) NOT_HERE;
  const int64_t ldo = leading(*out), lda = leading(*a), ldw = leading(*w);
  if (ldo < 0 || lda < 0 || ldw < 0 || lda % 8 || ldw % 8 || !aligned(*a, 16) || !aligned(*w, 16)) NOT_HERE;
  if (args[3] != Py_None) {
    const Tensor* w2 = gpu(args[3], 2);
    if (!w2 || oc != kBF16 || code_of(*w2) != kBF16 || w2->size(0) != N || w2->size(1) != K || leading(*w2) != ldw || !aligned(*w2, 16)) NOT_HERE;
  }
  if (args[4] != Py_None) {
    const Tensor* b = dense(args[4], 1, kF32);
    if (!b || b->size(0) != N) NOT_HERE;
  }
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) NOT_HERE;
  return Py_BuildValue("LLLLLLi", (long long)M, (long long)N, (long long)K, (long long)ldo, (long long)lda, (long long)ldw, oc);
}

// norm(out, x, weight, rows or None) -> (rows of out, width, code of out)
PyObject* norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) NOT_HERE;
  const Tensor *out = gpu(args[0], 2), *x = dense(args[1], 2, kF32), *w = dense(args[2], 1, kF32);
  if (!out || !x || !w || !out->is_contiguous()) NOT_HERE;
  const int oc = code_of(*out);
  const int64_t rows = out->size(0), width = out->size(1);
  if ((oc != kF32 && oc != kBF16) || x->size(1) != width || w->size(0) != width || rows > INT32_MAX || width > INT32_MAX) NOT_HERE;
  if (args[3] != Py_None) {
    const Tensor* r = dense(args[3], 1, kI32);
    if (!r || r->size(0) != rows) NOT_HERE;
  } else if (x->size(0) != rows) {
    NOT_HERE;
  }
  return Py_BuildValue("LLi", (long long)rows, (long long)width, oc);
}

// caches [blocks, kv_heads, block_size, d] and [blocks, kv_heads, d, block_size] of one type: their block size, or -1
int64_t pages(PyObject* k_o, PyObject* v_o, int64_t kv_heads, int64_t d) {
  const Tensor *k = gpu(k_o, 4), *v = gpu(v_o, 4);
  if (!k || !v || k->scalar_type() != v->scalar_type() || !k->is_contiguous() || !v->is_contiguous()) return -1;
  if (k->size(1) != kv_heads || v->size(1) != kv_heads || k->size(3) != d || v->size(2) != d || k->size(2) != v->size(3) || k->size(0) != v->size(0)) return -1;
  return k->size(2) <= INT32_MAX ? k->size(2) : -1;
}

// caches(k_cache, v_cache, kv_heads, d) -> block size
PyObject* caches(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) NOT_HERE;
  const int64_t kv = PyLong_AsLongLong(args[2]), d = PyLong_AsLongLong(args[3]);
  if (PyErr_Occurred()) { PyErr_Clear(); NOT_HERE; }
  const int64_t bs = pages(args[0], args[1], kv, d);
  if (bs < 0) NOT_HERE;
  return PyLong_FromLongLong(bs);
}

// turn(qkv, cos, sin, positions, slots, k_cache, v_cache, heads, kv_heads, d) -> (rows, leading dimension, code, block size)
PyObject* turn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 10) NOT_HERE;
  const Tensor *qkv = gpu(args[0], 2), *cos = dense(args[1], 2, kF32), *sin = dense(args[2], 2, kF32), *pos = dense(args[3], 1, kI32), *slots = dense(args[4], 1, kI64);
  const int64_t heads = PyLong_AsLongLong(args[7]), kv = PyLong_AsLongLong(args[8]), d = PyLong_AsLongLong(args[9]);
  if (PyErr_Occurred()) { PyErr_Clear(); NOT_HERE; }
  if (!qkv || !cos || !sin || !pos || !slots || heads <= 0 || kv <= 0 || d <= 0 || d % 2) NOT_HERE;
  const int code = code_of(*qkv);
  const int64_t T = qkv->size(0), ld = leading(*qkv);
  if ((code != kF32 && code != kBF16) || T > INT32_MAX || qkv->size(1) != (heads + 2 * kv) * d || ld < 0) NOT_HERE;
  if (cos->size(0) != sin->size(0) || cos->size(1) != d / 2 || sin->size(1) != d / 2 || pos->size(0) != T || slots->size(0) != T) NOT_HERE;
  const int64_t bs = pages(args[5], args[6], kv, d);
  if (bs < 0 || THPVariable_Unpack(args[5]).scalar_type() != qkv->scalar_type()) NOT_HERE;
  return Py_BuildValue("LLiL", (long long)T, (long long)ld, code, (long long)bs);
}

// attention(out, q, k_cache, v_cache, block_table, heads, kv_heads, d) -> (rows, block size): bfloat16 queries and caches as the matrix-core kernels take
// them, out bfloat16 or float32
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 8) NOT_HERE;
  const Tensor *out = gpu(args[0], 2), *q = gpu(args[1], 2), *table = dense(args[4], 2, kI32);
  const int64_t heads = PyLong_AsLongLong(args[5]), kv = PyLong_AsLongLong(args[6]), d = PyLong_AsLongLong(args[7]);
  if (PyErr_Occurred()) { PyErr_Clear(); NOT_HERE; }
  if (!out || !q || !table || code_of(*q) != kBF16 || heads <= 0 || kv <= 0 || heads % kv || d % 16 || d < 16 || d > 256) NOT_HERE;
  const int oc = code_of(*out);
  const int64_t T = q->size(0), ldo = leading(*out), ldq = leading(*q);
  if ((oc != kBF16 && oc != kF32) || out->size(0) != T || out->size(1) < heads * d || q->size(1) < heads * d || ldo < 0 || ldq < 0 || ldo % 4 || ldq % 8) NOT_HERE;
  if (!aligned(*q, 16) || !aligned(*out, oc == kF32 ? 16 : 8)) NOT_HERE;
  const int64_t bs = pages(args[2], args[3], kv, d);
  if (bs < 8 || (bs & (bs - 1)) || THPVariable_Unpack(args[2]).scalar_type() != at::kBFloat16) NOT_HERE;
  return Py_BuildValue("LL", (long long)T, (long long)bs);
}

// call(address, ...): the C entry at that address with a tensor's memory, a number, a float or nothing (a null pointer) for each parameter; its
// answer. In the calling convention of x86-64 (System V), the only host that this library is built for, integers and pointers travel apart from
// floats, each kind in its own order whatever the order between them, floats up to the eighth in registers only, and the caller takes its
// parameters off the stack again: one signature of many 64-bit integers and eight floats serves every entry, which looks at what it has.
#if !defined(__x86_64__) || !defined(__linux__)
#error "call() is written for the x86-64 System V calling convention"
#endif
constexpr int kInts = 48, kFloats = 8;
using I = int64_t;
using F = float;
using Entry = int (*)(I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I,
                      I, I, I, I, I, F, F, F, F, F, F, F, F);

// A call as it was made: for `note` and `play`.
struct Call {
  Entry entry;
  I i[kInts];
  F f[kFloats];
  int ni;
};
int make(const Call& c) {
  const I* i = c.i;
  const F* f = c.f;
  return c.entry(i[0], i[1], i[2], i[3], i[4], i[5], i[6], i[7], i[8], i[9], i[10], i[11], i[12], i[13], i[14], i[15], i[16], i[17], i[18], i[19], i[20],
                 i[21], i[22], i[23], i[24], i[25], i[26], i[27], i[28], i[29], i[30], i[31], i[32], i[33], i[34], i[35], i[36], i[37], i[38], i[39],
                 i[40], i[41], i[42], i[43], i[44], i[45], i[46], i[47], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
}

// A tape: calls in their order, and which of their parameters lie in a memory range of the layer that they were made for (range, offset); `play` makes them for another layer.
struct Tape {
  struct Patch {
    int call, parameter, range;
    I offset;
  };
  std::vector<Call> calls;
  std::vector<Patch> patches;
  int ranges = 0;
};
thread_local Tape* noting = nullptr;

bool read_call(PyObject* const* args, Py_ssize_t n, Call& c) {
  I* i = c.i;
  F* f = c.f;
  int ni = 0, nf = 0;
  if (n < 1) {
    PyErr_SetString(PyExc_TypeError, "call: an address comes first");
    return false;
  }
  const Entry entry = reinterpret_cast<Entry>(PyLong_AsVoidPtr(args[0]));
  if (PyErr_Occurred() || entry == nullptr) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "call: no such entry");
    return false;
  }
  for (Py_ssize_t k = 1; k < n; ++k) {
    PyObject* o = args[k];
    if (PyFloat_Check(o)) {
      if (nf == kFloats) { PyErr_SetString(PyExc_TypeError, "call: too many floats"); return false; }
      f[nf++] = static_cast<float>(PyFloat_AS_DOUBLE(o));
      continue;
    }
    if (ni == kInts) { PyErr_SetString(PyExc_TypeError, "call: too many parameters"); return false; }
    if (PyLong_Check(o)) {
      i[ni] = PyLong_AsLongLong(o);
      if (i[ni++] == -1 && PyErr_Occurred()) return false;
    } else if (o == Py_None) {
      i[ni++] = 0;
    } else if (THPVariable_Check(o)) {
      i[ni++] = reinterpret_cast<I>(THPVariable_Unpack(o).data_ptr());
    } else {
      PyErr_Format(PyExc_TypeError, "call: parameter %zd is no tensor, number or None", k);
      return false;
    }
  }
  c.entry = entry, c.ni = ni;
  return true;
}

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Call c{};
  if (!read_call(args, n, c)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = make(c);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// note(address, ...): call, kept on this thread's tape as well (if it is being written and the call went well)
PyObject* note(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Call c{};
  if (!read_call(args, n, c)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = make(c);
  Py_END_ALLOW_THREADS
  if (noting && rc == 0) noting->calls.push_back(c);
  return PyLong_FromLong(rc);
}

void drop_tape(PyObject* capsule) { delete static_cast<Tape*>(PyCapsule_GetPointer(capsule, "alofa.tape")); }

// tape(): this thread's calls are noted from now on (what an interrupted step left is dropped)
PyObject* tape(PyObject*, PyObject* const*, Py_ssize_t) {
  delete noting;
  noting = nullptr;
  noting = new Tape;
  Py_RETURN_NONE;
}

// taped((address, bytes), ...): the calls since, for `play`; the ranges are the memory of the layer that they were made for
PyObject* taped(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!noting) {
    PyErr_SetString(PyExc_RuntimeError, "taped: no tape is being written");
    return nullptr;
  }
  std::unique_ptr<Tape> t(noting);
  noting = nullptr;
  std::vector<std::pair<I, I>> ranges;
  for (Py_ssize_t k = 0; k < n; ++k) {
    if (!PyTuple_Check(args[k]) || PyTuple_GET_SIZE(args[k]) != 2) { PyErr_SetString(PyExc_TypeError, "taped: ranges are pairs"); return nullptr; }
    ranges.emplace_back(PyLong_AsLongLong(PyTuple_GET_ITEM(args[k], 0)), PyLong_AsLongLong(PyTuple_GET_ITEM(args[k], 1)));
  }
  if (PyErr_Occurred()) return nullptr;
  t->ranges = static_cast<int>(ranges.size());
  for (size_t c = 0; c < t->calls.size(); ++c)
    for (int k = 0; k < t->calls[c].ni; ++k)
      for (size_t r = 0; r < ranges.size(); ++r) {
        const I off = t->calls[c].i[k] - ranges[r].first;
        if (off >= 0 && off < ranges[r].second) {
          t->patches.push_back({static_cast<int>(c), k, static_cast<int>(r), off});
          break;
        }
      }
  PyObject* capsule = PyCapsule_New(t.get(), "alofa.tape", drop_tape);
  if (capsule) t.release();
  return capsule;
}

// play(tape, (address, ...)): the tape's calls for a layer whose memory ranges begin there; the first answer that is not zero, or zero
PyObject* play(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyCapsule_IsValid(args[0], "alofa.tape") || !PyTuple_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "play: a tape and the addresses of a layer");
    return nullptr;
  }
  Tape& t = *static_cast<Tape*>(PyCapsule_GetPointer(args[0], "alofa.tape"));
  if (PyTuple_GET_SIZE(args[1]) != t.ranges) { PyErr_SetString(PyExc_ValueError, "play: another count of ranges than the tape's"); return nullptr; }
  std::vector<I> at(t.ranges);
  for (int r = 0; r < t.ranges; ++r) at[r] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[1], r));
  if (PyErr_Occurred()) return nullptr;
  for (const Tape::Patch& p : t.patches) t.calls[p.call].i[p.parameter] = at[p.range] + p.offset;
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS
  for (const Call& c : t.calls) {
    rc = make(c);
    if (rc != 0) break;
  }
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// a C++ exception does not pass through the interpreter: what could not be looked at is "not here"
template <PyObject* (*kCheck)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  try {
    return kCheck(self, args, n);
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}
template <PyObject* (*kCall)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded_call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  try {
    return kCall(self, args, n);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

#define METHOD(name, function) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(function)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD("product", guarded<product>), METHOD("norm", guarded<norm>), METHOD("caches", guarded<caches>), METHOD("turn", guarded<turn>), METHOD("attention", guarded<attention>),
                         METHOD("call", guarded_call<call>), METHOD("note", guarded_call<note>), METHOD("tape", guarded_call<tape>), METHOD("taped", guarded_call<taped>),
                         METHOD("play", guarded_call<play>), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "alofa_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_alofa_fastcall() { return PyModule_Create(&module); }
