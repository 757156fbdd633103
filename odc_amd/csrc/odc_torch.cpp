// odc_torch.cpp — the host path between a service call in Python and the C ABI of include/odc_hip.h:
// reads tensors and Python lists, fills the item arrays and makes the call. A CPython extension
// module (no pybind), plain C++ against torch's headers; it links no HIP code and no libodc_hip.so:
// the entry points are bound by address (bind()), so that it always calls the library that
// odc_amd/_native.py loaded. It reads at::Tensor and CPython objects by their layout and fills the
// structures of the C ABI, so it says what it was built for (built_for) and the loader compares.
//
// What bounds small calls is this path: a launch itself costs the host 2.5-3.5 us and the device
// 2-3 us, while reading the tensors of a call attribute by attribute in Python took 3-5 us for one
// tensor and about 0.9 us for each further one (300 slices: 130 us), and hashing the lists that
// named a cached plan as much again. In C++ a tensor costs about 30 ns and the items are simply
// filled anew on every call: nothing is remembered from one call to the next, so nothing can be
// stale. The GIL is released around the library calls.

#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/as_strided.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstddef>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "odc_hip.h"

#ifndef ODC_TORCH_VERSION
#error "ODC_TORCH_VERSION: the torch.__version__ that this is compiled against"
#endif

namespace {

// ------------------------------------------------------------------------------------------------
// the library
// ------------------------------------------------------------------------------------------------
decltype(&odc_gather) p_gather = nullptr;
decltype(&odc_gather_cast) p_gather_cast = nullptr;
decltype(&odc_scatter_accumulate) p_scatter_accumulate = nullptr;
decltype(&odc_scatter_store) p_scatter_store = nullptr;
decltype(&odc_clear) p_clear = nullptr;
decltype(&odc_publish) p_publish = nullptr;
decltype(&odc_arena_locate) p_arena_locate = nullptr;
decltype(&odc_last_error) p_last_error = nullptr;

// bind(name, address, ...): every entry point this module calls.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i + 1 < n; i += 2) {
    const char* name = PyUnicode_AsUTF8(args[i]);
    void* address = PyLong_AsVoidPtr(args[i + 1]);
    if (PyErr_Occurred()) return nullptr;
#define ODC_BIND(symbol) \
  if (!strcmp(name, "odc_" #symbol)) { p_##symbol = reinterpret_cast<decltype(p_##symbol)>(address); continue; }
    ODC_BIND(gather)
    ODC_BIND(gather_cast)
    ODC_BIND(scatter_accumulate)
    ODC_BIND(scatter_store)
    ODC_BIND(clear)
    ODC_BIND(publish)
    ODC_BIND(arena_locate)
    ODC_BIND(last_error)
#undef ODC_BIND
    PyErr_Format(PyExc_ValueError, "bind: unknown entry point %s", name);
    return nullptr;
  }
  if (!p_gather || !p_gather_cast || !p_scatter_accumulate || !p_scatter_store || !p_clear || !p_publish ||
      !p_arena_locate || !p_last_error) {
    PyErr_SetString(PyExc_RuntimeError, "bind: an entry point is missing");
    return nullptr;
  }
  Py_RETURN_NONE;
}

// ------------------------------------------------------------------------------------------------
// reading Python values
// ------------------------------------------------------------------------------------------------
struct Failed {};  // a Python exception is set

template <class... Args>
[[noreturn]] void raise(PyObject* type, const char* format, Args... args) {
  PyErr_Format(type, format, args...);
  throw Failed();
}

#define ODC_ASSERT(cond, ...) \
  do {                        \
    if (!(cond)) raise(PyExc_AssertionError, __VA_ARGS__); \
  } while (0)

// A C++ exception (from torch) or Failed becomes the Python exception of a nullptr return.
template <class F>
PyObject* guarded(F body) {
  try {
    return body();
  } catch (const Failed&) {
    return nullptr;
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

void expect_args(Py_ssize_t n, Py_ssize_t want) {
  if (n != want) raise(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
}

// The value of an int object; the reference to it is given up. Negative ones fail like the size
// checks they come from.
uint64_t take_u64(PyObject* i) {
  if (!i) throw Failed();
  const unsigned long long v = PyLong_AsUnsignedLongLong(i);
  Py_DECREF(i);
  if (v == (unsigned long long)-1 && PyErr_Occurred()) {
    PyErr_Clear();
    raise(PyExc_AssertionError, "an offset or a size is negative or does not fit 64 bits");
  }
  return v;
}

uint64_t as_u64(PyObject* o) {
  if (PyLong_CheckExact(o)) {
    Py_INCREF(o);
    return take_u64(o);
  }
  return take_u64(PyNumber_Index(o));  // anything with __index__ (numpy integers)
}

// int(o): a count that the caller may have left a float or a tensor of one element
uint64_t as_count(PyObject* o) { return PyLong_CheckExact(o) ? as_u64(o) : take_u64(PyNumber_Long(o)); }

void* as_pointer(PyObject* o) { return reinterpret_cast<void*>((uintptr_t)as_u64(o)); }

// A list or tuple, or any other sequence as a list of its items.
class Sequence {
 public:
  Sequence(PyObject* o, const char* what) : fast_(PySequence_Fast(o, what)) {
    if (!fast_) throw Failed();
  }
  ~Sequence() { Py_DECREF(fast_); }
  Sequence(const Sequence&) = delete;
  Sequence& operator=(const Sequence&) = delete;
  Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(fast_); }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(fast_, i); }

 private:
  PyObject* fast_;
};

const at::Tensor& as_tensor(PyObject* o) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "expected a torch.Tensor, got %s", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return ODC_DTYPE_BF16;
    case at::kHalf: return ODC_DTYPE_F16;
    case at::kFloat: return ODC_DTYPE_F32;
    default: return -1;
  }
}

int supported_dtype_code(const char* what, at::ScalarType t) {
  const int code = dtype_code(t);
  if (code < 0) raise(PyExc_TypeError, "%s supports bf16/fp16/fp32, not %s", what, at::toString(t));
  return code;
}

uint64_t dtype_bytes(int code) { return code == ODC_DTYPE_F32 ? 4 : 2; }

// Symmetric byte offset of a tensor that is (a contiguous view into) a live symmetric allocation.
uint64_t symmetric_offset(const odc_arena* arena, const at::Tensor& t) {
  uint64_t allocation = 0, inner = 0;
  if (p_arena_locate(arena, t.data_ptr(), nullptr, &allocation, &inner) != ODC_OK)
    raise(PyExc_ValueError, "tensor is not in the symmetric arena: %s", p_last_error());
  return allocation + inner;
}

// ------------------------------------------------------------------------------------------------
// gather
// ------------------------------------------------------------------------------------------------
struct GatherCall {
  odc_arena* arena;
  uint32_t world, rank;
  void* stream;
  at::ScalarType src;
  bool started = false;
  at::ScalarType dst = at::kByte;
  std::vector<odc_gather_item> plain;  // the same three words as odc_gather_cast_item

  // `out` takes W x numel elements gathered from symmetric byte offset `offset`
  void add(const at::Tensor& out, uint64_t offset, uint64_t numel) {
    if (!started) {
      dst = out.scalar_type();
      started = true;
    }
    ODC_ASSERT(out.is_cuda(), "gather runs on the GPU only");
    ODC_ASSERT(out.scalar_type() == dst, "one launch takes one dtype pair");
    ODC_ASSERT(out.is_contiguous(), "outputs are contiguous");
    ODC_ASSERT((uint64_t)out.numel() == numel * world, "output numel %lld != %u * shard numel %llu",
               (long long)out.numel(), world, (unsigned long long)numel);
    add_raw(out.data_ptr(), offset, numel);
  }

  void add_raw(void* out, uint64_t offset, uint64_t numel) {
    plain.push_back({out, offset, src == dst ? numel * at::elementSize(src) : numel});
  }

  int launch() {
    if (plain.empty()) return ODC_OK;
    if (src == dst) {
      int status;
      Py_BEGIN_ALLOW_THREADS
      status = p_gather(arena, plain.data(), (uint32_t)plain.size(), rank, stream);
      Py_END_ALLOW_THREADS
      return status;
    }
    static_assert(sizeof(odc_gather_item) == sizeof(odc_gather_cast_item) &&
                      offsetof(odc_gather_item, src_offset) == offsetof(odc_gather_cast_item, src_offset) &&
                      offsetof(odc_gather_item, shard_bytes) == offsetof(odc_gather_cast_item, shard_elems),
                  "one item array serves both gathers");
    const int s = supported_dtype_code("a converting gather", src), d = supported_dtype_code("a converting gather", dst);
    const auto* items = reinterpret_cast<const odc_gather_cast_item*>(plain.data());
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = p_gather_cast(arena, items, (uint32_t)plain.size(), s, d, rank, stream);
    Py_END_ALLOW_THREADS
    return status;
  }
};

// gather(arena, world, rank, stream, outputs, shards) -> status
PyObject* gather(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 6);
    const Sequence outs(args[4], "outputs are a sequence"), shards(args[5], "shards are a sequence");
    ODC_ASSERT(outs.size() == shards.size() && shards.size() > 0, "one output per shard");
    GatherCall call{static_cast<odc_arena*>(as_pointer(args[0])), (uint32_t)as_u64(args[1]), (uint32_t)as_u64(args[2]),
                    as_pointer(args[3]), as_tensor(shards[0]).scalar_type()};
    call.plain.reserve((size_t)shards.size());
    for (Py_ssize_t k = 0; k < shards.size(); ++k) {
      const at::Tensor& shard = as_tensor(shards[k]);
      ODC_ASSERT(shard.is_cuda() && shard.is_contiguous(), "shards are contiguous GPU tensors");
      ODC_ASSERT(shard.scalar_type() == call.src, "one launch takes one dtype pair");
      const at::Tensor& out = as_tensor(outs[k]);
      if (shard.numel() == 0) {  // an empty shard has an empty output and takes no part in the launch
        ODC_ASSERT(out.numel() == 0, "output %zd is not empty but its shard is", k);
        continue;
      }
      call.add(out, symmetric_offset(call.arena, shard), (uint64_t)shard.numel());
    }
    return PyLong_FromLong(call.launch());
  });
}

// gather_slices(arena, world, rank, stream, outputs, input, slice_offsets, slice_numels) -> status
PyObject* gather_slices(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 8);
    const Sequence outs(args[4], "outputs are a sequence"), offsets(args[6], "slice offsets are a sequence"),
        numels(args[7], "slice sizes are a sequence");
    ODC_ASSERT(outs.size() == offsets.size() && outs.size() == numels.size(), "one offset and size per output");
    const at::Tensor& input = as_tensor(args[5]);
    GatherCall call{static_cast<odc_arena*>(as_pointer(args[0])), (uint32_t)as_u64(args[1]), (uint32_t)as_u64(args[2]),
                    as_pointer(args[3]), input.scalar_type()};
    const uint64_t total = (uint64_t)input.numel(), bytes = input.element_size();
    uint64_t base = 0;
    bool located = false;  // an empty buffer has no address
    call.plain.reserve((size_t)outs.size());
    for (Py_ssize_t k = 0; k < outs.size(); ++k) {
      const uint64_t off = as_u64(offsets[k]), m = as_u64(numels[k]);
      ODC_ASSERT(off <= total && m <= total - off, "slice leaves the buffer");
      const at::Tensor& out = as_tensor(outs[k]);
      if (m == 0 && out.numel() == 0) continue;
      if (!located) base = symmetric_offset(call.arena, input);
      located = true;
      call.add(out, base + off * bytes, m);
    }
    return PyLong_FromLong(call.launch());
  });
}

// ------------------------------------------------------------------------------------------------
// scatter-accumulate: a batch is the item array of one call, filled and checked before the
// service's bookkeeping decides how it is launched
// ------------------------------------------------------------------------------------------------
struct Batch {
  PyObject_HEAD
  std::vector<odc_accum_item>* items;
  int grad_code, acc_code;
};

PyTypeObject* batch_type = nullptr;

Batch* new_batch() {
  Batch* b = PyObject_New(Batch, batch_type);
  if (!b) throw Failed();
  b->items = new std::vector<odc_accum_item>();
  b->grad_code = b->acc_code = -1;
  return b;
}

void batch_dealloc(PyObject* self) {
  PyTypeObject* type = Py_TYPE(self);
  delete reinterpret_cast<Batch*>(self)->items;
  PyObject_Free(self);
  Py_DECREF(type);
}

// Owns a batch until it is handed to Python.
struct BatchRef {
  Batch* b = new_batch();
  ~BatchRef() { Py_XDECREF(reinterpret_cast<PyObject*>(b)); }
  PyObject* release() {
    PyObject* o = reinterpret_cast<PyObject*>(b);
    b = nullptr;
    return o;
  }
};

// Where an accumulation lies, as the service notes it at registration: (offset, elements, dtype code)
struct Accumulation {
  uint64_t offset, numel;
  int code;
};

Accumulation as_accumulation(PyObject* entry) {
  if (!PyTuple_Check(entry) || PyTuple_GET_SIZE(entry) != 3) raise(PyExc_TypeError, "bad accumulation table entry");
  return {as_u64(PyTuple_GET_ITEM(entry, 0)), as_u64(PyTuple_GET_ITEM(entry, 1)), (int)as_u64(PyTuple_GET_ITEM(entry, 2))};
}

void check_grad(const at::Tensor& grad, at::ScalarType dtype) {
  ODC_ASSERT(grad.is_cuda(), "scatter-accumulate runs on the GPU only");
  ODC_ASSERT(grad.scalar_type() == dtype, "one launch takes one gradient dtype");
  ODC_ASSERT(grad.is_contiguous(), "gradients are contiguous");
}

// accumulate_batch(table, world, keys, gradients, valid_numels or None) -> batch, or None when a
// key is not in the table (the service registers it and asks again)
PyObject* accumulate_batch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    expect_args(n, 5);
    const uint64_t world = as_u64(args[1]);
    const Sequence keys(args[2], "keys are a sequence"), grads(args[3], "gradients are a sequence");
    const bool padded = args[4] != Py_None;
    const Sequence valid(padded ? args[4] : args[2], "valid_numels is a sequence");
    ODC_ASSERT(grads.size() == keys.size(), "one gradient per key");
    ODC_ASSERT(valid.size() >= keys.size(), "one valid_numel per key");
    if (!keys.size()) Py_RETURN_NONE;
    BatchRef ref;
    std::vector<odc_accum_item>& items = *ref.b->items;
    items.reserve((size_t)keys.size());
    const at::ScalarType dtype = as_tensor(grads[0]).scalar_type();
    ref.b->grad_code = supported_dtype_code("scatter-accumulate", dtype);
    for (Py_ssize_t k = 0; k < keys.size(); ++k) {
      PyObject* entry = PyDict_GetItemWithError(args[0], keys[k]);
      if (!entry) {
        if (PyErr_Occurred()) throw Failed();
        Py_RETURN_NONE;
      }
      const Accumulation acc = as_accumulation(entry);
      const at::Tensor& grad = as_tensor(grads[k]);
      check_grad(grad, dtype);
      const uint64_t numel = (uint64_t)grad.numel();
      uint64_t elems = numel;
      if (padded) {
        elems = as_count(valid[k]);
        ODC_ASSERT(elems <= numel && elems <= world * acc.numel,
                   "valid_numel %llu exceeds the gradient (%llu) or the %llu elements of the key's shards",
                   (unsigned long long)elems, (unsigned long long)numel, (unsigned long long)(world * acc.numel));
      } else {
        ODC_ASSERT(grad.dim() == 1, "gradients are flat");
        ODC_ASSERT(numel % world == 0, "gradient of %llu elements does not divide over %llu ranks",
                   (unsigned long long)numel, (unsigned long long)world);
        ODC_ASSERT(numel / world == acc.numel, "key %R: registered shard %llu, gradient implies %llu", keys[k],
                   (unsigned long long)acc.numel, (unsigned long long)(numel / world));
      }
      ODC_ASSERT(ref.b->acc_code < 0 || ref.b->acc_code == acc.code, "one launch takes one accumulation dtype");
      ref.b->acc_code = acc.code;
      items.push_back({grad.data_ptr(), elems, acc.offset, acc.numel});
    }
    return ref.release();
  });
}

// batch.launch(arena, stream, store) -> status
PyObject* batch_launch(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 3);
    Batch* b = reinterpret_cast<Batch*>(self);
    odc_arena* arena = static_cast<odc_arena*>(as_pointer(args[0]));
    void* stream = as_pointer(args[1]);
    const auto entry = args[2] == Py_True ? p_scatter_store : p_scatter_accumulate;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = entry(arena, b->items->data(), (uint32_t)b->items->size(), b->grad_code, b->acc_code, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
  });
}

// batch.pick(indices) -> a batch of those items
PyObject* batch_pick(PyObject* self, PyObject* indices) {
  return guarded([&] {
    Batch* b = reinterpret_cast<Batch*>(self);
    const Sequence picked(indices, "indices are a sequence");
    BatchRef ref;
    ref.b->grad_code = b->grad_code;
    ref.b->acc_code = b->acc_code;
    for (Py_ssize_t k = 0; k < picked.size(); ++k) ref.b->items->push_back(b->items->at(as_u64(picked[k])));
    return ref.release();
  });
}

Py_ssize_t batch_len(PyObject* self) { return (Py_ssize_t)reinterpret_cast<Batch*>(self)->items->size(); }
PyObject* batch_grad_code(PyObject* self, void*) { return PyLong_FromLong(reinterpret_cast<Batch*>(self)->grad_code); }
PyObject* batch_acc_code(PyObject* self, void*) { return PyLong_FromLong(reinterpret_cast<Batch*>(self)->acc_code); }

PyMethodDef batch_methods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(batch_launch)), METH_FASTCALL, nullptr},
    {"pick", batch_pick, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef batch_getset[] = {{"grad_code", batch_grad_code, nullptr, nullptr, nullptr},
                              {"acc_code", batch_acc_code, nullptr, nullptr, nullptr},
                              {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyType_Slot batch_slots[] = {{Py_tp_dealloc, reinterpret_cast<void*>(batch_dealloc)},
                             {Py_tp_methods, batch_methods},
                             {Py_tp_getset, batch_getset},
                             {Py_sq_length, reinterpret_cast<void*>(batch_len)},
                             {0, nullptr}};
PyType_Spec batch_spec = {"odc_torch.Batch", sizeof(Batch), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_DISALLOW_INSTANTIATION, batch_slots};

// ------------------------------------------------------------------------------------------------
// slices of one accumulation
// ------------------------------------------------------------------------------------------------
struct SliceLayout {
  PyObject_HEAD
  std::vector<uint64_t>* offsets;
  std::vector<uint64_t>* numels;
};

PyTypeObject* slice_layout_type = nullptr;

void slice_layout_dealloc(PyObject* self) {
  PyTypeObject* type = Py_TYPE(self);
  delete reinterpret_cast<SliceLayout*>(self)->offsets;
  delete reinterpret_cast<SliceLayout*>(self)->numels;
  PyObject_Free(self);
  Py_DECREF(type);
}

// slice_layout(offsets, numels): the slices of one group, for the service to recognise and to fill
PyObject* slice_layout(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 2);
    const Sequence offsets(args[0], "slice offsets are a sequence"), numels(args[1], "slice sizes are a sequence");
    ODC_ASSERT(offsets.size() == numels.size(), "one offset per slice");
    auto o = std::make_unique<std::vector<uint64_t>>(), m = std::make_unique<std::vector<uint64_t>>();
    for (Py_ssize_t k = 0; k < offsets.size(); ++k) {
      o->push_back(as_u64(offsets[k]));
      m->push_back(as_u64(numels[k]));
    }
    SliceLayout* s = PyObject_New(SliceLayout, slice_layout_type);
    if (!s) throw Failed();
    s->offsets = o.release();
    s->numels = m.release();
    return reinterpret_cast<PyObject*>(s);
  });
}

// layout.matches(offsets, numels) -> whether these are its slices, number for number
PyObject* slice_layout_matches(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    expect_args(n, 2);
    const SliceLayout* s = reinterpret_cast<SliceLayout*>(self);
    const Sequence offsets(args[0], "slice offsets are a sequence"), numels(args[1], "slice sizes are a sequence");
    if (offsets.size() != (Py_ssize_t)s->offsets->size() || numels.size() != offsets.size()) Py_RETURN_FALSE;
    for (Py_ssize_t k = 0; k < offsets.size(); ++k)
      if (as_u64(offsets[k]) != (*s->offsets)[k] || as_u64(numels[k]) != (*s->numels)[k]) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
  });
}

// layout.batch(accumulation table entry, world, gradients) -> batch; gradient i holds at most
// world * numels[i] elements, what is missing reads as +0
PyObject* slice_layout_batch(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 3);
    const SliceLayout* s = reinterpret_cast<SliceLayout*>(self);
    const Accumulation acc = as_accumulation(args[0]);
    const uint64_t world = as_u64(args[1]), bytes = dtype_bytes(acc.code);
    const Sequence grads(args[2], "gradients are a sequence");
    ODC_ASSERT((size_t)grads.size() == s->offsets->size() && grads.size() > 0, "one gradient per slice");
    BatchRef ref;
    ref.b->acc_code = acc.code;
    ref.b->items->reserve((size_t)grads.size());
    const at::ScalarType dtype = as_tensor(grads[0]).scalar_type();
    ref.b->grad_code = supported_dtype_code("scatter-accumulate", dtype);
    for (Py_ssize_t k = 0; k < grads.size(); ++k) {
      const at::Tensor& grad = as_tensor(grads[k]);
      check_grad(grad, dtype);
      const uint64_t off = (*s->offsets)[k], m = (*s->numels)[k], numel = (uint64_t)grad.numel();
      ODC_ASSERT(off <= acc.numel && m <= acc.numel - off, "slice leaves the accumulation");
      ODC_ASSERT(numel <= world * m, "gradient %zd has %llu > %llu * %llu elements", k, (unsigned long long)numel,
                 (unsigned long long)world, (unsigned long long)m);
      ref.b->items->push_back({grad.data_ptr(), numel, acc.offset + off * bytes, m});
    }
    return ref.release();
  });
}

PyMethodDef slice_layout_methods[] = {
    {"matches", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(slice_layout_matches)), METH_FASTCALL, nullptr},
    {"batch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(slice_layout_batch)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyType_Slot slice_layout_slots[] = {{Py_tp_dealloc, reinterpret_cast<void*>(slice_layout_dealloc)},
                                    {Py_tp_methods, slice_layout_methods},
                                    {0, nullptr}};
PyType_Spec slice_layout_spec = {"odc_torch.SliceLayout", sizeof(SliceLayout), 0,
                                 Py_TPFLAGS_DEFAULT | Py_TPFLAGS_DISALLOW_INSTANTIATION, slice_layout_slots};

// ------------------------------------------------------------------------------------------------
// clear, publish
// ------------------------------------------------------------------------------------------------
Accumulation look_up(PyObject* table, PyObject* key) {
  PyObject* entry = PyDict_GetItemWithError(table, key);
  if (!entry) {
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, key);
    throw Failed();
  }
  return as_accumulation(entry);
}

// clear(arena, stream, table, keys) -> status
PyObject* clear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 4);
    const Sequence keys(args[3], "keys are a sequence");
    std::vector<odc_span> spans;
    spans.reserve((size_t)keys.size());
    for (Py_ssize_t k = 0; k < keys.size(); ++k) {
      const Accumulation acc = look_up(args[2], keys[k]);
      spans.push_back({acc.offset, acc.numel * dtype_bytes(acc.code)});
    }
    odc_arena* arena = static_cast<odc_arena*>(as_pointer(args[0]));
    void* stream = as_pointer(args[1]);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = p_clear(arena, spans.data(), (uint32_t)spans.size(), stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
  });
}

// publish(arena, rank, stream, table, keys, outputs (None: in place only), out code, divisor) -> status
PyObject* publish(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 8);
    const Sequence keys(args[4], "keys are a sequence"), outs(args[5], "outputs are a sequence");
    ODC_ASSERT(outs.size() == keys.size(), "one output per key");
    std::vector<odc_publish_item> items;
    items.reserve((size_t)keys.size());
    int acc_code = -1;
    for (Py_ssize_t k = 0; k < keys.size(); ++k) {
      const Accumulation acc = look_up(args[3], keys[k]);
      acc_code = acc.code;
      items.push_back({acc.offset, acc.numel, outs[k] == Py_None ? nullptr : as_tensor(outs[k]).data_ptr()});
    }
    odc_arena* arena = static_cast<odc_arena*>(as_pointer(args[0]));
    const uint32_t rank = (uint32_t)as_u64(args[1]);
    void* stream = as_pointer(args[2]);
    const int out_code = (int)as_u64(args[6]);
    const double divisor = PyFloat_AsDouble(args[7]);
    if (PyErr_Occurred()) throw Failed();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = p_publish(arena, rank, items.data(), (uint32_t)items.size(), acc_code, out_code, (float)divisor, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
  });
}

// ------------------------------------------------------------------------------------------------
// tensors that a parameter group hands out
// ------------------------------------------------------------------------------------------------
// The GIL is not held in its scope: the allocator may wait for a thread that wants it.
class WithoutGil {
 public:
  WithoutGil() : state_(PyEval_SaveThread()) {}
  ~WithoutGil() { PyEval_RestoreThread(state_); }
  WithoutGil(const WithoutGil&) = delete;
  WithoutGil& operator=(const WithoutGil&) = delete;

 private:
  PyThreadState* state_;
};

std::vector<int64_t> as_sizes(PyObject* o) {
  const Sequence items(o, "sizes are a sequence");
  std::vector<int64_t> sizes((size_t)items.size());
  for (Py_ssize_t k = 0; k < items.size(); ++k) sizes[(size_t)k] = (int64_t)as_u64(items[k]);
  return sizes;
}

PyObject* as_list(const std::vector<at::Tensor>& tensors) {
  PyObject* list = PyList_New((Py_ssize_t)tensors.size());
  if (!list) throw Failed();
  for (size_t k = 0; k < tensors.size(); ++k) {
    PyObject* t = THPVariable_Wrap(tensors[k]);
    if (!t) {
      Py_DECREF(list);
      throw Failed();
    }
    PyList_SET_ITEM(list, (Py_ssize_t)k, t);
  }
  return list;
}

// Whatever `body` makes of tensors, in a list; what it throws becomes the exception that torch's own functions
// raise (out of memory among them).
template <class F>
PyObject* tensor_list(F body) {
  HANDLE_TH_ERRORS
  try {
    return body();
  } catch (const Failed&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// empty_list(shapes, dtype, device index) -> a new GPU tensor of each shape, memory of its own
PyObject* empty_list(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return tensor_list([&] {
    expect_args(n, 3);
    const Sequence shapes(args[0], "shapes are a sequence");
    if (!THPDtype_Check(args[1])) raise(PyExc_TypeError, "expected a torch.dtype, got %s", Py_TYPE(args[1])->tp_name);
    const auto options = at::TensorOptions()
                             .dtype(reinterpret_cast<THPDtype*>(args[1])->scalar_type)
                             .device(at::Device(at::kCUDA, (c10::DeviceIndex)as_u64(args[2])));
    std::vector<std::vector<int64_t>> sizes;
    sizes.reserve((size_t)shapes.size());
    for (Py_ssize_t k = 0; k < shapes.size(); ++k) sizes.push_back(as_sizes(shapes[k]));
    std::vector<at::Tensor> out;
    out.reserve(sizes.size());
    {
      WithoutGil nobody;
      for (const auto& size : sizes) out.push_back(at::empty(size, options));
    }
    return as_list(out);
  });
}

// strided_list(tensor, [(sizes, strides, offset), ...]) -> tensor.as_strided of each, offsets from the tensor's own
PyObject* strided_list(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return tensor_list([&] {
    expect_args(n, 2);
    const at::Tensor& t = as_tensor(args[0]);
    const Sequence views(args[1], "views are a sequence");
    std::vector<at::Tensor> out;
    out.reserve((size_t)views.size());
    for (Py_ssize_t k = 0; k < views.size(); ++k) {
      const Sequence view(views[k], "a view is a sequence");
      if (view.size() != 3) raise(PyExc_TypeError, "a view is sizes, strides and an offset");
      out.push_back(at::as_strided(t, as_sizes(view[0]), as_sizes(view[1]), t.storage_offset() + (int64_t)as_u64(view[2])));
    }
    return as_list(out);
  });
}

PyMethodDef module_methods[] = {
#define ODC_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
    ODC_METHOD(bind),
    ODC_METHOD(gather),
    ODC_METHOD(gather_slices),
    ODC_METHOD(accumulate_batch),
    ODC_METHOD(slice_layout),
    ODC_METHOD(clear),
    ODC_METHOD(empty_list),
    ODC_METHOD(strided_list),
    ODC_METHOD(publish),
#undef ODC_METHOD
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "odc_torch", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_odc_torch(void) {
  batch_type = reinterpret_cast<PyTypeObject*>(PyType_FromSpec(&batch_spec));
  slice_layout_type = reinterpret_cast<PyTypeObject*>(PyType_FromSpec(&slice_layout_spec));
  if (!batch_type || !slice_layout_type) return nullptr;
  PyObject* module = PyModule_Create(&module_def);
#define ODC_TEXT_(x) #x
#define ODC_TEXT(x) ODC_TEXT_(x)
  if (module && PyModule_AddStringConstant(module, "built_for",
                                           "ABI " ODC_TEXT(ODC_HIP_ABI_VERSION) ", torch " ODC_TORCH_VERSION
                                           ", CPython " ODC_TEXT(PY_MAJOR_VERSION) "." ODC_TEXT(PY_MINOR_VERSION)) < 0) {
    Py_DECREF(module);
    return nullptr;
  }
  return module;
}
