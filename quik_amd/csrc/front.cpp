// Host front end of the hot calls: one Python -> C++ crossing per operation.
//
// A decode-size forward is one or two kernels of 4 .. 20 us, and the interpreter work around them (attribute and
// buffer checks of the module, two tensor allocations through the dispatcher, a ctypes call of ten arguments) took
// 17 us of host time per layer and 43 us per q/k/v group.  The same checks, allocations and library call made here
// take 5 .. 6 us (one launch included), so that a loop over layers is bound by the GPU again.
//
// Every function answers None when a call is not one it serves (another device is current, a tensor subclass,
// unusual strides, sizes or types that do not fit, a buffer or switch of the module that changed): the Python
// functions then run as they always did and raise the errors that belong to the call.
#include <Python.h>

#include <ATen/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <memory>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/quik_hip.h"

namespace {

constexpr const char *kPlanName = "quik_amd.plan";
constexpr const char *kGroupName = "quik_amd.group";

struct PyRef {  // owned reference
  PyObject *p = nullptr;
  PyRef() = default;
  explicit PyRef(PyObject *o) : p(o) { Py_XINCREF(p); }
  PyRef(PyRef &&o) noexcept : p(o.p) { o.p = nullptr; }
  PyRef(const PyRef &) = delete;
  PyRef &operator=(const PyRef &) = delete;
  PyRef &operator=(PyRef &&o) noexcept {
    std::swap(p, o.p);
    return *this;
  }
  ~PyRef() { Py_XDECREF(p); }
};

PyObject *s_buffers, *s_mid_event, *s_cuda_event, *s_cur, *s_outs, *s_fast, *s_fused, *s_workspaces, *s_split_k, *s_group_size;
PyObject *s_shared[6];  // what SharedQuantizedInput.finish drops at the end of a round

// A class keeps its version tag until one of its attributes (or of its bases') is set: methods and class-wide
// switches are as they were when the plan was made.
unsigned type_tag(PyTypeObject *t) {
#if PY_VERSION_HEX < 0x030c0000
  if (!(t->tp_flags & Py_TPFLAGS_VALID_VERSION_TAG)) return 0;
#endif
  return t->tp_version_tag;
}

// What was found under `name` in the module's _buffers: no tensor, or one whose object and storage are known weakly (a plan
// keeps no weights alive, and a tensor or block that got the address of a freed one is another), with address and version.
struct Buffer {
  PyRef name, weak;  // weak: the tensor's weak reference, or what stood in its place (None, or nothing)
  std::optional<c10::weak_intrusive_ptr<c10::StorageImpl>> storage;  // of a tensor
  const void *data = nullptr;
  uint32_t version = 0;
};

const void *data_of(const at::Tensor &t) { return t.unsafeGetTensorImpl()->data(); }
uint32_t version_of(const at::Tensor &t) { return t.unsafeGetTensorImpl()->version_counter().current_version(); }

bool snapshot(PyObject *buffers, PyObject *names, std::vector<Buffer> &out) {
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); ++i) {
    PyObject *name = PyTuple_GET_ITEM(names, i), *t = PyDict_GetItemWithError(buffers, name);
    Buffer b{PyRef(name), PyRef()};
    if (t && t != Py_None) {
      if (!THPVariable_CheckExact(t)) return false;
      const at::Tensor &v = THPVariable_Unpack(t);
      if (v.is_inference() || !v.has_storage()) return false;
      if (!(b.weak.p = PyWeakref_NewRef(t, nullptr))) return false;
      b.storage.emplace(v.storage().getWeakStorageImpl());
      b.data = v.numel() ? data_of(v) : nullptr;
      b.version = version_of(v);
    } else {
      b.weak = PyRef(t);
    }
    out.push_back(std::move(b));
  }
  return true;
}

PyObject *dict_of(PyObject *o) {
  PyObject **d = _PyObject_GetDictPtr(o);
  return d ? *d : nullptr;
}

// the module's buffers are the tensors they were: same objects, storages and addresses, not written in place since
bool unchanged(PyObject *module_dict, const std::vector<Buffer> &bufs) {
  PyObject *buffers = PyDict_GetItemWithError(module_dict, s_buffers);
  if (!buffers || !PyDict_Check(buffers)) return false;
  for (const Buffer &b : bufs) {
    PyObject *t = PyDict_GetItemWithError(buffers, b.name.p);
    if (!b.storage) {
      if (t != b.weak.p) return false;
      continue;
    }
    if (!t || t == Py_None || PyWeakref_GetObject(b.weak.p) != t) return false;
    const at::Tensor &v = THPVariable_Unpack(t);
    if (!v.has_storage() || v.storage().unsafeGetStorageImpl() != b.storage->_unsafe_get_target()) return false;
    if (version_of(v) != b.version || (v.numel() ? data_of(v) : nullptr) != b.data) return false;
  }
  return true;
}

struct Plan {
  PyTypeObject *type = nullptr;
  unsigned tag = 0;
  std::vector<Buffer> bufs;
  quik_layer row{}, tiled{};
  bool has_row = false, has_tiled = false;
  int64_t tiled_from = INT64_MAX;
  c10::DeviceIndex device = 0;
  at::ScalarType dtype = at::kHalf;
  PyRef keep, device_obj, splitk_fn;
  Plan(PyObject *k, PyObject *d, PyObject *f) : keep(k), device_obj(d), splitk_fn(f) {}
};

struct Group {
  struct Member {
    PyRef weak, key;
    PyTypeObject *type = nullptr;
    unsigned tag = 0;
    int64_t out = 0;
    std::vector<Buffer> bufs;
    Member(PyObject *w, PyObject *k) : weak(w), key(k) {}
  };
  PyRef shared_weak, fused, inner, methods;  // inner: the fused layer's plan capsule; methods: names that the front end goes past
  PyTypeObject *type = nullptr;              // of the shared object
  unsigned tag = 0;
  std::vector<Member> members;
  Group(PyObject *s, PyObject *f, PyObject *i, PyObject *m) : shared_weak(s), fused(f), inner(i), methods(m) {}
};

PyObject *fail(const char *op, int rc) {
  if (rc == QUIK_ERR_LAUNCH) return PyErr_Format(PyExc_RuntimeError, "%s: %s: %s", op, quik_status_string(rc), quik_last_hip_error());
  return PyErr_Format(PyExc_RuntimeError, "%s: %s", op, quik_status_string(rc));
}

// the current GPU; -1 where there is none
c10::DeviceIndex current_gpu() {
  c10::DeviceIndex dev = -1;
  return c10::hip::GetDevice(&dev) == hipSuccess ? dev : c10::DeviceIndex(-1);
}

void *stream_of(c10::DeviceIndex dev) { return c10::hip::getCurrentHIPStream(dev).stream(); }

at::Tensor new_empty(at::IntArrayRef size, at::ScalarType type, c10::DeviceIndex dev) {
  return at::Tensor(at::detail::empty_cuda(size, type, at::Device(at::kCUDA, dev), std::nullopt));
}

// Dispatch modes (tracing, fake tensors, counters) see the operations of the Python functions, and tensors of vmap, grad
// and functionalization levels have no memory of their own: both stay with those functions.
constexpr c10::DispatchKeySet kInterposedKeys({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                               c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                               c10::DispatchKey::BatchedNestedTensor});

// A plain contiguous tensor on the current GPU, or null.
const at::Tensor *plain(PyObject *o, c10::DeviceIndex dev) {
  if (!THPVariable_CheckExact(o) || c10::impl::TorchDispatchModeTLS::any_modes_set()) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || t.key_set().has_any(kInterposedKeys) || !t.has_storage() || !t.is_cuda() || t.get_device() != dev || t.layout() != at::kStrided || !t.is_contiguous() ||
      t.is_conj() || t.is_neg())
    return nullptr;
  return &t;
}

// The layer's forward on x through its plan: output [rows, N] in `out` (given the shape `shape`).  False: not served
// (no error set) or failed (error set).
bool layer_run(const Plan &p, PyObject *module, PyObject *xo, const at::Tensor &x, at::IntArrayRef shape, at::Tensor &out) {
  PyObject *dict = dict_of(module);
  if (!dict || Py_TYPE(module) != p.type || p.tag == 0 || type_tag(p.type) != p.tag) return false;
  const quik_layer &probe = p.has_row ? p.row : p.tiled;
  const int64_t n_in = probe.in_features;
  if (x.scalar_type() != p.dtype || x.size(-1) != n_in || x.numel() == 0 ||
      reinterpret_cast<uintptr_t>(data_of(x)) % 16 != 0)
    return false;
  const int64_t rows = x.numel() / n_in;
  const bool tiled = rows >= p.tiled_from;
  if (tiled ? !p.has_tiled : !p.has_row) return false;
  const quik_layer &l = tiled ? p.tiled : p.row;
  void *sk = nullptr;
  int64_t sk_bytes = 0;
  PyRef sk_tensor;
  const bool four_bit = l.tiled_format == QUIK_TILED_4;  // (whose GEMMs split K by a plan of their own)
  if (tiled && (four_bit ? quik_tile4_splitk_bytes(rows, l.out_features, l.num_int, l.num_fp)
                         : quik_splitk_workspace_bytes(rows, l.out_features, l.num_int, l.bits)) > 0) {
    // the stream's workspace as matmul._splitk_workspace keeps it, or that function where there is none yet
    PyObject *globals = PyFunction_GetGlobals(p.splitk_fn.p), *known = PyDict_GetItemWithError(globals, s_workspaces);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const c10::hip::HIPStream cur = c10::hip::getCurrentHIPStream(p.device);
    if (known && PyDict_GetItemWithError(globals, s_split_k) == Py_True &&
        hipStreamIsCapturing(cur.stream(), &capture) == hipSuccess && capture == hipStreamCaptureStatusNone) {
      PyRef key;
      key.p = Py_BuildValue("(iK)", static_cast<int>(p.device), reinterpret_cast<unsigned long long>(cur.stream()));
      if (!key.p) return false;
      if (PyObject *t = PyDict_GetItemWithError(known, key.p); t && THPVariable_CheckExact(t)) {
        sk = const_cast<void *>(data_of(THPVariable_Unpack(t)));
        sk_bytes = THPVariable_Unpack(t).numel();
      }
    }
    if (!sk) {
      PyObject *r = PyObject_CallFunction(p.splitk_fn.p, "OLLLiL", p.device_obj.p, static_cast<long long>(rows),
                                          static_cast<long long>(l.out_features), static_cast<long long>(l.num_int),
                                          static_cast<int>(l.bits), static_cast<long long>(four_bit ? l.num_fp : -1));
      if (!r) return false;
      sk_tensor.p = r;
      PyObject *t = PyTuple_GET_ITEM(r, 0);
      if (t != Py_None) {
        sk = const_cast<void *>(data_of(THPVariable_Unpack(t)));
        sk_bytes = PyLong_AsLongLong(PyTuple_GET_ITEM(r, 1));
      }
    }
  }
  // (no Python code runs from here to the launch: what the buffers are now is what the kernels read)
  if (!unchanged(dict, p.bufs)) return false;
  try {
    const int64_t nbytes = quik_layer_workspace_bytes(&l, rows);
    const c10::DataPtr ws = c10::hip::HIPCachingAllocator::get()->allocate(static_cast<size_t>(nbytes));
    out = new_empty(shape, p.dtype, p.device);
    void *mid = nullptr;  // profiling hook of the module, taken once nothing sends the call back to the Python function
    const PyRef ev(PyDict_GetItemWithError(dict, s_mid_event));
    if (ev.p && ev.p != Py_None) {
      PyRef raw;
      if (!(raw.p = PyObject_GetAttr(ev.p, s_cuda_event))) return false;
      mid = PyLong_AsVoidPtr(raw.p);
      if (PyErr_Occurred() || PyDict_SetItem(dict, s_mid_event, Py_None) < 0) return false;
    }
    const int rc = quik_layer_forward(&l, data_of(x), rows, ws.get(), nbytes, sk, sk_bytes, const_cast<void *>(data_of(out)), mid,
                                      stream_of(p.device));
    if (rc != QUIK_OK) {
      fail("MixedQLinear.forward", rc);
      return false;
    }
  } catch (const c10::OutOfMemoryError &) {
    return false;  // (the Python path repeats the allocation and raises torch's own error)
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return false;
  }
  return true;
}

PyObject *none_or_error() {
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// C++ exceptions end here: out of memory goes back to the Python path, which raises torch's own error
template <typename F>
PyObject *guarded(F &&f) {
  try {
    return f();
  } catch (const c10::OutOfMemoryError &) {
    Py_RETURN_NONE;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// forward(plan, module, x) -> Tensor [.., N] or None
PyObject *forward(PyObject *const *args, Py_ssize_t n) {
  if (n != 3) return PyErr_Format(PyExc_TypeError, "forward takes 3 arguments");
  const Plan *p = static_cast<const Plan *>(PyCapsule_GetPointer(args[0], kPlanName));
  if (!p) return nullptr;
  if (current_gpu() != p->device) Py_RETURN_NONE;
  const at::Tensor *x = plain(args[2], p->device);
  if (!x || (x->dim() != 2 && x->dim() != 3)) Py_RETURN_NONE;
  const int64_t N = (p->has_row ? p->row : p->tiled).out_features;
  const int64_t shape[3] = {x->dim() == 3 ? x->size(0) : 1, x->size(x->dim() - 2), N};
  at::Tensor out;
  if (!layer_run(*p, args[1], args[2], *x, at::IntArrayRef(shape, 3), out)) return none_or_error();
  return THPVariable_Wrap(std::move(out));
}

PyObject *py_forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  return guarded([&] { return forward(args, n); });
}

// columns [at, at + n) of rows that are `stride` elements apart, as [lead0, lead1, n]; `at`: in elements from the storage's start
at::Tensor columns(const at::Tensor &t, int64_t lead0, int64_t lead1, int64_t stride, int64_t at, int64_t n) {
  const int64_t shape[3] = {lead0, lead1, n}, strides[3] = {lead1 * stride, stride, 1};
  return t.as_strided(at::IntArrayRef(shape, 3), at::IntArrayRef(strides, 3), at);
}

// group_forward(group, index, module, x) -> member `index`'s columns [.., N_index] or None
PyObject *group_forward(PyObject *const *args, Py_ssize_t n) {
  if (n != 4) return PyErr_Format(PyExc_TypeError, "group_forward takes 4 arguments");
  const Group *g = static_cast<const Group *>(PyCapsule_GetPointer(args[0], kGroupName));
  if (!g) return nullptr;
  const Plan *p = static_cast<const Plan *>(PyCapsule_GetPointer(g->inner.p, kPlanName));
  if (!p) return nullptr;
  const size_t index = PyLong_AsSize_t(args[1]);
  if (index >= g->members.size()) return none_or_error();
  PyObject *shared = PyWeakref_GetObject(g->shared_weak.p);
  PyObject *sd = shared && shared != Py_None ? dict_of(shared) : nullptr;
  if (!sd || PyDict_GetItemWithError(sd, s_fast) != args[0] || PyDict_GetItemWithError(sd, s_fused) != g->fused.p)
    Py_RETURN_NONE;
  // the shared object is of the class it was, has no methods of its own, and the group is as large as its members
  if (Py_TYPE(shared) != g->type || g->tag == 0 || type_tag(g->type) != g->tag) Py_RETURN_NONE;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(g->methods.p); ++i)
    if (PyDict_GetItemWithError(sd, PyTuple_GET_ITEM(g->methods.p, i))) Py_RETURN_NONE;
  PyObject *size = PyDict_GetItemWithError(sd, s_group_size);
  if (!size || !PyLong_Check(size) || PyLong_AsSize_t(size) != g->members.size()) return none_or_error();
  if (current_gpu() != p->device) Py_RETURN_NONE;
  const at::Tensor *x = plain(args[3], p->device);
  if (!x || (x->dim() != 2 && x->dim() != 3)) Py_RETURN_NONE;
  PyObject *cur = PyDict_GetItemWithError(sd, s_cur);
  if (!cur || !PyLong_Check(cur)) Py_RETURN_NONE;
  const long at_elem = PyLong_AsLong(cur);
  const int64_t lead0 = x->dim() == 3 ? x->size(0) : 1, lead1 = x->size(x->dim() - 2);
  if (at_elem == 0) {  // first member of a round: one quantize and one GEMM for all of them
    for (const Group::Member &m : g->members) {
      PyObject *mod = PyWeakref_GetObject(m.weak.p);
      if (!mod || mod == Py_None || Py_TYPE(mod) != m.type || m.tag == 0 || type_tag(m.type) != m.tag) Py_RETURN_NONE;
      PyObject *d = dict_of(mod);
      if (!d || !unchanged(d, m.bufs)) Py_RETURN_NONE;
    }
    const int64_t total = (p->has_row ? p->row : p->tiled).out_features, shape[3] = {lead0, lead1, total};
    at::Tensor whole;
    if (!layer_run(*p, g->fused.p, args[3], *x, at::IntArrayRef(shape, 3), whole)) return none_or_error();
    PyRef outs;
    outs.p = PyDict_New();
    if (!outs.p) return nullptr;
    int64_t lo = 0;
    for (const Group::Member &m : g->members) {  // (in the shape the members are called for: nothing is left to do then)
      PyRef v;
      v.p = THPVariable_Wrap(columns(whole, lead0, lead1, total, lo, m.out));
      if (!v.p || PyDict_SetItem(outs.p, m.key.p, v.p) < 0) return nullptr;
      lo += m.out;
    }
    if (PyDict_SetItem(sd, s_outs, outs.p) < 0) return nullptr;
  }
  PyObject *outs = PyDict_GetItemWithError(sd, s_outs);
  if (!outs || !PyDict_Check(outs)) return none_or_error();
  PyObject *mine = PyDict_GetItemWithError(outs, g->members[index].key.p);
  if (!mine || !THPVariable_CheckExact(mine)) return none_or_error();
  PyRef r;
  {
    const at::Tensor &t = THPVariable_Unpack(mine);
    const int64_t dim = t.dim();
    if (dim == 3 && t.size(0) == lead0 && t.size(1) == lead1) {
      r = PyRef(mine);
    } else {  // (of a round begun by the Python function, or with other leading sizes)
      if ((dim == 3 ? t.size(0) * t.size(1) : t.size(0)) != lead0 * lead1) Py_RETURN_NONE;
      r.p = THPVariable_Wrap(columns(t, lead0, lead1, t.stride(dim - 2), t.storage_offset(), t.size(dim - 1)));
      if (!r.p) return nullptr;
    }
  }
  // SharedQuantizedInput.finish (the class's own: see the plan's methods)
  PyRef next;
  const bool last = at_elem + 1 == static_cast<long>(g->members.size());
  next.p = PyLong_FromLong(last ? 0 : at_elem + 1);
  if (!next.p) return nullptr;
  if (last)
    for (PyObject *name : s_shared)
      if (PyDict_SetItem(sd, name, Py_None) < 0) return nullptr;
  if (PyDict_SetItem(sd, s_cur, next.p) < 0) return nullptr;
  return std::exchange(r.p, nullptr);
}

PyObject *py_group_forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  return guarded([&] { return group_forward(args, n); });
}

// plan(module, names, row_desc, tiled_desc, tiled_from, device_index, is_bf16, device, splitk_fn, keep)
PyObject *plan(PyObject *args) {
  PyObject *module, *names, *row, *tiled, *device, *fn, *keep;
  long long from;
  int dev, bf16;
  if (!PyArg_ParseTuple(args, "OO!OOLipOOO", &module, &PyTuple_Type, &names, &row, &tiled, &from, &dev, &bf16, &device, &fn,
                        &keep))
    return nullptr;
  auto p = std::make_unique<Plan>(keep, device, fn);
  PyObject *d = dict_of(module), *buffers = d ? PyDict_GetItemWithError(d, s_buffers) : nullptr;
  if (!buffers || !snapshot(buffers, names, p->bufs)) return none_or_error();
  auto take = [](PyObject *b, quik_layer &l, bool &has) {
    has = PyBytes_Check(b) && PyBytes_GET_SIZE(b) == static_cast<Py_ssize_t>(sizeof(quik_layer));
    if (has) std::memcpy(&l, PyBytes_AS_STRING(b), sizeof(quik_layer));
  };
  take(row, p->row, p->has_row);
  take(tiled, p->tiled, p->has_tiled);
  if (!p->has_row && !p->has_tiled) Py_RETURN_NONE;
  p->type = Py_TYPE(module);
  p->tag = type_tag(p->type);
  p->tiled_from = from;
  p->device = static_cast<c10::DeviceIndex>(dev);
  p->dtype = bf16 ? at::kBFloat16 : at::kHalf;
  return PyCapsule_New(p.release(), kPlanName,
                       [](PyObject *c) { delete static_cast<Plan *>(PyCapsule_GetPointer(c, kPlanName)); });
}

PyObject *py_plan(PyObject *, PyObject *args) {
  return guarded([&] { return plan(args); });
}

// group(shared_weakref, fused_module, fused_plan, method_names, ((weakref, key, out_features, names), ...))
PyObject *group(PyObject *args) {
  PyObject *shared, *fused, *inner, *methods, *members;
  if (!PyArg_ParseTuple(args, "OOOO!O!", &shared, &fused, &inner, &PyTuple_Type, &methods, &PyTuple_Type, &members)) return nullptr;
  PyObject *obj = PyCapsule_IsValid(inner, kPlanName) ? PyWeakref_GetObject(shared) : Py_None;
  if (!obj) return nullptr;
  if (obj == Py_None) Py_RETURN_NONE;
  auto g = std::make_unique<Group>(shared, fused, inner, methods);
  g->type = Py_TYPE(obj);
  g->tag = type_tag(g->type);
  g->members.reserve(static_cast<size_t>(PyTuple_GET_SIZE(members)));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(members); ++i) {
    PyObject *weak, *key, *names;
    long long out;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(members, i), "OOLO!", &weak, &key, &out, &PyTuple_Type, &names)) return nullptr;
    PyObject *mod = PyWeakref_GetObject(weak);
    if (!mod) return nullptr;
    if (mod == Py_None) Py_RETURN_NONE;
    Group::Member m(weak, key);
    m.type = Py_TYPE(mod);
    m.tag = type_tag(m.type);
    m.out = out;
    PyObject *d = dict_of(mod), *buffers = d ? PyDict_GetItemWithError(d, s_buffers) : nullptr;
    if (!buffers || !snapshot(buffers, names, m.bufs)) return none_or_error();
    g->members.push_back(std::move(m));
  }
  return PyCapsule_New(g.release(), kGroupName,
                       [](PyObject *c) { delete static_cast<Group *>(PyCapsule_GetPointer(c, kGroupName)); });
}

PyObject *py_group(PyObject *, PyObject *args) {
  return guarded([&] { return group(args); });
}

// ---------------------------------------------------------------------------------------------- stand-alone operations
const void *ptr(const at::Tensor &t) { return t.numel() ? data_of(t) : nullptr; }
void *out_ptr(const at::Tensor &t) { return const_cast<void *>(t.numel() ? data_of(t) : nullptr); }

PyObject *triple(at::Tensor a, at::Tensor b, at::Tensor c) {
  PyObject *t = PyTuple_New(3);
  if (!t) return nullptr;
  at::Tensor v[3] = {std::move(a), std::move(b), std::move(c)};
  for (int i = 0; i < 3; ++i) {
    PyObject *o = THPVariable_Wrap(std::move(v[i]));
    if (!o) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i, o);
  }
  return t;
}

int dtype_of(const at::Tensor &t) { return t.scalar_type() == at::kHalf ? QUIK_F16 : t.scalar_type() == at::kBFloat16 ? QUIK_BF16 : -1; }

// quantize(src, int_indices, fp_indices, bits) -> (dst, meta, fp_x) or None
PyObject *py_quantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 4) Py_RETURN_NONE;
  const c10::DeviceIndex dev = current_gpu();
  const at::Tensor *src = plain(args[0], dev), *ii = plain(args[1], dev), *fi = plain(args[2], dev);
  if (!src || !ii || !fi || !PyLong_Check(args[3])) Py_RETURN_NONE;
  const long bits = PyLong_AsLong(args[3]);
  const int dt = dtype_of(*src);
  if ((bits != 4 && bits != 8) || dt < 0 || src->dim() != 2 || ii->scalar_type() != at::kLong || fi->scalar_type() != at::kLong)
    return none_or_error();
  const int64_t rows = src->size(0), cols = src->size(1), num_int = ii->numel(), num_fp = fi->numel();
  if (num_int + num_fp != cols || num_int % 2 != 0 || num_int == 0 || rows == 0) Py_RETURN_NONE;
  return guarded([&]() -> PyObject * {
    void *st = stream_of(dev);
    const c10::DataPtr cm = c10::hip::HIPCachingAllocator::get()->allocate(static_cast<size_t>(quik_colmap_bytes(cols, num_int, num_fp)));
    at::Tensor dst = bits == 4 ? new_empty({rows, num_int / 2}, at::kByte, dev) : new_empty({rows, num_int}, at::kChar, dev);
    at::Tensor meta = new_empty({2 * rows}, src->scalar_type(), dev), fp_x = new_empty({rows, num_fp}, src->scalar_type(), dev);
    const int rc = quik_asym_quantize_indexed(ptr(*src), dt, rows, cols, static_cast<const int64_t *>(ptr(*ii)), num_int,
                                              static_cast<const int64_t *>(ptr(*fi)), num_fp, static_cast<int>(bits), cm.get(),
                                              out_ptr(dst), out_ptr(meta), out_ptr(fp_x), st);
    if (rc != QUIK_OK) return fail("quantize", rc);
    return triple(std::move(dst), std::move(meta), std::move(fp_x));
  });
}

// matmul(A, B, bits) -> C int32 or None
PyObject *py_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3) Py_RETURN_NONE;
  const c10::DeviceIndex dev = current_gpu();
  const at::Tensor *A = plain(args[0], dev), *B = plain(args[1], dev);
  const long bits = PyLong_AsLong(args[2]);
  const at::ScalarType want = bits == 4 ? at::kByte : at::kChar;
  if (!A || !B || A->scalar_type() != want || B->scalar_type() != want || A->dim() != 2 || B->dim() != 2 ||
      A->size(1) != B->size(1) || A->numel() == 0 || B->numel() == 0)
    return none_or_error();
  return guarded([&]() -> PyObject * {
    const int64_t M = A->size(0), N = B->size(0), K = A->size(1) * (bits == 4 ? 2 : 1);
    at::Tensor C = new_empty({M, N}, at::kInt, dev);
    int rc = bits == 4 ? quik_int4_matmul(static_cast<const uint8_t *>(ptr(*A)), static_cast<const uint8_t *>(ptr(*B)),
                                          static_cast<int32_t *>(out_ptr(C)), M, N, K, stream_of(dev))
                       : quik_int8_matmul(static_cast<const int8_t *>(ptr(*A)), static_cast<const int8_t *>(ptr(*B)),
                                          static_cast<int32_t *>(out_ptr(C)), M, N, K, stream_of(dev));
    if (rc != QUIK_OK) return fail(bits == 4 ? "int4Matmul" : "int8Matmul", rc);
    return THPVariable_Wrap(std::move(C));
  });
}

// dequantize(x, meta, scale_col, wReduced, y, bits) -> out or None
PyObject *py_dequantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 6) Py_RETURN_NONE;
  const c10::DeviceIndex dev = current_gpu();
  const at::Tensor *t[5];
  for (int i = 0; i < 5; ++i)
    if (!(t[i] = plain(args[i], dev))) Py_RETURN_NONE;
  if (!PyLong_Check(args[5])) Py_RETURN_NONE;
  const long bits = PyLong_AsLong(args[5]);
  const at::Tensor &x = *t[0], &meta = *t[1], &sc = *t[2], &wr = *t[3], &y = *t[4];
  const int dt = dtype_of(y);
  if ((bits != 4 && bits != 8) || dt < 0 || x.scalar_type() != at::kInt || x.dim() != 2 || x.numel() == 0 ||
      y.numel() != x.numel() || meta.dim() < 1 || sc.dim() < 1 || wr.dim() < 2)
    return none_or_error();
  const int64_t rows = x.size(0), cols = x.size(1);
  if (meta.size(0) != 2 * rows || meta.numel() != 2 * rows || sc.size(0) != cols || sc.numel() != cols || wr.size(1) != cols ||
      wr.numel() != cols || meta.scalar_type() != y.scalar_type() || sc.scalar_type() != y.scalar_type() ||
      wr.scalar_type() != y.scalar_type())
    Py_RETURN_NONE;
  return guarded([&]() -> PyObject * {
    at::Tensor out = new_empty(y.sizes(), y.scalar_type(), dev);
    const int rc = quik_asym_dequantize(static_cast<const int32_t *>(ptr(x)), ptr(meta), ptr(sc), ptr(wr), ptr(y), dt, rows, cols,
                                        static_cast<int>(bits), out_ptr(out), stream_of(dev));
    if (rc != QUIK_OK) return fail("dequantize", rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// fused_dequantize(A, B, scale_row, scale_col, shift_value, zero_row, w_reduced, y, bits, product) -> out or None; zero_row and
// w_reduced None: the symmetric form.  product(A, B): makes the int32 matrix of a call in two launches (some of at most 32
// rows); called once the call is known to fit.
PyObject *py_fused_dequantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 10) Py_RETURN_NONE;
  const c10::DeviceIndex dev = current_gpu();
  const bool sym = args[5] == Py_None;
  const at::Tensor *A = plain(args[0], dev), *B = plain(args[1], dev), *sr = plain(args[2], dev), *sc = plain(args[3], dev),
                   *y = plain(args[7], dev), *zr = nullptr, *wr = nullptr;
  if (!A || !B || !sr || !sc || !y) Py_RETURN_NONE;
  if (!sym && (!(zr = plain(args[5], dev)) || !(wr = plain(args[6], dev)))) Py_RETURN_NONE;
  const double shift = sym ? 0.0 : PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const long bits = PyLong_AsLong(args[8]);
  const at::ScalarType want = bits == 4 ? at::kByte : at::kChar;
  if (A->scalar_type() != want || B->scalar_type() != want || A->dim() != 2 || B->dim() != 2 || A->size(1) != B->size(1))
    Py_RETURN_NONE;
  const int64_t M = A->size(0), N = B->size(0), K = A->size(1) * (bits == 4 ? 2 : 1);
  auto half = [](const at::Tensor *t, int64_t count) { return t->scalar_type() == at::kHalf && t->numel() == count; };
  if (M * N == 0 || K == 0 || !half(sr, M) || !half(sc, N) || !half(y, M * N) || (!sym && (!half(zr, M) || !half(wr, N))))
    Py_RETURN_NONE;
  PyRef product;
  int32_t *acc = nullptr;
  if (quik_fused_dequantize_acc_bytes(M, N, K, static_cast<int>(bits)) > 0) {
    product.p = PyObject_CallFunctionObjArgs(args[9], args[0], args[1], nullptr);
    if (!product.p) return nullptr;
    const at::Tensor *t = plain(product.p, dev);
    if (!t || t->scalar_type() != at::kInt || t->numel() != M * N) Py_RETURN_NONE;
    acc = static_cast<int32_t *>(out_ptr(*t));
  }
  return guarded([&]() -> PyObject * {
    at::Tensor out = new_empty({M, N}, at::kHalf, dev);
    const int rc = sym ? quik_sym_fused_dequantize(ptr(*A), ptr(*B), ptr(*sr), ptr(*sc), ptr(*y), M, N, K, static_cast<int>(bits),
                                                   acc, out_ptr(out), stream_of(dev))
                       : quik_asym_fused_dequantize(ptr(*A), ptr(*B), ptr(*sr), ptr(*sc), static_cast<float>(shift), ptr(*zr),
                                                    ptr(*wr), ptr(*y), M, N, K, static_cast<int>(bits), acc, out_ptr(out),
                                                    stream_of(dev));
    if (rc != QUIK_OK) return fail(bits == 4 ? "int4FusedDequantize" : "int8FusedDequantize", rc);
    return THPVariable_Wrap(std::move(out));
  });
}

PyMethodDef kMethods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_forward)), METH_FASTCALL, nullptr},
    {"group_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_group_forward)), METH_FASTCALL, nullptr},
    {"plan", py_plan, METH_VARARGS, nullptr},
    {"group", py_group, METH_VARARGS, nullptr},
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_quantize)), METH_FASTCALL, nullptr},
    {"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_matmul)), METH_FASTCALL, nullptr},
    {"dequantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_dequantize)), METH_FASTCALL, nullptr},
    {"fused_dequantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_fused_dequantize)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_front", "Host front end of quik_amd's hot calls.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front() {
  s_buffers = PyUnicode_InternFromString("_buffers");
  s_mid_event = PyUnicode_InternFromString("mid_event");
  s_cuda_event = PyUnicode_InternFromString("cuda_event");
  s_cur = PyUnicode_InternFromString("cur_group_elem");
  s_outs = PyUnicode_InternFromString("_outs");
  s_fast = PyUnicode_InternFromString("_fast");
  s_fused = PyUnicode_InternFromString("_fused");
  const char *shared[6] = {"qint_x", "qscale_x", "meta", "fp_x", "x6", "_outs"};
  for (int i = 0; i < 6; ++i) s_shared[i] = PyUnicode_InternFromString(shared[i]);
  s_workspaces = PyUnicode_InternFromString("_splitk_workspaces");
  s_group_size = PyUnicode_InternFromString("group_size");
  s_split_k = PyUnicode_InternFromString("split_k");
  PyObject *m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "built_for", QUIK_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
