// The decode step's argument checks and launch in one native call.
//
// A step of the 32-layer model passes 192 weight tensors and 32 caches.  Checking them from Python (type,
// device, dtype, shape, contiguity, alignment, address, about a microsecond each) took 200 us a call, as long
// as a third of the step itself.  `step` makes the same checks on the same arguments on every call (nothing is
// remembered about a tensor) and calls the library's entry point.  It answers only for the arguments that it
// finds right: for anything else, errors included, it returns None, and the caller's own checks decide and
// word the error.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>

#include <cstdint>
#include <cstring>
#include <vector>

namespace {

struct Weight {
  at::ScalarType dtype;
  std::vector<int64_t> shape;
};
struct Spec {
  int model, hidden, kv_heads, head_dim, max_batch, max_seq, max_layers, vocab, block;
  std::vector<Weight> layer;
};
constexpr const char* kSpec = "prime_kernels_amd.step_spec";

using Decode = int (*)(void*, int, int, int, const void*, int, const void*, const void*, const void*, const void*,
                       const void*, int, const void*, const void*, void* const*, long long, long long, long long,
                       long long, long long, int, const void*, int, void*, void*, void*, void*, void*, size_t, int);
using DecodeEncoded = int (*)(void*, int, int, int, const void*, int, const void*, const void*, const void*, const void*,
                              const void*, int, const void*, const void*, void* const*, long long, long long, long long,
                              long long, long long, int, const void*, int, void*, void*, void*, void*, void*, size_t, int,
                              const void*);

// A plain tensor (no subclass: those answer for themselves in Python), or null.
const at::Tensor* plain(PyObject* o) {
  return o && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}
bool is(const at::Tensor* t, const c10::Device& dev, at::ScalarType dtype, at::IntArrayRef shape) {
  return t && t->is_cuda() && t->device() == dev && t->scalar_type() == dtype && t->sizes() == shape;
}
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

PyObject* make_spec(PyObject*, PyObject* args) {
  int model, hidden, kv_heads, head_dim, max_batch, max_seq, max_layers, vocab, block;
  PyObject* layer;
  if (!PyArg_ParseTuple(args, "iiiiiiiiiO!", &model, &hidden, &kv_heads, &head_dim, &max_batch, &max_seq, &max_layers,
                        &vocab, &block, &PyList_Type, &layer))
    return nullptr;
  auto* s = new Spec{model, hidden, kv_heads, head_dim, max_batch, max_seq, max_layers, vocab, block, {}};
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(layer); ++i) {  // (is_bf16, shape)
    int bf16;
    PyObject* shape;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(layer, i), "pO!", &bf16, &PyTuple_Type, &shape)) {
      delete s;
      return nullptr;
    }
    Weight w{bf16 ? at::kBFloat16 : at::kByte, {}};
    for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(shape); ++k) w.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, k)));
    s->layer.push_back(std::move(w));
  }
  if (PyErr_Occurred()) {
    delete s;
    return nullptr;
  }
  return PyCapsule_New(s, kSpec, [](PyObject* c) { delete static_cast<Spec*>(PyCapsule_GetPointer(c, kSpec)); });
}

// step(function, stream, spec, n_layers, input_ids, positions, seq_lens, slot_mapping, block_table, embed, final_norm,
//      layers, kv_caches, cos_sin_cache, layer_outputs, logits_out, want_ids, out, ids, scratch, scratch_bytes,
//      layer_table, kv_table, table_key, encoded_table, encoded_weights)
// -> the entry point's status; or the bytes that table_key should be (the addresses of the layers' tensors, then of
// the caches) when they are others; or None when an argument is not plainly right.
PyObject* step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 26) {
    PyErr_SetString(PyExc_TypeError, "step takes 26 arguments");
    return nullptr;
  }
  auto address = [&](int i) { return reinterpret_cast<void*>(a[i] == Py_None ? 0 : PyLong_AsUnsignedLongLong(a[i])); };
  void* fn = address(0);
  void* stream = address(1);
  const auto* s = static_cast<const Spec*>(PyCapsule_GetPointer(a[2], kSpec));
  int overflow = 0;  // a count past a long is no error here: below it is out of range
  const long nl = PyLong_AsLongAndOverflow(a[3], &overflow);
  const int want_ids = PyObject_IsTrue(a[16]);
  void *out = address(17), *ids = address(18), *scratch = address(19);
  const size_t scratch_bytes = PyLong_AsSize_t(a[20]);
  void *layer_table = address(21), *kv_table = address(22), *encoded = address(24);
  if (PyErr_Occurred() || !s || !fn) return PyErr_Occurred() ? nullptr : (PyErr_SetString(PyExc_TypeError, "no function"), nullptr);
  try {
    const at::Tensor *input_ids = plain(a[4]), *positions = plain(a[5]), *seq_lens = plain(a[6]), *slots = plain(a[7]),
                     *table = plain(a[8]), *embed = plain(a[9]), *final_norm = plain(a[10]), *cos_sin = plain(a[13]);
    if (!input_ids || !input_ids->is_cuda() || input_ids->dim() != 1 || !table || !cos_sin) Py_RETURN_NONE;
    const auto ids_type = input_ids->scalar_type();
    if (ids_type != at::kLong && ids_type != at::kInt) Py_RETURN_NONE;
    const int64_t B = input_ids->size(0);
    if (B < 1 || B > s->max_batch || nl < 1 || nl > s->max_layers) Py_RETURN_NONE;
    const c10::Device dev = input_ids->device();
    if (!is(positions, dev, at::kLong, {B}) || !is(seq_lens, dev, at::kInt, {B}) || !is(slots, dev, at::kLong, {B})) Py_RETURN_NONE;
    if (table->scalar_type() != at::kInt || table->device() != dev || table->dim() != 2 || table->size(0) < B ||
        table->stride(1) != 1 || table->size(1) < 1 || table->size(1) * s->block > s->max_seq)
      Py_RETURN_NONE;
    if (!is(embed, dev, at::kBFloat16, {s->vocab, s->hidden}) || !embed->is_contiguous()) Py_RETURN_NONE;
    if (!is(final_norm, dev, at::kBFloat16, {s->hidden})) Py_RETURN_NONE;
    if (!cos_sin->is_cuda() || cos_sin->device() != dev || cos_sin->dim() != 2 || cos_sin->size(1) != s->head_dim ||
        !cos_sin->is_contiguous() || (cos_sin->scalar_type() != at::kBFloat16 && cos_sin->scalar_type() != at::kFloat))
      Py_RETURN_NONE;
    // layers and caches: lists or tuples
    auto items = [](PyObject* o, Py_ssize_t want) -> PyObject** {
      if (PyList_CheckExact(o)) return PyList_GET_SIZE(o) == want ? reinterpret_cast<PyListObject*>(o)->ob_item : nullptr;
      if (PyTuple_CheckExact(o)) return PyTuple_GET_SIZE(o) == want ? reinterpret_cast<PyTupleObject*>(o)->ob_item : nullptr;
      return nullptr;
    };
    const Py_ssize_t per = Py_ssize_t(s->layer.size());
    PyObject** layers = items(a[11], nl);
    PyObject** caches = items(a[12], nl);
    if (!layers || !caches) Py_RETURN_NONE;
    std::vector<int64_t> key;
    key.reserve(size_t(nl) * (size_t(per) + 1));
    for (long l = 0; l < nl; ++l) {
      PyObject** layer = items(layers[l], per);
      if (!layer) Py_RETURN_NONE;
      for (Py_ssize_t k = 0; k < per; ++k) {
        const at::Tensor* t = plain(layer[k]);
        if (!is(t, dev, s->layer[k].dtype, s->layer[k].shape) || !t->is_contiguous()) Py_RETURN_NONE;
        const void* p = t->data_ptr();
        if (!aligned16(p)) Py_RETURN_NONE;
        key.push_back(reinterpret_cast<int64_t>(p));
      }
    }
    const at::Tensor* kv0 = plain(caches[0]);
    if (!kv0 || !kv0->is_cuda() || kv0->device() != dev || kv0->scalar_type() != at::kBFloat16 || kv0->dim() != 4 ||
        kv0->size(1) != s->kv_heads || kv0->size(2) != s->block || kv0->size(3) != 2 * s->head_dim || kv0->stride(3) != 1)
      Py_RETURN_NONE;
    for (long l = 0; l < nl; ++l) {
      const at::Tensor* t = plain(caches[l]);
      if (!is(t, dev, at::kBFloat16, kv0->sizes()) || t->strides() != kv0->strides()) Py_RETURN_NONE;
      key.push_back(reinterpret_cast<int64_t>(t->data_ptr()));
    }
    void *layer_outputs = nullptr, *logits = nullptr;
    if (a[14] != Py_None) {
      const at::Tensor* t = plain(a[14]);
      if (!is(t, dev, at::kBFloat16, {nl, B, s->hidden}) || !t->is_contiguous()) Py_RETURN_NONE;
      layer_outputs = t->data_ptr();
    }
    if (a[15] != Py_None) {
      const at::Tensor* t = plain(a[15]);
      if (!is(t, dev, at::kBFloat16, {B, s->vocab}) || !t->is_contiguous()) Py_RETURN_NONE;
      logits = t->data_ptr();
    }
    if (encoded) {  // the encoded weights are those of these layers
      if (!PyTuple_CheckExact(a[25]) || PyTuple_GET_SIZE(a[25]) < nl || per != 6) Py_RETURN_NONE;
      for (long l = 0; l < nl; ++l) {
        const at::Tensor* t = plain(PyTuple_GET_ITEM(a[25], l));
        if (!t || reinterpret_cast<int64_t>(t->data_ptr()) != key[size_t(l) * 6 + 4]) Py_RETURN_NONE;
      }
    }
    const size_t bytes = key.size() * sizeof(int64_t);
    if (!PyBytes_Check(a[23]) || size_t(PyBytes_GET_SIZE(a[23])) != bytes ||
        std::memcmp(PyBytes_AS_STRING(a[23]), key.data(), bytes) != 0)
      return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(key.data()), Py_ssize_t(bytes));
    const void *p_ids = input_ids->data_ptr(), *p_embed = embed->data_ptr(), *p_norm = final_norm->data_ptr(),
               *p_pos = positions->data_ptr(), *p_len = seq_lens->data_ptr(), *p_table = table->data_ptr(),
               *p_slots = slots->data_ptr(), *p_cs = cos_sin->data_ptr();
    const int i64 = ids_type == at::kLong, cs32 = cos_sin->scalar_type() == at::kFloat;
    const int bt_stride = int(table->stride(0)), max_seq = int(table->size(1)) * s->block;
    if (table->stride(0) != bt_stride) Py_RETURN_NONE;
    const long long st0 = kv0->stride(0), st1 = kv0->stride(1), st2 = kv0->stride(2);
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    if (encoded)
      rc = reinterpret_cast<DecodeEncoded>(fn)(stream, s->model, int(B), int(nl), p_ids, i64, p_embed, p_norm, p_pos, p_len,
                                               p_table, bt_stride, p_slots, layer_table, static_cast<void* const*>(kv_table), 0,
                                               s->head_dim, st0, st2, st1, s->block, p_cs, cs32, out, layer_outputs,
                                               want_ids ? ids : nullptr, logits, scratch, scratch_bytes, max_seq, encoded);
    else
      rc = reinterpret_cast<Decode>(fn)(stream, s->model, int(B), int(nl), p_ids, i64, p_embed, p_norm, p_pos, p_len, p_table,
                                        bt_stride, p_slots, layer_table, static_cast<void* const*>(kv_table), 0, s->head_dim, st0,
                                        st2, st1, s->block, p_cs, cs32, out, layer_outputs, want_ids ? ids : nullptr, logits,
                                        scratch, scratch_bytes, max_seq);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
  } catch (const std::exception&) {  // a tensor without storage, say: the caller's checks word it
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {{"make_spec", make_spec, METH_VARARGS, "A model's argument shapes, for step."},
                         {"step", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(step)), METH_FASTCALL,
                          "Check a decode step's arguments and launch it."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_step", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_step(void) { return PyModule_Create(&module); }
