// A step of the attention types with a plain cache (_sink_window.py): what lies between the layer's projections and the native call,
// infllm_window_forward.  Such a step is bound by its host: checks, views, two allocations and the argument block were some eighty
// calls into Python's and torch's objects, 15 us beside a launch of 8 to 18.  Here they are reads of the same fields.
//
// Everything out of the ordinary - the first call of a cache, other widths, rows to be copied or aligned, buffers that are full, words
// that are missing - is handed back (None) and takes the general way in _sink_window.py, which also makes the errors.
//
// The buffers of a cache that still holds every token, and the words that a step counts in, hang on the cache's storage.  What this
// file does to either it does under the interpreter's lock and without running Python code, so that threads see it as one operation.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Storage.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>

#include "../../include/infllm_hip.h"

namespace {

PyObject *room_name, *words_name;
PyObject *forward_object = nullptr;                    // infllm_window_forward as ctypes has it, and its address
int (*forward_address)(const infllm_window_args *, void *) = nullptr;

// a new reference to the attributes of the storage's one Python object
PyObject *attributes(const at::Tensor &t) {
    PyObject *storage = THPStorage_Wrap(t.storage());
    if (!storage) throw python_error();
    PyObject *dict = PyObject_GenericGetDict(storage, nullptr);
    Py_DECREF(storage);
    if (!dict) throw python_error();
    return dict;
}

// How far the buffers [B, Hkv, capacity, dim] of a cache are filled: the first `used` rows are the newest cache in them.  It keeps
// numbers only (a tensor here would keep the storage alive).  A call on another stream than the buffers' own takes new ones: what it
// returns has to be memory of ITS stream, which the allocator gives out again in that stream's order once the caller drops it.
struct Room {
    const void *k, *v;
    int64_t shape[4], strides[4], used, stream;
};
const char *const kRoom = "infllm_amd.room";

void free_room(PyObject *capsule) { delete (Room *)PyCapsule_GetPointer(capsule, kRoom); }

bool four(const at::Tensor &t, const int64_t *shape, const int64_t *strides) {
    if (t.dim() != 4) return false;
    for (int i = 0; i < 4; ++i)
        if (t.stride(i) != strides[i] || (i != 2 && t.size(i) != shape[i])) return false;
    return true;
}

// Whether a call on `stream` may write the n rows behind the given cache; then they are its.
bool claim(const at::Tensor &k, const at::Tensor &v, int64_t n, int64_t stream) {
    PyObject *dict = attributes(k), *capsule = PyDict_GetItemWithError(dict, room_name);
    Room *room = capsule ? (Room *)PyCapsule_GetPointer(capsule, kRoom) : nullptr;
    const bool mine = room && room->stream == stream && k.data_ptr() == room->k && v.data_ptr() == room->v && four(k, room->shape, room->strides) &&
                      four(v, room->shape, room->strides) && v.size(2) == k.size(2) && room->used == k.size(2) && room->used + n <= room->shape[2];
    if (mine) room->used += n;
    Py_DECREF(dict);                                   // (the storage has it)
    if (PyErr_Occurred()) throw python_error();
    return mine;
}

std::pair<at::Tensor, at::Tensor> grown(const at::Tensor &k, const at::Tensor &v, int64_t n) {
    const int64_t shape[4] = {k.size(0), k.size(1), k.size(2) + n, k.size(3)};
    return {k.as_strided(shape, k.strides(), k.storage_offset()), v.as_strided(shape, v.strides(), v.storage_offset())};
}

const at::Tensor *tensor(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

// projected rows [batch, 1, heads * dim] that a kernel can read as they lie
bool rows_of(const at::Tensor *t, const at::Tensor &like, int64_t batch, int64_t width) {
    return t && t->dim() == 3 && t->size(0) == batch && t->size(1) == 1 && t->size(2) == width && t->scalar_type() == at::kBFloat16 &&
           t->device() == like.device() && t->layout() == at::kStrided && t->stride(2) == 1 && ((t->stride(0) | t->stride(1)) & 7) == 0 &&
           ((uintptr_t)t->data_ptr() & 15) == 0;
}

// cached rows [batch, heads, rows, dim]
bool cached_of(const at::Tensor *t, const at::Tensor &like, int64_t batch, int64_t heads, int64_t rows, int64_t dim) {
    return t && t->dim() == 4 && t->size(0) == batch && t->size(1) == heads && t->size(2) == rows && t->size(3) == dim &&
           t->scalar_type() == at::kBFloat16 && t->device() == like.device() && t->layout() == at::kStrided && t->stride(3) == 1 && t->stride(2) == dim &&
           ((t->stride(0) | t->stride(1)) & 7) == 0 && ((uintptr_t)t->data_ptr() & 15) == 0;
}

// make_room(both [2, B, Hkv, capacity, dim], rows in use, stream)
PyObject *py_make_room(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *both = n == 3 ? tensor(args[0]) : nullptr;
    if (!both || both->dim() != 5 || both->size(0) != 2) {
        PyErr_SetString(PyExc_TypeError, "make_room(both, used, stream)");
        return nullptr;
    }
    Room *room = new Room{};
    room->k = both->data_ptr();
    room->v = (const char *)both->data_ptr() + both->stride(0) * both->element_size();
    for (int i = 0; i < 4; ++i) room->shape[i] = both->size(i + 1), room->strides[i] = both->stride(i + 1);
    room->used = PyLong_AsLongLong(args[1]);
    room->stream = PyLong_AsLongLong(args[2]);
    PyObject *capsule = PyErr_Occurred() ? nullptr : PyCapsule_New(room, kRoom, free_room);
    if (!capsule) {
        delete room;
        return nullptr;
    }
    PyObject *dict = attributes(*both);
    const int bad = PyDict_SetItem(dict, room_name, capsule);
    Py_DECREF(dict);
    Py_DECREF(capsule);
    if (bad) return nullptr;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// claim(keys, values, new rows, stream): (keys, values) with the rows behind them, or None where the call needs buffers of its own
PyObject *py_claim(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "claim(keys, values, rows, stream)");
        return nullptr;
    }
    const at::Tensor &k = THPVariable_Unpack(args[0]), &v = THPVariable_Unpack(args[1]);
    const int64_t rows = PyLong_AsLongLong(args[2]), stream = PyLong_AsLongLong(args[3]);
    if (PyErr_Occurred()) return nullptr;
    if (!claim(k, v, rows, stream)) Py_RETURN_NONE;
    auto kv = grown(k, v, rows);
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(kv.first)), THPVariable_Wrap(std::move(kv.second)));
    END_HANDLE_TH_ERRORS
}

// bind(infllm_window_forward, its address, ABI version, size of its argument block, torch's version): what step calls by itself when it is
// given this object.  The block is filled here as this file was compiled with it, and torch's objects are read as that torch lays them out:
// a module of another build is refused.
PyObject *py_bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "bind(function, address, ABI version, size of the argument block, torch's version)");
        return nullptr;
    }
    void *address = PyLong_AsVoidPtr(args[1]);
    const long long version = PyLong_AsLongLong(args[2]), bytes = PyLong_AsLongLong(args[3]);
    const char *torch_version = PyErr_Occurred() ? nullptr : PyUnicode_AsUTF8(args[4]);
    if (!torch_version) return nullptr;
    if (version != INFLLM_ABI_VERSION || bytes != (long long)sizeof(infllm_window_args) || std::strcmp(torch_version, INFLLM_TORCH_VERSION) != 0)
        return PyErr_Format(PyExc_ImportError, "built for ABI version %d with blocks of %zu bytes and torch %s, not for %lld, %lld and %s", INFLLM_ABI_VERSION,
                            sizeof(infllm_window_args), INFLLM_TORCH_VERSION, version, bytes, torch_version);
    Py_INCREF(args[0]);
    Py_XDECREF(forward_object);
    forward_object = args[0];
    forward_address = (int (*)(const infllm_window_args *, void *))address;
    Py_RETURN_NONE;
}

// step(kind, n_local, n_init, q, k, v, past (keys, values, tokens seen, un-rotated sinks), inv_freq, distance_scale, batch, heads, kv heads,
//      dim, scratch of a step, stream, infllm_window_forward, function that gives the address of words):
// (output rows, new past); None where the step is not a plain one; the status of a native call that failed.
PyObject *py_step(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 17) {
        PyErr_SetString(PyExc_TypeError, "step: 17 arguments");
        return nullptr;
    }
    int64_t num[9];
    const int places[9] = {0, 1, 2, 9, 10, 11, 12, 13, 14};
    for (int i = 0; i < 9; ++i) num[i] = PyLong_AsLongLong(args[places[i]]);
    const double distance_scale = PyFloat_AsDouble(args[8]);
    if (PyErr_Occurred()) return nullptr;
    const int64_t kind = num[0], n_local = num[1], n_init = num[2], batch = num[3], heads = num[4], kv_heads = num[5], dim = num[6], step_bytes = num[7],
                  stream = num[8];
    PyObject *past = args[6];
    if (!PyTuple_CheckExact(past) || PyTuple_GET_SIZE(past) != 4 || !PyLong_CheckExact(PyTuple_GET_ITEM(past, 2))) Py_RETURN_NONE;
    const at::Tensor *q = tensor(args[3]), *k = tensor(args[4]), *v = tensor(args[5]), *old_k = tensor(PyTuple_GET_ITEM(past, 0)),
                     *old_v = tensor(PyTuple_GET_ITEM(past, 1)), *freq = tensor(args[7]), *raw = nullptr;
    PyObject *raw_object = PyTuple_GET_ITEM(past, 3);
    if (raw_object != Py_None && !(raw = tensor(raw_object))) Py_RETURN_NONE;
    if (!q || !old_k || old_k->dim() != 4) Py_RETURN_NONE;
    const int64_t rows_old = old_k->size(2), seen = PyLong_AsLongLong(PyTuple_GET_ITEM(past, 2)), rows_all = rows_old + 1, len_k = seen + 1;
    if (PyErr_Occurred()) return nullptr;
    if (n_init < 0 || n_init > INT32_MAX || rows_old < 1 || rows_old >= INT32_MAX || !rows_of(q, *q, batch, heads * dim) ||
        !rows_of(k, *q, batch, kv_heads * dim) || !rows_of(v, *q, batch, kv_heads * dim) ||
        !cached_of(old_k, *q, batch, kv_heads, rows_old, dim) || !cached_of(old_v, *q, batch, kv_heads, rows_old, dim))
        Py_RETURN_NONE;
    if (!freq || freq->device() != q->device() || freq->scalar_type() != at::kFloat || freq->numel() != dim / 2 || !freq->is_contiguous()) Py_RETURN_NONE;
    const int64_t raw_rows = raw ? (raw->dim() == 4 ? raw->size(2) : -1) : 0;
    if (raw && (!cached_of(raw, *q, batch, kv_heads, raw_rows, dim) || !raw->is_contiguous())) Py_RETURN_NONE;
    if (kind == 2 && raw_rows < n_init && seen == raw_rows) Py_RETURN_NONE;             // (sinks to be copied)
    const bool cut = kind && len_k > n_local + n_init && rows_all > n_local + n_init;

    // ---- the words, and the scratch behind them (see _take_words): (tensor, address, words, stream, address of the scratch, its bytes)
    PyObject *dict = attributes(*old_k), *words = PyDict_GetItemWithError(dict, words_name);
    int64_t held[4] = {};                               // (the last four)
    bool fits = words && PyTuple_CheckExact(words) && PyTuple_GET_SIZE(words) == 6;
    for (int i = 0; fits && i < 4; ++i) held[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(words, i + 2));
    fits = fits && !PyErr_Occurred() && held[0] >= batch * heads && held[1] == stream && held[3] >= step_bytes;
    if (fits && !cut) fits = claim(*old_k, *old_v, 1, stream);
    if (!fits) {
        Py_DECREF(dict);
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    Py_INCREF(words);
    const int bad = PyDict_DelItem(dict, words_name);
    Py_DECREF(dict);
    struct Held {
        PyObject *o;
        ~Held() { Py_DECREF(o); }
    } words_held{words};
    if (bad) return nullptr;
    // (behind this point other threads may run: views and tensors are made by torch's dispatcher, which can be a Python mode's)
    PyObject *address = PyObject_CallFunctionObjArgs(args[16], words, nullptr);
    if (!address) return nullptr;
    void *const ticket = PyLong_AsVoidPtr(address);
    Py_DECREF(address);
    if (PyErr_Occurred()) return nullptr;

    const auto options = at::TensorOptions().dtype(at::kBFloat16).device(q->device());
    const int64_t rows_new = cut ? n_init + n_local : rows_all;
    at::Tensor new_k, new_v;
    if (!cut) std::tie(new_k, new_v) = grown(*old_k, *old_v, 1);
    else {
        const at::Tensor cache = at::empty({2, batch, kv_heads, rows_new, dim}, options);
        new_k = cache.select(0, 0);
        new_v = cache.select(0, 1);
    }
    at::Tensor out = at::empty({batch, 1, heads * dim}, options);

    infllm_window_args a;
    std::memset(&a, 0, sizeof(a));
    a.d_q = q->data_ptr(); a.d_k = k->data_ptr(); a.d_v = v->data_ptr();
    a.q_sb = q->stride(0); a.q_sh = dim; a.q_sl = q->stride(1);
    a.k_sb = k->stride(0); a.k_sh = dim; a.k_sl = k->stride(1);
    a.v_sb = v->stride(0); a.v_sh = dim; a.v_sl = v->stride(1);
    a.B = (int32_t)batch; a.H = (int32_t)heads; a.Hkv = (int32_t)kv_heads; a.dim = (int32_t)dim;
    a.n_q = a.n_new = 1;
    a.kind = (int32_t)kind; a.n_init = (int32_t)n_init; a.n_local = n_local; a.seen = seen;
    a.d_inv_freq = (const float *)freq->data_ptr(); a.distance_scale = distance_scale;
    a.d_old_k = old_k->data_ptr(); a.d_old_v = old_v->data_ptr();
    a.ok_sb = old_k->stride(0); a.ok_sh = old_k->stride(1); a.ov_sb = old_v->stride(0); a.ov_sh = old_v->stride(1);
    a.d_cache_k = new_k.data_ptr(); a.d_cache_v = new_v.data_ptr();
    a.ck_sb = new_k.stride(0); a.ck_sh = new_k.stride(1); a.cv_sb = new_v.stride(0); a.cv_sh = new_v.stride(1);
    a.rows_old = (int32_t)rows_old; a.rows_new = (int32_t)rows_new;
    a.d_raw_old = raw ? raw->data_ptr() : nullptr; a.d_raw = raw ? raw->data_ptr() : nullptr;
    a.raw_old = a.raw_new = (int32_t)raw_rows;
    a.d_work = (void *)held[2]; a.work_bytes = step_bytes;
    a.d_out = out.data_ptr(); a.o_sb = heads * dim; a.o_sh = dim; a.o_sl = heads * dim;
    a.d_ticket = ticket;
    a.softmax_scale = (float)(1.0 / std::sqrt((double)dim));

    long status;
    if (args[15] == forward_object) {
        Py_BEGIN_ALLOW_THREADS
        status = forward_address(&a, (void *)stream);
        Py_END_ALLOW_THREADS
    } else {
        PyObject *bytes = PyBytes_FromStringAndSize((const char *)&a, sizeof(a));
        PyObject *r = bytes ? PyObject_CallFunctionObjArgs(args[15], bytes, args[14], nullptr) : nullptr;
        Py_XDECREF(bytes);
        if (!r) return nullptr;
        status = PyLong_AsLong(r);
        Py_DECREF(r);
        if (PyErr_Occurred()) return nullptr;
    }
    if (status) return PyLong_FromLong(status);
    dict = attributes(new_k);                           // the words stay with the cache that goes on
    const int failed = PyDict_SetItem(dict, words_name, words);
    Py_DECREF(dict);
    if (failed) return nullptr;
    return Py_BuildValue("(N(NNLO))", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(new_k)), THPVariable_Wrap(std::move(new_v)), (long long)len_k,
                         raw_object);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"make_room", (PyCFunction)(void (*)(void))py_make_room, METH_FASTCALL, nullptr},
                         {"claim", (PyCFunction)(void (*)(void))py_claim, METH_FASTCALL, nullptr},
                         {"bind", (PyCFunction)(void (*)(void))py_bind, METH_FASTCALL, nullptr},
                         {"step", (PyCFunction)(void (*)(void))py_step, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    constexpr size_t kMinor = sizeof("3.1") - 1 + (PY_MINOR_VERSION >= 10);             // of "3.10.12"; the file's name names no interpreter
    if (std::strncmp(Py_GetVersion(), PY_VERSION, kMinor + 1) != 0)
        return PyErr_Format(PyExc_ImportError, "built for Python %s, not for %s", PY_VERSION, Py_GetVersion());
    room_name = PyUnicode_InternFromString("_infllm_room");
    words_name = PyUnicode_InternFromString("_infllm_words");
    return room_name && words_name ? PyModule_Create(&module) : nullptr;
}
