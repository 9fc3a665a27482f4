// CPython module of the package's host paths that run once per layer and step: what a call costs before its
// launches.  A decode call's argument checks and launch arguments took ~5.6 us of Python and ctypes next to
// ~6.8 us for the launches themselves, more than a small cache's time on the GPU: 11.8 -> 9.2 us per call at
// 3B's heads over 4k tokens, 11.7 -> 10.7 (GPU-bound) over 32k.  A cache build's allocations, launch
// arguments and ~45 metadata views took ~80 us next to 9 us of kernels: 92 -> 68 us (4k tokens), 99 -> 75
// (64k, 38 us of kernels).
//
// The decode entry takes the forms that a model's step uses and returns None for every other (strided or
// misaligned rows, other types, a full ring, a folded rotation, any error): those keep the Python path and
// its checks and messages.  It keeps nothing from a call.  The library's functions come as addresses, so
// that the module follows whichever library the package loaded.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "r2o_sspa.h"

namespace {

const at::Tensor* exact_tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool on_device(const at::Tensor& t, int64_t device) {
    return t.device().type() == at::kCUDA && t.device().index() == device && t.layout() == at::kStrided;
}

int row_code(const at::Tensor& t) {
    return t.scalar_type() == at::kBFloat16 ? 0 : (t.scalar_type() == at::kHalf ? 1 : -1);
}

bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// ------------------------------------------------------------------------------------ decode call
struct Decode {
    r2o_decode_params params;  // what stays from call to call (SplitKExecutor._static_params)
    int (*launch)(const r2o_decode_params*, void*);
    int64_t device;
};

void decode_free(PyObject* capsule) { delete static_cast<Decode*>(PyCapsule_GetPointer(capsule, "r2o_decode")); }

// decode_handle(params address, r2o_decode address, device index)
PyObject* decode_handle(PyObject*, PyObject* args) {
    unsigned long long params, fn;
    long long device;
    if (!PyArg_ParseTuple(args, "KKL", &params, &fn, &device)) return nullptr;
    auto* d = new Decode;
    std::memcpy(&d->params, reinterpret_cast<const void*>(params), sizeof(d->params));
    d->launch = reinterpret_cast<int (*)(const r2o_decode_params*, void*)>(fn);
    d->device = device;
    PyObject* capsule = PyCapsule_New(d, "r2o_decode", decode_free);
    if (!capsule) delete d;
    return capsule;
}

bool plain_int(PyObject* o, int64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

// One value per request: an int for all, or a list or tuple of b ints.
bool per_request(PyObject* o, int64_t b, int64_t* out) {
    if (plain_int(o, out[0])) {
        std::fill(out + 1, out + b, out[0]);
        return true;
    }
    if (!(PyList_CheckExact(o) || PyTuple_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != b) return false;
    for (int64_t i = 0; i < b; ++i)
        if (!plain_int(PySequence_Fast_GET_ITEM(o, i), out[i])) return false;
    return true;
}

PyObject* const kRecentPool = PyUnicode_InternFromString("recent_fp_pool");
PyObject* const kActiveLength = PyUnicode_InternFromString("active_length");
PyObject* const kCapacity = PyUnicode_InternFromString("capacity");

// An int attribute of o; false (with no exception set) if it is anything else.
bool int_attr(PyObject* o, PyObject* name, int64_t& v) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a) {
        PyErr_Clear();
        return false;
    }
    const bool ok = plain_int(a, v);
    Py_DECREF(a);
    return ok;
}

// decode(handle, query, append or None, output, caches list, own ring lengths list or None): the status of
// r2o_decode, or None for a call that the Python path makes.  With ring lengths of its own (a stacked
// executor) a call with an append advances them.
PyObject* decode_call(PyObject* const* args) {
    auto* d = static_cast<Decode*>(PyCapsule_GetPointer(args[0], "r2o_decode"));
    if (!d) return nullptr;
    r2o_decode_params p = d->params;
    const int64_t b = p.batch;
    if (b < 1 || b > R2O_MAX_BATCH) Py_RETURN_NONE;
    const at::Tensor *q = exact_tensor(args[1]), *out = exact_tensor(args[3]);
    if (!q || !out || !on_device(*q, d->device) || !on_device(*out, d->device)) Py_RETURN_NONE;
    const bool token_axis = q->dim() == 4 && q->size(2) == 1;
    if (!(q->dim() == 3 || token_axis) || q->size(0) != b || q->size(1) != p.hq || q->size(-1) != R2O_HEAD_DIM ||
        !q->is_contiguous() || !aligned16(*q) || row_code(*q) < 0)
        Py_RETURN_NONE;
    if (out->dim() != 3 || out->size(0) != b || out->size(1) != p.hq || out->size(2) != R2O_HEAD_DIM) Py_RETURN_NONE;
    p.query = static_cast<const uint16_t*>(q->data_ptr());
    p.q_dtype = row_code(*q);
    p.out = static_cast<uint16_t*>(out->data_ptr());

    PyObject *caches = args[4], *own = args[5];
    if (!PyList_CheckExact(caches) || PyList_GET_SIZE(caches) != b) Py_RETURN_NONE;
    const bool stacked = own != Py_None;
    if (stacked && (!PyList_CheckExact(own) || PyList_GET_SIZE(own) != b)) Py_RETURN_NONE;
    bool room = true;
    int64_t lengths[R2O_MAX_BATCH];
    for (int64_t i = 0; i < b; ++i) {
        int64_t capacity = 0;
        if (stacked && i > 0) {  // one capacity for all, as the Python path checks
            if (!plain_int(PyList_GET_ITEM(own, i), lengths[i])) Py_RETURN_NONE;
            room = room && lengths[i] < p.recent_len[0];
            continue;
        }
        PyObject* pool = PyObject_GetAttr(PyList_GET_ITEM(caches, i), kRecentPool);
        if (!pool) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const bool ok = int_attr(pool, kCapacity, capacity) &&
                        (stacked ? plain_int(PyList_GET_ITEM(own, i), lengths[i]) : int_attr(pool, kActiveLength, lengths[i]));
        Py_DECREF(pool);
        if (!ok || capacity > 0x7fffffff) Py_RETURN_NONE;
        room = room && lengths[i] < capacity;
        if (stacked) p.recent_len[0] = (int32_t)capacity;
    }
    for (int64_t i = 0; i < b; ++i) {
        if (lengths[i] < 0 || lengths[i] > 0x7fffffff) Py_RETURN_NONE;
        p.recent_len[i] = (int32_t)lengths[i];
    }

    PyObject* append = args[2];
    if (append != Py_None) {
        if (!PyTuple_CheckExact(append) || PyTuple_GET_SIZE(append) != 4 || !room) Py_RETURN_NONE;
        const at::Tensor *k = exact_tensor(PyTuple_GET_ITEM(append, 0)), *v = exact_tensor(PyTuple_GET_ITEM(append, 1));
        const int64_t n = b * p.hkv * R2O_HEAD_DIM;
        for (const at::Tensor* t : {k, v})
            if (!t || !on_device(*t, d->device) || !t->is_contiguous() || t->numel() != n || !aligned16(*t) ||
                row_code(*t) != p.row_dtype)
                Py_RETURN_NONE;
        if (!per_request(PyTuple_GET_ITEM(append, 2), b, p.append_global) ||
            !per_request(PyTuple_GET_ITEM(append, 3), b, p.append_logical))
            Py_RETURN_NONE;
        p.append_k = static_cast<const uint16_t*>(k->data_ptr());
        p.append_v = static_cast<const uint16_t*>(v->data_ptr());
        p.do_append = 1;
    }
    void* stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)d->device).stream();
    int rc;
    {
        WithoutGil released;
        rc = d->launch(&p, stream);
    }
    if (rc == R2O_OK && stacked && append != Py_None)
        for (int64_t i = 0; i < b; ++i) {
            PyObject* next = PyLong_FromLongLong(lengths[i] + 1);
            if (!next || PyList_SetItem(own, i, next)) return nullptr;
        }
    return PyLong_FromLong(rc);
}

PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 6) Py_RETURN_NONE;
    try {
        return decode_call(args);
    } catch (...) {  // a tensor without memory of its own (vmap, a subclass): the Python path's error
        Py_RETURN_NONE;
    }
}

// ------------------------------------------------------------------------------------- cache build
int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

PyObject* wrap(const at::Tensor& t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}

// A tuple of the tensors (None where undefined).
PyObject* wrap_all(const std::vector<at::Tensor>& ts) {
    PyObject* tuple = PyTuple_New((Py_ssize_t)ts.size());
    for (size_t i = 0; tuple && i < ts.size(); ++i) {
        PyObject* o = wrap(ts[i]);
        if (!o) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, (Py_ssize_t)i, o);
    }
    return tuple;
}

// cache_build(key, value, global, logical, page table [3, pages] on the host, r2o_cache_page_words address,
// r2o_cache_build address, tier pages (4), tier tokens (4), page size, ring capacity, append capacity,
// superblock, INT2 group, key bits (4, 2, 16), INT4 generated values): allocates every tensor of the cache,
// uploads the page words and launches; the callers have checked shapes, types and devices.  Returns
// (status, payload tensors, metadata tensors) in the order that cache.py unpacks.
PyObject* cache_build(PyObject*, PyObject* args) {
    PyObject *key_o, *value_o, *global_o, *logical_o, *table_o;
    unsigned long long words_fn, build_fn;
    long long tp[4], tt[4], page_size, ring, append, superblock, group, k_bits;
    int gen_int4;
    if (!PyArg_ParseTuple(args, "OOOOOKK(LLLL)(LLLL)LLLLLLp", &key_o, &value_o, &global_o, &logical_o, &table_o, &words_fn,
                          &build_fn, tp, tp + 1, tp + 2, tp + 3, tt, tt + 1, tt + 2, tt + 3, &page_size, &ring, &append,
                          &superblock, &group, &k_bits, &gen_int4))
        return nullptr;
    for (PyObject* o : {key_o, value_o, global_o, logical_o, table_o})
        if (!THPVariable_Check(o)) {
            PyErr_SetString(PyExc_TypeError, "cache_build takes tensors");
            return nullptr;
        }
    int rc = 0;
    std::vector<at::Tensor> payload, meta;
    try {
        WithoutGil released;
        const at::Tensor &key = THPVariable_Unpack(key_o), &value = THPVariable_Unpack(value_o),
                         &global = THPVariable_Unpack(global_o), &logical = THPVariable_Unpack(logical_o),
                         &table = THPVariable_Unpack(table_o);
        const int64_t h = key.size(0), s = key.size(1), n_pages = table.size(1);
        const int64_t s_fp = tt[0], s_i4 = tt[1], s_i2 = tt[2], n = s_fp + s_i4 + s_i2;
        const auto opt = at::TensorOptions().device(key.device());
        const auto u8 = opt.dtype(at::kByte), f16 = opt.dtype(at::kHalf), i64 = opt.dtype(at::kLong);

        at::Tensor fp_v, i4_v, i4_scale, k_packed, k_scale, k_zero, k_ops;
        if (s_fp) fp_v = at::empty({h, s_fp, 128}, opt.dtype(value.scalar_type()));
        int64_t i4_capacity = gen_int4 ? std::max<int64_t>(1, s_i4 + append) : s_i4;
        if (gen_int4) i4_v = at::empty({h, i4_capacity, 64}, u8);
        else if (s_i4) i4_v = at::empty({h * s_i4 * 64}, u8);
        if (i4_capacity) i4_scale = at::empty({h, i4_capacity, 1}, opt.dtype(at::kFloat));
        const int64_t i2_capacity = std::max<int64_t>(128, round_up(s_i2 + (gen_int4 ? 0 : append), 128));
        at::Tensor i2_v = at::empty({h, i2_capacity, 32}, u8), i2_scale = at::empty({h, i2_capacity, 128 / group, 1}, f16),
                   i2_zero = at::empty({h, i2_capacity, 128 / group, 1}, u8);
        const int64_t capacity = std::max<int64_t>(128, round_up(n + append, 128)), blocks = capacity / superblock;
        int64_t reserve2 = 0, reserve4 = 0;
        if (k_bits == 16) {  // no compact K arena to flush into: nothing is reserved
            k_packed = at::empty({h, capacity, 128}, opt.dtype(key.scalar_type()));
        } else {
            k_packed = at::empty({h, capacity, 16 * k_bits}, u8);
            k_scale = at::empty({h, blocks, 128}, f16);
            k_zero = at::empty({h, blocks, 128}, k_bits == 4 ? u8 : f16);
            k_ops = at::empty({h, blocks, 128}, opt.dtype(at::kInt));
            reserve2 = std::min(i2_capacity - s_i2, capacity - n) / page_size * page_size;
            if (gen_int4) reserve4 = std::min(i4_capacity - s_i4, capacity - n) / page_size * page_size;
        }
        at::Tensor ring_k = at::empty({h, ring, 128}, opt.dtype(key.scalar_type())), ring_v = at::empty_like(ring_k);

        const int64_t spans[3] = {tp[0], tp[1] + reserve4 / page_size, tp[2] + reserve2 / page_size};
        const int64_t tokens[3] = {s_fp, s_i4 + reserve4, s_i2 + reserve2};
        const int64_t ring_pages = ring / page_size;
        const int64_t page_words = 3 * (spans[0] + spans[1] + spans[2] + ring_pages) + 1;
        at::Tensor words = at::empty({page_words + 3 * n_pages}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
        rc = reinterpret_cast<decltype(&r2o_cache_page_words)>(words_fn)(
            table.data_ptr<int64_t>(), n_pages, page_size, reserve4, reserve2, ring, words.data_ptr<int64_t>(), words.numel());
        if (!rc) {
            // pinned: a copy from pageable memory would wait for the stream's earlier work
            at::Tensor pages = words.to(i64, /*non_blocking=*/true);
            at::Tensor storage = at::empty({page_words + 2 * (tokens[0] + tokens[1] + tokens[2]) + tt[3] + 2 * ring}, i64);
            at::Tensor index = at::empty({n}, i64);

            auto ptr = [](const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
            r2o_cache_build_params p{};
            p.key = static_cast<const uint16_t*>(ptr(key));
            p.value = static_cast<const uint16_t*>(ptr(value));
            p.key_dtype = row_code(key);
            p.value_dtype = row_code(value);
            p.hkv = h;
            p.tokens = s;
            p.plan_global = static_cast<const int64_t*>(ptr(global));
            p.plan_logical = static_cast<const int64_t*>(ptr(logical));
            p.pages = static_cast<const int64_t*>(ptr(pages));
            p.page_words = page_words;
            p.n_pages = n_pages;
            for (int t = 0; t < 4; ++t) p.tier_tokens[t] = tt[t];
            p.reserve4 = reserve4;
            p.reserve2 = reserve2;
            p.storage = static_cast<int64_t*>(ptr(storage));
            p.index = static_cast<int64_t*>(ptr(index));
            p.ring_k = static_cast<uint16_t*>(ptr(ring_k));
            p.ring_v = static_cast<uint16_t*>(ptr(ring_v));
            p.ring_capacity = ring;
            p.k_bits = k_bits;
            p.superblock = superblock;
            p.k_packed = static_cast<uint8_t*>(ptr(k_packed));
            p.k_scale = static_cast<uint16_t*>(ptr(k_scale));
            p.k_zero = ptr(k_zero);
            p.k_operands = static_cast<uint32_t*>(ptr(k_ops));
            p.k_capacity = capacity;
            p.k_superblocks = blocks;
            p.fp_v = static_cast<uint16_t*>(ptr(fp_v));
            p.i4_v = static_cast<uint8_t*>(ptr(i4_v));
            p.i4_scale = static_cast<float*>(ptr(i4_scale));
            p.i4_capacity = i4_capacity;
            p.i2_v = static_cast<uint8_t*>(ptr(i2_v));
            p.i2_scale = static_cast<uint16_t*>(ptr(i2_scale));
            p.i2_zero = static_cast<uint8_t*>(ptr(i2_zero));
            p.i2_capacity = i2_capacity;
            p.i2_group = group;
            void* stream = c10::hip::getCurrentHIPStream(key.device().index()).stream();
            rc = reinterpret_cast<decltype(&r2o_cache_build)>(build_fn)(&p, stream);

            // the metadata storage's fields: per tier and for the ring ids, offsets, lengths; the length word; global
            // and logical indices per tier; evicted; ring global and logical; then the INT4 and INT2 pools' five
            // fields without their reserve
            meta.push_back(storage);
            int64_t at_word = 0;
            auto take = [&](int64_t len) {
                meta.push_back(storage.narrow(0, at_word, len));
                at_word += len;
            };
            for (int64_t span : {spans[0], spans[1], spans[2], ring_pages})
                for (int f = 0; f < 3; ++f) take(span);
            take(1);
            for (int f = 0; f < 2; ++f)
                for (int64_t span : tokens) take(span);
            take(tt[3]);
            take(ring);
            take(ring);
            meta[13] = meta[13].view(at::kInt).select(0, 0);
            for (int t = 1; t < 3; ++t)  // active views
                for (int f = 0; f < 5; ++f) {
                    const at::Tensor& full = f < 3 ? meta[1 + 3 * t + f] : meta[14 + 3 * (f - 3) + t];
                    const int64_t len = f < 3 ? tp[t] : tt[t];
                    meta.push_back(full.size(0) == len ? full : full.narrow(0, 0, len));
                }
            payload = {fp_v, i4_v, i4_scale, i2_v, i2_scale, i2_zero, k_packed, k_scale, k_zero, k_ops, ring_k, ring_v};
        }
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
    PyObject* tensors = wrap_all(payload);
    PyObject* fields = tensors ? wrap_all(meta) : nullptr;
    if (!fields) {
        Py_XDECREF(tensors);
        return nullptr;
    }
    return Py_BuildValue("(iNN)", rc, tensors, fields);
}

PyMethodDef kMethods[] = {
    {"decode_handle", decode_handle, METH_VARARGS, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, nullptr},
    {"cache_build", cache_build, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_r2o_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__r2o_host() { return PyModule_Create(&kModule); }
