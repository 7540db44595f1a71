// The per-call host path of the Python entry points: the extension module
// kvq_decode_amd._host.
//
// A decode of one short sequence runs about 10 us on the GPU, but the Python entry point
// took about 22 us to launch it: some sixty attribute reads and checks of tensors, 33
// ctypes field stores, three allocations and two ctypes calls. These functions do the same
// checks, allocations and calls natively, straight on the tensors.
//
// Each returns None, having launched nothing, for a call it does not take: one that fails a
// check, an argument of another Python type than the usual one (a numpy integer, a tensor
// subclass, a tensor without storage), a q that needs a copy, a call the library refuses.
// The Python entry point then takes the call through its own path, which reports every error
// and converts what can be converted; so the calls accepted and the errors raised are those of
// the Python path. A failed launch (KVQ_ERR_HIP) is raised here: a kernel may be running, and
// the error is reported once. Nothing is kept from one call for the next.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "kvq.h"

namespace {

// libkvq.so's entry points, set once the Python binding has loaded it (bind), and the
// compute units of each device (0: not known yet).
struct Library {
    int (*head_blocks)(int32_t, int32_t);
    int (*plan_decode)(int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t,
                       int32_t*, int32_t*);
    int (*plan_units)(int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t,
                      int32_t*, int32_t*);
    int (*normalize_splits)(int32_t, int32_t, int32_t*, int32_t*);
    int (*paged_decode)(const kvq_decode_args*, int32_t, float*, float*, kvq_stream_t);
    int (*decode_units)(const kvq_decode_args*, int32_t, float*, float*, kvq_stream_t);
    int (*quantize_cache)(const kvq_decode_args*, const void*, const void*, int64_t, int64_t,
                          int64_t, kvq_stream_t);
    int (*quantize_append)(const kvq_decode_args*, const void*, const void*, void*, kvq_stream_t);
    int (*append_kv)(const kvq_decode_args*, const void*, const void*, kvq_stream_t);
    int (*reshape_and_cache)(const kvq_decode_args*, const void*, const void*, int64_t, int64_t,
                             const int64_t*, int32_t, kvq_stream_t);
};
Library L{};
bool bound = false;
PyObject* check_status = nullptr;  // _lib.check(func, status), which raises KvqError
constexpr int kMaxDevices = 64;
int32_t cu_count[kMaxDevices];

// nullptr for a library status below zero: not taken, except a failed launch, whose KvqError
// is set.
PyObject* refused(const char* func, int status) {
    if (status == KVQ_ERR_HIP) Py_XDECREF(PyObject_CallFunction(check_status, "si", func, status));
    return nullptr;
}

// An ordinary GPU tensor: exactly torch.Tensor (or Parameter), strided, with storage of its
// own; nullptr otherwise.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided ||
        t.unsafeGetTensorImpl()->is_python_dispatch() || t.is_neg())
        return nullptr;
    return &t;
}

bool int_arg(PyObject* o, int64_t* v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    *v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0 && *v >= INT32_MIN && *v <= INT32_MAX;
}

// kvq_kv_format of a format name, -1 for another
int format_of(PyObject* o) {
    if (!PyUnicode_CheckExact(o)) return -1;
    if (PyUnicode_CompareWithASCIIString(o, "fp16") == 0) return KVQ_KV_F16;
    if (PyUnicode_CompareWithASCIIString(o, "int8") == 0) return KVQ_KV_INT8;
    if (PyUnicode_CompareWithASCIIString(o, "fp8_e4m3") == 0) return KVQ_KV_FP8_E4M3;
    if (PyUnicode_CompareWithASCIIString(o, "int4") == 0) return KVQ_KV_INT4;
    return -1;
}

bool pow2_16(int64_t x) { return x >= 16 && (x & (x - 1)) == 0; }

// ops.check_scale_pairs: fp16 [a, b, c] views of an interleaved (scale, zero) tensor
bool scale_pairs(const at::Tensor* s, const at::Tensor* z, int64_t a, int64_t b, int64_t c) {
    for (const at::Tensor* t : {s, z}) {
        if (!t || t->scalar_type() != at::kHalf || t->dim() != 3 || t->size(0) != a ||
            t->size(1) != b || t->size(2) != c || t->stride(2) != 2 || t->stride(1) != 2 * c ||
            t->stride(0) != 2 * b * c)
            return false;
    }
    return static_cast<char*>(z->data_ptr()) == static_cast<char*>(s->data_ptr()) + 2;
}

void caches(kvq_decode_args* a, const at::Tensor& k, const at::Tensor& v) {
    a->k_cache = k.data_ptr();
    a->k_stride_blk = k.stride(0);
    a->k_stride_tok = k.stride(1);
    a->k_stride_head = k.stride(2);
    a->v_cache = v.data_ptr();
    a->v_stride_blk = v.stride(0);
    a->v_stride_tok = v.stride(1);
    a->v_stride_head = v.stride(2);
    a->num_blocks = int32_t(k.size(0));
    a->block_size = int32_t(k.size(1));
    a->kv_heads = int32_t(k.size(2));
}

// block_table [B, max_blocks] and seq_lens [B], int32
bool tables(kvq_decode_args* a, const at::Tensor& bt, const at::Tensor& sl, int64_t B) {
    if (bt.scalar_type() != at::kInt || sl.scalar_type() != at::kInt || bt.dim() != 2 ||
        bt.size(0) != B || bt.stride(1) != 1 || sl.dim() != 1 || sl.size(0) != B ||
        !sl.is_contiguous())
        return false;
    a->block_table = static_cast<const int32_t*>(bt.data_ptr());
    a->bt_stride_b = bt.stride(0);
    a->seq_lens = static_cast<const int32_t*>(sl.data_ptr());
    a->batch = int32_t(B);
    a->max_blocks = int32_t(bt.size(1));
    return true;
}

kvq_stream_t stream_of(const at::Tensor& t) {
    return reinterpret_cast<kvq_stream_t>(
        c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

// every size the argument struct holds as int32 fits one
bool fits(const at::Tensor& t) {
    for (int64_t n : t.sizes())
        if (n > INT32_MAX) return false;
    return true;
}

// decode(q, k_cache, v_cache, block_table, seq_lens, scale, num_splits, kv_format, k_scale,
//        k_zero, v_scale, v_zero, k_group, out, workspace, waves_per_group, pipeline, units)
PyObject* decode(PyObject* const* o, Py_ssize_t n) {
    if (n != 18) return nullptr;
    const at::Tensor *q = plain(o[0]), *k = plain(o[1]), *v = plain(o[2]), *bt = plain(o[3]),
                     *sl = plain(o[4]);
    if (!q || !k || !v || !bt || !sl || q->dim() != 3 || k->dim() != 4 || !fits(*q) ||
        !fits(*k) || !fits(*bt))
        return nullptr;
    const c10::Device dev = q->device();
    if (k->device() != dev || v->device() != dev || bt->device() != dev || sl->device() != dev)
        return nullptr;
    const int64_t B = q->size(0), Hq = q->size(1), D = q->size(2), bs = k->size(1),
                  Hkv = k->size(2), Dc = k->size(3);
    const int fmt = format_of(o[7]);
    if (fmt < 0 || B < 1 || Hkv < 1 || Hq % Hkv || Hq < 1 || !pow2_16(D) || !pow2_16(bs) ||
        q->scalar_type() != at::kHalf || v->sizes() != k->sizes() || q->stride(2) != 1 ||
        k->stride(3) != 1 || v->stride(3) != 1)
        return nullptr;
    kvq_decode_args a{};
    if (fmt == KVQ_KV_F16) {
        if (k->scalar_type() != at::kHalf || v->scalar_type() != at::kHalf || Dc != D) return nullptr;
        a.k_scale = a.k_zero = a.v_scale = a.v_zero = nullptr;
    } else {
        const at::Tensor *ks = plain(o[8]), *kz = plain(o[9]), *vs = plain(o[10]), *vz = plain(o[11]);
        if (k->scalar_type() != at::kByte || v->scalar_type() != at::kByte ||
            Dc != (fmt == KVQ_KV_INT4 ? D / 2 : D) || !scale_pairs(ks, kz, k->size(0), Hkv, D) ||
            !scale_pairs(vs, vz, k->size(0), Hkv, bs > 32 ? bs : 32))
            return nullptr;
        a.k_scale = ks->data_ptr();
        a.k_zero = kz->data_ptr();
        a.v_scale = vs->data_ptr();
        a.v_zero = vz->data_ptr();
    }
    if (!tables(&a, *bt, *sl, B)) return nullptr;
    // rows the kernels' vector loads can take; the Python path copies others
    if (q->stride(0) % 8 || q->stride(1) % 8 || reinterpret_cast<uintptr_t>(q->data_ptr()) % 16)
        return nullptr;
    double scale;
    if (o[5] == Py_None) scale = 1.0 / std::sqrt(double(D));
    else if (PyFloat_CheckExact(o[5])) scale = PyFloat_AS_DOUBLE(o[5]);
    else return nullptr;
    int64_t splits = 0, k_group, waves, pipeline, units;
    const bool auto_plan = o[6] == Py_None;
    if ((!auto_plan && !int_arg(o[6], &splits)) || !int_arg(o[12], &k_group) ||
        !int_arg(o[15], &waves) || !int_arg(o[16], &pipeline) || !int_arg(o[17], &units) ||
        units < 0 || (units > 0 && !auto_plan))
        return nullptr;
    caches(&a, *k, *v);
    a.q = q->data_ptr();
    a.q_stride_b = q->stride(0);
    a.q_stride_h = q->stride(1);
    a.q_heads = int32_t(Hq);
    a.head_dim = int32_t(D);
    a.scale = float(scale);
    a.kv_format = fmt;
    a.k_group = int32_t(k_group);
    a.waves_per_group = int32_t(waves);
    a.pipeline = int32_t(pipeline);

    const at::Tensor *op = nullptr, *lse = nullptr;
    if (o[14] != Py_None) {
        if (!PyTuple_CheckExact(o[14]) || PyTuple_GET_SIZE(o[14]) != 2) return nullptr;
        op = plain(PyTuple_GET_ITEM(o[14], 0));
        lse = plain(PyTuple_GET_ITEM(o[14], 1));
        if (!op || !lse || op->scalar_type() != at::kFloat || lse->scalar_type() != at::kFloat ||
            !op->is_contiguous() || !lse->is_contiguous() || op->device() != dev ||
            lse->device() != dev)
            return nullptr;
    }
    const at::Tensor* out_given = nullptr;
    if (o[13] != Py_None) {
        out_given = plain(o[13]);
        if (!out_given || out_given->device() != dev || out_given->scalar_type() != at::kHalf ||
            out_given->sizes() != q->sizes() || out_given->stride(2) != 1)
            return nullptr;
    }

    // the partition
    const int hb = L.head_blocks(int32_t(Hq), int32_t(Hkv));
    const int idx = dev.index();
    if (hb < 1 || idx < 0 || idx >= kMaxDevices || Hkv * hb > INT32_MAX) return nullptr;
    const int32_t heads = int32_t(Hkv * hb);
    int32_t u = int32_t(units), s = 1, w = 0, pps = 0;
    if (auto_plan && units == 0) {
        const int32_t cu = cu_count[idx];
        if (cu == 0) return nullptr;
        if (L.plan_units(a.batch, a.q_heads, heads, a.block_size, a.max_blocks, fmt, a.head_dim, cu,
                         &u, &w) < 0)
            return nullptr;
        if (u == 0) {
            if (L.plan_decode(a.batch, a.q_heads, heads, a.block_size, a.max_blocks, fmt, a.head_dim,
                              cu, &s, &w) < 0)
                return nullptr;
            splits = s;
        }
        if (waves == 0) a.waves_per_group = w;
    }
    if (u == 0 && L.normalize_splits(int32_t(splits), a.max_blocks, &s, &pps) < 0) return nullptr;

    // the workspace: [Hq, units + B, D] or [B, Hq, S, D], and one float per row
    const int64_t rows = u > 0 ? Hq * (int64_t(u) + B) : s > 1 ? B * Hq * s : 0;
    at::Tensor own_out, own_op, own_lse;
    const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
    if (rows > 0 && op) {
        if (op->numel() < rows * D || lse->numel() < rows) return nullptr;
    } else if (rows > 0) {
        own_op = at::empty({rows * D}, f32);
        own_lse = at::empty({rows}, f32);
        op = &own_op;
        lse = &own_lse;
    }
    if (!out_given) {
        own_out = at::empty({B, Hq, D}, at::TensorOptions().dtype(at::kHalf).device(dev));
        out_given = &own_out;
    }
    a.out = out_given->data_ptr();
    a.o_stride_b = out_given->stride(0);
    a.o_stride_h = out_given->stride(1);
    float* opp = rows > 0 ? static_cast<float*>(op->data_ptr()) : nullptr;
    float* lsp = rows > 0 ? static_cast<float*>(lse->data_ptr()) : nullptr;
    const kvq_stream_t stream = stream_of(*q);
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = u > 0 ? L.decode_units(&a, u, opp, lsp, stream) : L.paged_decode(&a, s, opp, lsp, stream);
    Py_END_ALLOW_THREADS;
    if (st < 0) return refused(u > 0 ? "kvq_decode_units" : "kvq_paged_decode", st);
    if (own_out.defined()) return THPVariable_Wrap(std::move(own_out));
    return Py_NewRef(o[13]);
}

// The quantized cache given as quant.QuantizedKVCache's fields, checked as
// quant._check_cache does, for batches of B sequences.
bool quant_cache(kvq_decode_args* a, PyObject* cache, const at::Tensor& bt, const at::Tensor& sl,
                 int64_t B, int64_t D, const at::Tensor** codes) {
    if (!PyTuple_Check(cache) || PyTuple_GET_SIZE(cache) != 8) return false;
    const at::Tensor* t[6];
    for (int i = 0; i < 6; ++i) {
        t[i] = plain(PyTuple_GET_ITEM(cache, i));
        if (!t[i] || t[i]->device() != bt.device() || !fits(*t[i])) return false;
    }
    const at::Tensor &k = *t[0], &v = *t[1];
    const int fmt = format_of(PyTuple_GET_ITEM(cache, 6));
    int64_t k_group;
    if (fmt <= KVQ_KV_F16 || !int_arg(PyTuple_GET_ITEM(cache, 7), &k_group)) return false;
    if (D != 64 && D != 128 && D != 256) return false;
    if (k.dim() != 4 || v.sizes() != k.sizes() || k.scalar_type() != at::kByte ||
        v.scalar_type() != at::kByte || k.size(3) != (fmt == KVQ_KV_INT4 ? D / 2 : D))
        return false;
    const int64_t nb = k.size(0), bs = k.size(1), h = k.size(2);
    if (bs < 1 || k_group % bs || !scale_pairs(t[2], t[3], nb, h, D) ||
        !scale_pairs(t[4], t[5], nb, h, bs > 32 ? bs : 32) || sl.device() != bt.device() ||
        !fits(bt) || !tables(a, bt, sl, B))
        return false;
    caches(a, k, v);
    a->q_heads = a->kv_heads;
    a->head_dim = int32_t(D);
    a->kv_format = fmt;
    a->k_group = int32_t(k_group);
    a->k_scale = t[2]->data_ptr();
    a->k_zero = t[3]->data_ptr();
    a->v_scale = t[4]->data_ptr();
    a->v_zero = t[5]->data_ptr();
    *codes = t[0];
    return true;
}

bool half_rows(const at::Tensor* t, at::IntArrayRef shape, c10::Device dev) {
    return t && t->scalar_type() == at::kHalf && t->sizes() == shape && t->is_contiguous() &&
           t->device() == dev;
}

// quantize(cache, k_cache, v_cache, block_table, seq_lens)
PyObject* quantize(PyObject* const* o, Py_ssize_t n) {
    if (n != 5) return nullptr;
    const at::Tensor *k = plain(o[1]), *v = plain(o[2]), *bt = plain(o[3]), *sl = plain(o[4]);
    if (!k || !v || !bt || !sl || k->dim() != 4 || k->scalar_type() != at::kHalf ||
        v->scalar_type() != at::kHalf || k->sizes() != v->sizes() || k->strides() != v->strides() ||
        k->stride(3) != 1 || bt->dim() != 2 || k->device() != bt->device() ||
        v->device() != bt->device())
        return nullptr;
    kvq_decode_args a{};
    const at::Tensor* codes;
    if (!quant_cache(&a, o[0], *bt, *sl, bt->size(0), k->size(3), &codes)) return nullptr;
    for (int d = 0; d < 3; ++d)
        if (codes->size(d) != k->size(d)) return nullptr;
    const kvq_stream_t stream = stream_of(*k);
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = L.quantize_cache(&a, k->data_ptr(), v->data_ptr(), k->stride(0), k->stride(1),
                          k->stride(2), stream);
    Py_END_ALLOW_THREADS;
    return st < 0 ? refused("kvq_quantize_cache", st) : Py_NewRef(Py_True);
}

// quantize_append(cache, k_new, v_new, block_table, seq_lens, k_resid)
PyObject* quantize_append(PyObject* const* o, Py_ssize_t n) {
    if (n != 6) return nullptr;
    const at::Tensor *kn = plain(o[1]), *vn = plain(o[2]), *bt = plain(o[3]), *sl = plain(o[4]),
                     *res = plain(o[5]);
    if (!kn || !vn || !bt || !sl || !res || kn->dim() != 3) return nullptr;
    const int64_t B = kn->size(0), h = kn->size(1), D = kn->size(2);
    kvq_decode_args a{};
    const at::Tensor* codes;
    if (!quant_cache(&a, o[0], *bt, *sl, B, D, &codes) || a.kv_heads != h) return nullptr;
    const c10::Device dev = bt->device();
    if (!half_rows(kn, {B, h, D}, dev) || !half_rows(vn, {B, h, D}, dev) ||
        !half_rows(res, {B, h, int64_t(a.k_group) + 2, D}, dev))
        return nullptr;
    const kvq_stream_t stream = stream_of(*kn);
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = L.quantize_append(&a, kn->data_ptr(), vn->data_ptr(), res->data_ptr(), stream);
    Py_END_ALLOW_THREADS;
    return st < 0 ? refused("kvq_quantize_append", st) : Py_NewRef(Py_True);
}

// The fp16 caches of the append entry points (cache._cache_args).
bool f16_caches(kvq_decode_args* a, const at::Tensor* k, const at::Tensor* v) {
    if (!k || !v || k->scalar_type() != at::kHalf || v->scalar_type() != at::kHalf ||
        k->dim() != 4 || v->sizes() != k->sizes() || k->stride(3) != 1 || v->stride(3) != 1 ||
        v->device() != k->device() || !fits(*k))
        return false;
    caches(a, *k, *v);
    a->head_dim = int32_t(k->size(3));
    a->kv_format = KVQ_KV_F16;
    return true;
}

// append_kv(k_cache, v_cache, k_new, v_new, block_table, seq_lens)
PyObject* append_kv(PyObject* const* o, Py_ssize_t n) {
    if (n != 6) return nullptr;
    const at::Tensor *k = plain(o[0]), *v = plain(o[1]), *kn = plain(o[2]), *vn = plain(o[3]),
                     *bt = plain(o[4]), *sl = plain(o[5]);
    kvq_decode_args a{};
    if (!f16_caches(&a, k, v) || !bt || !sl || bt->dim() != 2 || !fits(*bt)) return nullptr;
    const int64_t B = bt->size(0);
    const c10::Device dev = k->device();
    if (!half_rows(kn, {B, a.kv_heads, a.head_dim}, dev) ||
        !half_rows(vn, {B, a.kv_heads, a.head_dim}, dev) || bt->device() != dev ||
        sl->device() != dev || !tables(&a, *bt, *sl, B))
        return nullptr;
    const kvq_stream_t stream = stream_of(*k);
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = L.append_kv(&a, kn->data_ptr(), vn->data_ptr(), stream);
    Py_END_ALLOW_THREADS;
    return st < 0 ? refused("kvq_append_kv", st) : Py_NewRef(Py_True);
}

// reshape_and_cache(key, value, k_cache, v_cache, slot_mapping)
PyObject* reshape_and_cache(PyObject* const* o, Py_ssize_t n) {
    if (n != 5) return nullptr;
    const at::Tensor *key = plain(o[0]), *val = plain(o[1]), *k = plain(o[2]), *v = plain(o[3]),
                     *slots = plain(o[4]);
    kvq_decode_args a{};
    if (!f16_caches(&a, k, v) || !key || !val || !slots || key->dim() != 3 || !fits(*key))
        return nullptr;
    const int64_t shape[3] = {key->size(0), a.kv_heads, a.head_dim};
    const c10::Device dev = k->device();
    for (const at::Tensor* t : {key, val})
        if (t->scalar_type() != at::kHalf || t->sizes() != at::IntArrayRef(shape, 3) ||
            t->stride(2) != 1 || t->device() != dev)
            return nullptr;
    if (key->strides() != val->strides() || slots->scalar_type() != at::kLong ||
        slots->dim() != 1 || slots->size(0) != shape[0] || !slots->is_contiguous() ||
        slots->device() != dev)
        return nullptr;
    const kvq_stream_t stream = stream_of(*k);
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = L.reshape_and_cache(&a, key->data_ptr(), val->data_ptr(), key->stride(0), key->stride(1),
                             static_cast<const int64_t*>(slots->data_ptr()), int32_t(shape[0]),
                             stream);
    Py_END_ALLOW_THREADS;
    return st < 0 ? refused("kvq_reshape_and_cache", st) : Py_NewRef(Py_True);
}

// The Python-callable form: None for a call not taken. A C++ exception of torch (an
// allocation that fails, a tensor that gives no pointer) is one too: the Python path meets
// it again and raises it.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* entry(PyObject*, PyObject* const* o, Py_ssize_t n) {
    PyObject* r = nullptr;
    if (bound) {
        try {
            r = F(o, n);
        } catch (...) {
            r = nullptr;
        }
    }
    if (PyErr_Occurred()) return nullptr;
    return r ? r : Py_NewRef(Py_None);
}

// bind(check, address, ...): _lib.check, and libkvq.so's entry points in the order of
// Library's members
PyObject* bind(PyObject*, PyObject* const* o, Py_ssize_t n) {
    constexpr int kCount = sizeof(Library) / sizeof(void*);
    if (n != 1 + kCount || !PyCallable_Check(o[0])) {
        PyErr_SetString(PyExc_TypeError,
                        "bind takes the status check and one address per library entry point");
        return nullptr;
    }
    void* p[kCount];
    for (int i = 0; i < kCount; ++i) {
        p[i] = PyLong_AsVoidPtr(o[1 + i]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    memcpy(&L, p, sizeof(L));
    Py_XSETREF(check_status, Py_NewRef(o[0]));
    bound = true;
    Py_RETURN_NONE;
}

// set_cu_count(device, count)
PyObject* set_cu_count(PyObject*, PyObject* const* o, Py_ssize_t n) {
    int64_t i, c;
    if (n != 2 || !int_arg(o[0], &i) || !int_arg(o[1], &c) || i < 0 || c < 1) {
        PyErr_SetString(PyExc_TypeError, "set_cu_count takes a device index and a positive count");
        return nullptr;
    }
    if (i < kMaxDevices) cu_count[i] = int32_t(c);
    Py_RETURN_NONE;
}

template <typename F>
PyMethodDef method(const char* name, F f) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL,
            nullptr};
}

PyMethodDef methods[] = {method("bind", bind),
                         method("set_cu_count", set_cu_count),
                         method("decode", entry<decode>),
                         method("quantize", entry<quantize>),
                         method("quantize_append", entry<quantize_append>),
                         method("append_kv", entry<append_kv>),
                         method("reshape_and_cache", entry<reshape_and_cache>),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
