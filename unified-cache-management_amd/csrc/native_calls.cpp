// Native fronts of the calls that a serving process makes once per layer and step: arguments are read
// from the tensors and passed to libucm_hip.so here instead of one by one through ctypes.
//
// What bounds the small calls is host time: the three kernels of a decode step of one request take 10 us
// and issuing them took 17.5 us, 8 of them for reading some twenty tensor properties in Python, the current
// stream and a ctypes call of forty arguments.  Host time of a call before and with a front: grouped-query
// step 17.5 and 9.0 us, latent step 18.8 and 9.9, encode into the cache 10.7 and 3.3, rehash 11.1 and 3.4,
// float retrieval 14.0 and 8.2, softmax-mass retrieval 17.5 and 10.6; what is left is launches.
//
// A front handles the plain case only - exact torch.Tensor arguments on one GPU, of the types, shapes and
// layouts the kernels take as they are - and returns None for anything else; the Python caller then goes
// through its general path, which converts what can be converted and raises what has to be raised.  The
// conditions here are therefore the same or narrower ones, never wider.
#include <torch/csrc/autograd/python_variable.h>  // includes Python.h

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "ucm_hip.h"

namespace {

using at::Tensor;

// Reads the arguments one after the other; `ok` turns false at the first that is not plain.
struct Reader {
    PyObject* const* a;
    Py_ssize_t n, i = 0;
    bool ok = true;
    c10::Device dev{c10::DeviceType::CPU};

    Reader(PyObject* const* args, Py_ssize_t count, Py_ssize_t want) : a(args), n(count) { ok = count == want; }

    // A GPU tensor with memory of its own, on the device of those before it.  `none`: None is accepted (null).
    const Tensor* tensor(bool none = false)
    {
        if (!ok) return nullptr;
        PyObject* o = a[i++];
        if (none && o == Py_None) return nullptr;
        if (!THPVariable_CheckExact(o)) return fail();
        const Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return fail();
        if (dev.is_cpu()) dev = t.device();
        if (t.device() != dev) return fail();
        return &t;
    }
    int64_t integer()
    {
        if (!ok) return 0;
        PyObject* o = a[i++];
        if (!PyLong_CheckExact(o)) return fail(), 0;
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            return fail(), 0;
        }
        return v;
    }
    int32_t int32()
    {
        const int64_t v = integer();
        if (v < INT32_MIN || v > INT32_MAX) return fail(), 0;
        return (int32_t)v;
    }
    void need(bool cond) { ok = ok && cond; }
    std::nullptr_t fail()
    {
        ok = false;
        return nullptr;
    }
};

int dtype_code(const Tensor& t)
{
    switch (t.scalar_type()) {
        case at::kBFloat16: return UCM_DT_BF16;
        case at::kHalf: return UCM_DT_F16;
        case at::kFloat: return UCM_DT_F32;
        default: return -1;
    }
}

ucm_stream_t stream_of(const c10::Device& dev) { return (ucm_stream_t)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// Stride in elements; the dense one for an extent of 1, whose recorded stride is arbitrary.
int64_t extent_stride(const Tensor& t, int64_t dim)
{
    if (t.size(dim) > 1) return t.stride(dim);
    int64_t s = 1;
    for (int64_t d = dim + 1; d < t.dim(); ++d) s *= t.size(d);
    return s;
}

bool shape_is(const Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }

bool is_index(const Tensor& t) { return t.scalar_type() == at::kInt || t.scalar_type() == at::kLong; }

// Body of a front: runs f, which returns a new reference or null: for "not plain", or with a Python error set
// (an output that could not be wrapped; its kernels have been issued).
template <class F>
PyObject* front(F&& f)
{
    PyObject* r = nullptr;
    try {
        r = f();
    } catch (...) {  // raised again, as Python has it, by the general path
        PyErr_Clear();
        r = nullptr;
    }
    if (!r && !PyErr_Occurred()) Py_RETURN_NONE;
    return r;
}

template <class F>
int without_gil(F&& f)
{
    struct Released {  // taken again also where reading a tensor throws
        PyThreadState* s = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(s); }
    } released;
    return f();
}

// The tensors of a grouped-query step, checked like the step's own _arguments().
struct GqaArgs {
    const Tensor *w, *keys, *slot, *q, *cache, *table, *lens;
    int64_t T = 0;
    void read_and_check(Reader& r, int64_t B, int64_t Hq, int64_t Hkv, int64_t K, int64_t N, int64_t width, int64_t BS,
                        bool exact_width)
    {
        keys = r.tensor(true);
        slot = r.tensor(true);
        q = r.tensor();
        cache = r.tensor();
        table = r.tensor();
        lens = r.tensor();
        if (!r.ok) return;
        const auto dt = w->scalar_type();
        r.need(dtype_code(*w) >= 0 && w->dim() == 3 && q->scalar_type() == dt && shape_is(*q, {B, Hq, K}) && q->stride(2) == 1);
        r.need(cache->scalar_type() == at::kInt && cache->dim() == 4 && cache->stride(3) == 1 && cache->size(1) == BS &&
               cache->size(2) == Hkv && cache->size(3) == N / 32);
        r.need(table->scalar_type() == at::kInt && lens->scalar_type() == at::kInt && table->dim() == 2);
        if (!r.ok) return;
        r.need(table->size(0) == B && (exact_width ? table->size(1) == width : table->size(1) >= width) && table->stride(1) == 1);
        r.need(lens->numel() == B && lens->is_contiguous());
        if (keys) {
            r.need(keys->scalar_type() == dt && keys->dim() >= 1);
            if (!r.ok) return;
            T = keys->size(0);
            if (T) {
                r.need(shape_is(*keys, {T, Hkv, K}) && keys->stride(2) == 1);
                r.need(slot && is_index(*slot) && slot->numel() == T && slot->is_contiguous());
            }
        }
    }
};

// (w, q_codes, new_table, new_lens, workspace, Hq, Hkv, B, K, N, width, BS, topk, sink, recent, threshold,
//  new_keys, slot_mapping, queries, k_hash_cache, block_table, seq_lens) -> status
PyObject* gsa_step(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 22);
        GqaArgs g;
        g.w = r.tensor();
        const Tensor *codes = r.tensor(), *new_table = r.tensor(), *new_lens = r.tensor(), *ws = r.tensor();
        const int32_t Hq = r.int32(), Hkv = r.int32(), B = r.int32(), K = r.int32(), N = r.int32(), width = r.int32(), BS = r.int32();
        const int32_t topk = r.int32(), sink = r.int32(), recent = r.int32(), thr = r.int32();
        if (!r.ok) return nullptr;
        g.read_and_check(r, B, Hq, Hkv, K, N, width, BS, true);
        if (!r.ok) return nullptr;
        const int64_t T = g.T;
        const int dt = dtype_code(*g.w);
        const int64_t ts = extent_stride(*g.table, 0);
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_gsa_decode_step(
                T ? g.keys->data_ptr() : nullptr, T, T ? extent_stride(*g.keys, 0) : 0, T ? extent_stride(*g.keys, 1) : 0,
                T ? g.slot->data_ptr() : nullptr, T && g.slot->scalar_type() == at::kLong, g.q->data_ptr(), extent_stride(*g.q, 0),
                extent_stride(*g.q, 1), dt, K, g.w->data_ptr(), dt, (int32_t)g.w->size(0), N, (uint32_t*)g.cache->data_ptr(),
                g.cache->size(0), BS, Hkv, extent_stride(*g.cache, 0), extent_stride(*g.cache, 1), extent_stride(*g.cache, 2),
                (const int32_t*)g.table->data_ptr(), (int32_t)(ts > width ? ts : width), width,
                (const int32_t*)g.lens->data_ptr(), B, Hq, topk, sink, recent, thr, (uint32_t*)codes->data_ptr(),
                (int32_t*)new_table->data_ptr(), width, (int32_t*)new_lens->data_ptr(), ws->data_ptr(), (size_t)ws->numel(), st);
        });
        return PyLong_FromLong(rc);
    });
}

// (w, q_codes, out_idx, out_score, workspace, Hq, Hkv, B, K, N, max_blocks, BS, k, sink, recent, flags,
//  new_keys, slot_mapping, queries, k_hash_cache, block_table, seq_lens) -> status
PyObject* sparse_step(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 22);
        GqaArgs g;
        g.w = r.tensor();
        const Tensor *codes = r.tensor(), *idx = r.tensor(), *score = r.tensor(), *ws = r.tensor();
        const int32_t Hq = r.int32(), Hkv = r.int32(), B = r.int32(), K = r.int32(), N = r.int32(), width = r.int32(), BS = r.int32();
        const int32_t k = r.int32(), sink = r.int32(), recent = r.int32(), flags = r.int32();
        if (!r.ok) return nullptr;
        g.read_and_check(r, B, Hq, Hkv, K, N, width, BS, false);
        if (!r.ok) return nullptr;
        const int64_t T = g.T;
        const int dt = dtype_code(*g.w);
        const int64_t ts = extent_stride(*g.table, 0);
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_sparse_decode_step(
                T ? g.keys->data_ptr() : nullptr, T, T ? extent_stride(*g.keys, 0) : 0, T ? extent_stride(*g.keys, 1) : 0,
                T ? g.slot->data_ptr() : nullptr, T && g.slot->scalar_type() == at::kLong, g.q->data_ptr(), extent_stride(*g.q, 0),
                extent_stride(*g.q, 1), dt, K, g.w->data_ptr(), dt, (int32_t)g.w->size(0), N, (uint32_t*)g.cache->data_ptr(),
                g.cache->size(0), BS, Hkv, extent_stride(*g.cache, 0), extent_stride(*g.cache, 1), extent_stride(*g.cache, 2),
                (const int32_t*)g.table->data_ptr(), (int32_t)(ts > width ? ts : width), width,
                (const int32_t*)g.lens->data_ptr(), B, Hq, k, sink, recent, (uint32_t)flags, (uint32_t*)codes->data_ptr(),
                (int32_t*)idx->data_ptr(), (int32_t*)score->data_ptr(), ws->data_ptr(), (size_t)ws->numel(), st);
        });
        return PyLong_FromLong(rc);
    });
}

// (w_nope, w_rope, q_codes, new_table, new_lens, workspace, Hq, R, B, width, BS, topk, sink, recent, threshold,
//  new_nope, new_rope, slot_mapping, q_nope, q_rope, k_hash_cache, block_table, seq_lens) -> status
PyObject* gsa_step_mla(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 23);
        const Tensor *wn = r.tensor(), *wr = r.tensor(), *codes = r.tensor(), *new_table = r.tensor(), *new_lens = r.tensor(),
                     *ws = r.tensor();
        const int32_t Hq = r.int32(), R = r.int32(), B = r.int32(), width = r.int32(), BS = r.int32();
        const int32_t topk = r.int32(), sink = r.int32(), recent = r.int32(), thr = r.int32();
        const Tensor *kn = r.tensor(true), *kr = r.tensor(true), *slot = r.tensor(true), *qn = r.tensor(), *qr = r.tensor(),
                     *cache = r.tensor(), *table = r.tensor(), *lens = r.tensor();
        if (!r.ok) return nullptr;
        const auto dt = wn->scalar_type();
        r.need(dtype_code(*wn) >= 0 && wr->scalar_type() == dt && wn->dim() == 2 && wr->dim() == 2);
        if (!r.ok) return nullptr;
        const int64_t Kn = wn->size(0), Nn = wn->size(1), Kr = wr->size(0), Nr = wr->size(1), Wd = (Nn + Nr) / 32;
        const int64_t T = kn ? (kn->dim() == 2 ? kn->size(0) : -1) : 0;
        r.need(T >= 0 && qn->scalar_type() == dt && qr->scalar_type() == dt && shape_is(*qn, {B, Hq, Kn}) &&
               shape_is(*qr, {B, Hq, Kr}));
        if (!r.ok) return nullptr;
        r.need(qn->stride(2) == 1 && qr->stride(2) == 1);
        r.need(cache->scalar_type() == at::kInt && cache->dim() == 3 && cache->size(1) == BS && cache->size(2) == Wd &&
               cache->stride(2) == 1);
        r.need(table->scalar_type() == at::kInt && lens->scalar_type() == at::kInt && shape_is(*table, {B, width}) &&
               table->stride(1) == 1 && lens->numel() == B && lens->is_contiguous());
        if (T)
            r.need(kr && kn->scalar_type() == dt && kr->scalar_type() == dt && shape_is(*kn, {T, Kn}) && shape_is(*kr, {T, Kr}) &&
                   kn->stride(1) == 1 && kr->stride(1) == 1 && slot && is_index(*slot) && slot->numel() == T &&
                   slot->is_contiguous());
        if (!r.ok) return nullptr;
        const int dtc = dtype_code(*wn);
        const int64_t ts = extent_stride(*table, 0);
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_gsa_decode_step_mla(
                T ? kn->data_ptr() : nullptr, T ? extent_stride(*kn, 0) : 0, T ? kr->data_ptr() : nullptr, T ? extent_stride(*kr, 0) : 0, T,
                T ? slot->data_ptr() : nullptr, T && slot->scalar_type() == at::kLong, qn->data_ptr(), extent_stride(*qn, 0),
                extent_stride(*qn, 1), qr->data_ptr(), extent_stride(*qr, 0), extent_stride(*qr, 1), dtc, (int32_t)Kn, (int32_t)Kr, wn->data_ptr(),
                wr->data_ptr(), dtc, (int32_t)Nn, (int32_t)Nr, (uint32_t*)cache->data_ptr(), cache->size(0), BS,
                extent_stride(*cache, 0), extent_stride(*cache, 1), (const int32_t*)table->data_ptr(), (int32_t)(ts > width ? ts : width),
                width, (const int32_t*)lens->data_ptr(), B, Hq, R, topk, sink, recent, thr, (uint32_t*)codes->data_ptr(),
                (int32_t*)new_table->data_ptr(), width, (int32_t*)new_lens->data_ptr(), ws->data_ptr(), (size_t)ws->numel(), st);
        });
        return PyLong_FromLong(rc);
    });
}

// A code cache [NB, BS, H, codes] of bytes or a wider type, as 32-bit words.
struct CodeCache {
    uint32_t* p;
    int64_t NB, sb, ss, sh;
    bool read(const Tensor& c, int64_t BS, int64_t H, int64_t code_bytes)
    {
        switch (c.scalar_type()) {
            case at::kByte: case at::kBFloat16: case at::kHalf: case at::kShort: case at::kInt: case at::kFloat: break;
            default: return false;
        }
        const int64_t es = c.element_size();
        if (c.dim() != 4 || c.size(1) != BS || c.size(2) != H || c.size(3) * es != code_bytes || c.stride(3) != 1) return false;
        NB = c.size(0);
        sb = extent_stride(c, 0) * es;
        ss = extent_stride(c, 1) * es;
        sh = extent_stride(c, 2) * es;
        p = (uint32_t*)c.data_ptr();
        if (sb % 4 || ss % 4 || sh % 4 || (uintptr_t)p % 4) return false;
        sb /= 4;
        ss /= 4;
        sh /= 4;
        return true;
    }
};

// (w [n_w, K, N], hash_weights, heads_per_w, block_size, x [T, H, K], slot_mapping, k_hash_cache) -> status
PyObject* encode_cache(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 7);
        const Tensor *w = r.tensor(), *hw = r.tensor();
        (void)hw;  // the encoder's own copy: on the same device
        const int32_t hpw = r.int32(), BS = r.int32();
        const Tensor *x = r.tensor(), *slot = r.tensor(), *cache = r.tensor();
        if (!r.ok) return nullptr;
        const int dt = dtype_code(*w);
        r.need(dt >= 0 && w->dim() == 3 && x->scalar_type() == w->scalar_type() && x->dim() == 3 && slot->dim() == 1);
        if (!r.ok) return nullptr;
        const int64_t T = x->size(0), H = x->size(1), K = x->size(2), N = w->size(2);
        CodeCache c;
        r.need(K == w->size(1) && K <= INT32_MAX && H <= INT32_MAX && x->stride(2) == 1 && N % 32 == 0 && slot->size(0) == T &&
               is_index(*slot) && slot->is_contiguous() && c.read(*cache, BS, H, N / 8));
        if (!r.ok || T == 0) return nullptr;
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_hash_encode_cache(x->data_ptr(), dt, T, (int32_t)H, (int32_t)K, extent_stride(*x, 0), extent_stride(*x, 1),
                                         w->data_ptr(), dt, (int32_t)w->size(0), hpw, (int32_t)N, slot->data_ptr(),
                                         slot->scalar_type() == at::kLong, c.p, c.NB, BS, c.sb, c.ss, c.sh, st);
        });
        return PyLong_FromLong(rc);
    });
}

// (w, hash_weights, heads_per_w, block_size, k_cache [NB, BS, H, K], block_ids, num_tokens, k_hash_cache) -> status
PyObject* encode_paged(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 8);
        const Tensor *w = r.tensor(), *hw = r.tensor();
        (void)hw;
        const int32_t hpw = r.int32(), BS = r.int32();
        const Tensor *x = r.tensor(), *ids = r.tensor();
        const int64_t tokens = r.integer();
        const Tensor* cache = r.tensor();
        if (!r.ok) return nullptr;
        const int dt = dtype_code(*w);
        r.need(dt >= 0 && w->dim() == 3 && x->scalar_type() == w->scalar_type() && x->dim() == 4 && ids->dim() == 1 &&
               ids->scalar_type() == at::kInt && ids->is_contiguous());
        if (!r.ok) return nullptr;
        const int64_t H = x->size(2), K = x->size(3), N = w->size(2), n = ids->size(0);
        CodeCache c;
        r.need(x->size(1) == BS && K == w->size(1) && K <= INT32_MAX && H <= INT32_MAX && x->stride(3) == 1 && N % 32 == 0 &&
               tokens > 0 && tokens <= n * BS && c.read(*cache, BS, H, N / 8));
        if (!r.ok) return nullptr;
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_hash_encode_paged(x->data_ptr(), dt, x->size(0), BS, (int32_t)H, (int32_t)K, extent_stride(*x, 0), extent_stride(*x, 1),
                                         extent_stride(*x, 2), (const int32_t*)ids->data_ptr(), n, tokens, w->data_ptr(), dt,
                                         (int32_t)w->size(0), hpw, (int32_t)N, c.p, c.NB, c.sb, c.ss, c.sh, st);
        });
        return PyLong_FromLong(rc);
    });
}

PyObject* pair_of(Tensor&& a, Tensor&& b)
{
    PyObject* pa = THPVariable_Wrap(std::move(a));
    if (!pa) return nullptr;
    PyObject* pb = THPVariable_Wrap(std::move(b));
    if (!pb) {
        Py_DECREF(pa);
        return nullptr;
    }
    PyObject* t = PyTuple_New(2);
    if (!t) {
        Py_DECREF(pa);
        Py_DECREF(pb);
        return nullptr;
    }
    PyTuple_SET_ITEM(t, 0, pa);
    PyTuple_SET_ITEM(t, 1, pb);
    return t;
}

// (data [n, dim], query [B, dim], indexes [B, max_n], topk, workspace or None) -> (indices, scores), or a status
PyObject* dot_topk(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 5);
        const Tensor *data = r.tensor(), *q = r.tensor(), *idx = r.tensor();
        const int32_t k = r.int32();
        const Tensor* given = r.tensor(true);
        if (!r.ok) return nullptr;
        r.need(data->scalar_type() == at::kFloat && q->scalar_type() == at::kFloat && idx->scalar_type() == at::kInt &&
               data->dim() == 2 && q->dim() == 2 && idx->dim() == 2 && data->is_contiguous() && q->is_contiguous() &&
               idx->is_contiguous() && k > 0);
        if (!r.ok) return nullptr;
        const int64_t n = data->size(0), dim = data->size(1), B = idx->size(0), max_n = idx->size(1);
        r.need(q->size(1) == dim && q->size(0) == B && B > 0 && max_n > 0 && dim <= INT32_MAX && B <= INT32_MAX && max_n <= INT32_MAX);
        if (!r.ok) return nullptr;
        const size_t need = ucm_dot_topk_workspace_bytes((int32_t)B, (int32_t)max_n);
        Tensor ws, out_idx = at::empty({B, k}, idx->options()), out_score = at::empty({B, k}, data->options());
        if (given && (size_t)given->numel() >= need) ws = *given;
        else ws = at::empty({(int64_t)need}, data->options().dtype(at::kByte));
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_dot_topk((const float*)data->data_ptr(), n, (int32_t)dim, (const float*)q->data_ptr(),
                                (const int32_t*)idx->data_ptr(), (int32_t)B, (int32_t)max_n, k, (int32_t*)out_idx.data_ptr(),
                                (float*)out_score.data_ptr(), ws.data_ptr(), (size_t)ws.numel(), st);
        });
        return rc == UCM_OK ? pair_of(std::move(out_idx), std::move(out_score)) : PyLong_FromLong(rc);
    });
}

// (query_group [x, Hq, d_orig], blk_repre [n, M, Hkv, d], pruned_index [Hkv, d] or None, topk, workspace or None)
// -> (block numbers, scores), or a status
PyObject* kvstar_topk(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    return front([&]() -> PyObject* {
        Reader r(args, nargs, 5);
        const Tensor *q = r.tensor(), *k = r.tensor(), *pr = r.tensor(true);
        const int32_t topk = r.int32();
        const Tensor* given = r.tensor(true);
        if (!r.ok) return nullptr;
        r.need(q->scalar_type() == at::kHalf && k->scalar_type() == at::kHalf && q->dim() == 3 && k->dim() == 4 &&
               q->is_contiguous() && k->is_contiguous());
        if (!r.ok) return nullptr;
        const int64_t X = q->size(0), Hq = q->size(1), d_orig = q->size(2), n = k->size(0), M = k->size(1), Hkv = k->size(2), d = k->size(3);
        r.need(!pr || (pr->scalar_type() == at::kLong && shape_is(*pr, {Hkv, d}) && pr->is_contiguous()));
        const int64_t kk = topk < n ? topk : n;
        r.need(kk > 0 && X <= INT32_MAX && Hq <= INT32_MAX && d_orig <= INT32_MAX && M <= INT32_MAX && Hkv <= INT32_MAX && d <= INT32_MAX);
        if (!r.ok) return nullptr;
        const size_t need = ucm_kvstar_topk_workspace_bytes((int32_t)X, (int32_t)Hq, n, (int32_t)M);
        Tensor ws, out_idx = at::empty({kk}, q->options().dtype(at::kInt)), out_score = at::empty({kk}, q->options().dtype(at::kFloat));
        if (given && (size_t)given->numel() >= need) ws = *given;
        else ws = at::empty({(int64_t)need}, q->options().dtype(at::kByte));
        const ucm_stream_t st = stream_of(r.dev);
        const int rc = without_gil([&] {
            return ucm_kvstar_topk(q->data_ptr(), (int32_t)X, (int32_t)Hq, (int32_t)d_orig, k->data_ptr(), n, (int32_t)M,
                                   (int32_t)Hkv, (int32_t)d, pr ? (const int64_t*)pr->data_ptr() : nullptr, (int32_t)kk,
                                   (int32_t*)out_idx.data_ptr(), (float*)out_score.data_ptr(), ws.data_ptr(),
                                   (size_t)ws.numel(), st);
        });
        return rc == UCM_OK ? pair_of(std::move(out_idx), std::move(out_score)) : PyLong_FromLong(rc);
    });
}

#define UCM_FRONT(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {UCM_FRONT(gsa_step),     UCM_FRONT(sparse_step), UCM_FRONT(gsa_step_mla), UCM_FRONT(encode_cache),
                         UCM_FRONT(encode_paged), UCM_FRONT(dot_topk),    UCM_FRONT(kvstar_topk),  {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ucm_native", "Fronts of libucm_hip.so's per-step calls.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ucm_native(void) { return PyModule_Create(&module); }
