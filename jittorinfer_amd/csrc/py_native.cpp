// The Python entry points' way from torch tensors to the C ABI (include/mla_attn.h, mla_kv_write.h, mla_front.h): one call that checks the
// tensors, fills the argument block and launches.  Filling a ctypes structure field by field took 6 us of a 13 us attention call and
// most of the 70 us a layer of a decode step spent on the host, more than its kernels run for small batches; here it takes
// under 1 us a call.  Every function takes its arguments by position; capi.py gives them names and defaults.
// What torch throws (out of memory, a tensor without strides or storage) ends at entry<>, as the Python exception torch itself would
// raise; every reference and buffer taken on the way has an owner that gives it back.
#include <Python.h>

#include <string.h>

#include <algorithm>
#include <vector>

#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/mla_attn.h"
#include "../../include/mla_front.h"
#include "../../include/mla_kv_write.h"

namespace {

constexpr int PAGE = MLA_PAGE_TOKENS;

// A launch may wait for room in the device's queue: other Python threads run meanwhile.
struct Unlocked {
    PyThreadState * t = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(t); }
};
template <typename F> int unlocked(F f) {
    const Unlocked u;
    return f();
}

// The library's entry points, the Python layer's workspace table and what grows it, torch's raw current stream: handed over by bind().
struct Bound {
    decltype(&mla_attn_workspace_size) workspace_size;
    decltype(&mla_attn_launch)         attn;
    decltype(&mla_kv_write_launch)     kv_write;
    decltype(&mla_kv_write_rope_launch) kv_write_rope;
    decltype(&mla_rope_launch)         rope;
    decltype(&mla_mul_mat_launch)      mul_mat;
    decltype(&mla_copy_f32_launch)     copy;
    decltype(&mla_front_batch_launch)  front_batch;
    PyObject * workspace, * workspaces, * raw_stream;
} lib;

#define REQUIRE(cond)                                        \
    do {                                                     \
        if (!(cond)) {                                       \
            PyErr_SetString(PyExc_AssertionError, #cond);    \
            return nullptr;                                  \
        }                                                    \
    } while (0)

const at::Tensor * tensor(PyObject * o) {
    if (THPVariable_Check(o)) return &THPVariable_Unpack(o);
    PyErr_SetString(PyExc_TypeError, "expected a torch tensor");
    return nullptr;
}
// a tensor or None
bool optional_tensor(PyObject * o, const at::Tensor *& t) {
    t = nullptr;
    if (o == Py_None) return true;
    t = tensor(o);
    return t != nullptr;
}
bool on_gpu(const at::Tensor & t) {
    if (t.is_cuda()) return true;
    PyErr_SetString(PyExc_RuntimeError, "jittorinfer_amd runs on a gfx950 GPU only (there is no CPU path)");
    return false;
}
bool arg_count(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return false;
}
PyObject * failed(const char * what, int rc) {
    PyErr_Format(PyExc_RuntimeError, "%s failed with code %d", what, rc);
    return nullptr;
}
// the stream to launch on: a raw handle, or None for the tensor's device's current one
bool stream_of(PyObject * o, const at::Tensor & t, void *& st) {
    if (o != Py_None) {
        st = PyLong_AsVoidPtr(o);
        return !PyErr_Occurred();
    }
    THPObjectPtr idx(PyLong_FromLong(t.device().index()));
    THPObjectPtr raw(idx ? PyObject_CallOneArg(lib.raw_stream, idx.get()) : nullptr);
    if (!raw) return false;
    st = PyLong_AsVoidPtr(raw.get());
    return !PyErr_Occurred();
}
// ggml-order sizes and byte strides of a tensor of up to 4 dimensions (last torch dimension = ggml dimension 0)
void nb4(const at::Tensor & t, int64_t ne[4], int64_t nb[4]) {
    const int d = (int) t.dim();
    const int64_t es = (int64_t) t.element_size();
    for (int i = 0; i < 4; i++) ne[i] = i < d ? t.size(d - 1 - i) : 1;
    for (int i = 0; i < 4; i++) nb[i] = i < d ? t.stride(d - 1 - i) * es : nb[i - 1] * ne[i - 1];
}
int64_t row_bytes(long kv_type) { return kv_type == MLA_TYPE_F16 || kv_type == MLA_TYPE_BF16 ? 1152 : kv_type == MLA_TYPE_Q8_0 ? 612 : -1; }

// The scratch area of (device, stream): a look-up in the Python layer's table; too small or missing, the Python layer makes one.  The
// caller keeps what is returned until its launch is queued: another thread may give areas back meanwhile.
THPObjectPtr workspace(PyObject * q, void * st, size_t need, mla_attn_args & a) {
    THPObjectPtr dev(PyObject_GetAttrString(q, "device")), handle(dev ? PyLong_FromVoidPtr(st) : nullptr);
    THPObjectPtr key(handle ? PyTuple_Pack(2, dev.get(), handle.get()) : nullptr);
    if (!key) return THPObjectPtr();
    PyObject * const found = PyDict_GetItemWithError(lib.workspaces, key.get());
    if (!found && PyErr_Occurred()) return THPObjectPtr();
    THPObjectPtr ws(Py_XNewRef(found));
    if (!ws || (size_t) THPVariable_Unpack(ws.get()).numel() < need) {
        THPObjectPtr n(PyLong_FromSize_t(need));
        ws = n ? PyObject_CallFunctionObjArgs(lib.workspace, dev.get(), n.get(), handle.get(), nullptr) : nullptr;
        if (!ws) return ws;
    }
    const at::Tensor * t = tensor(ws.get());
    if (!t) return THPObjectPtr();
    a.workspace = t->data_ptr(); a.workspace_size = (size_t) t->numel();
    return ws;
}

// attn(q, k, kv_type, dv, mask, scale, max_bias, logit_softcap, block_table, seq_lens, out, n_splits, flags, rows_per_wg, stream) -> out
PyObject * attn(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 15)) return nullptr;
    const at::Tensor * qp = tensor(v[0]), * kp = qp ? tensor(v[1]) : nullptr, * mask, * table, * lens, * outp;
    if (!kp || !optional_tensor(v[4], mask) || !optional_tensor(v[8], table) || !optional_tensor(v[9], lens) || !optional_tensor(v[10], outp)) return nullptr;
    const at::Tensor & q = *qp, & k = *kp;
    if (!on_gpu(q)) return nullptr;
    mla_attn_args a;
    memset(&a, 0, sizeof a);
    a.kv_type = (int32_t) PyLong_AsLong(v[2]); a.dv = (int32_t) PyLong_AsLong(v[3]);
    a.scale = (float) PyFloat_AsDouble(v[5]); a.max_bias = (float) PyFloat_AsDouble(v[6]); a.logit_softcap = (float) PyFloat_AsDouble(v[7]);
    a.n_splits = (int32_t) PyLong_AsLong(v[11]); a.flags = (uint32_t) PyLong_AsUnsignedLongMask(v[12]); a.rows_per_wg = (int32_t) PyLong_AsLong(v[13]);
    if (PyErr_Occurred()) return nullptr;
    REQUIRE(q.scalar_type() == at::kFloat && q.dim() == 4 && q.size(3) == 576 && q.stride(3) == 1);
    const int64_t row = row_bytes(a.kv_type), es = (int64_t) k.element_size();
    if (row < 0) { PyErr_SetObject(PyExc_KeyError, v[2]); return nullptr; }
    const int64_t n_seq = q.size(0), n_head = q.size(1), n_tok = q.size(2);
    a.n_seq = (int32_t) n_seq; a.n_head = (int32_t) n_head; a.n_tok = (int32_t) n_tok; a.dk = 576; a.q_type = MLA_TYPE_F32;
    a.q = q.data_ptr(); a.q_nb1 = q.stride(2) * 4; a.q_nb2 = q.stride(1) * 4; a.q_nb3 = q.stride(0) * 4;
    REQUIRE(k.dim() >= 1 && k.stride(-1) == 1 && k.size(-1) * es == row);
    a.kv = k.data_ptr();
    if (table) {
        REQUIRE(k.dim() == 2 && k.size(0) % PAGE == 0);
        a.kv_nb1 = k.stride(0) * es; a.n_kv = k.size(0);
        REQUIRE(table->scalar_type() == at::kInt && table->dim() == 2 && table->size(0) == n_seq && table->is_contiguous());
        REQUIRE(lens && lens->scalar_type() == at::kInt && lens->numel() == n_seq && lens->is_contiguous());
        a.block_table = (const int32_t *) table->data_ptr(); a.bt_stride = table->size(1); a.seq_lens = (const int32_t *) lens->data_ptr();
    } else {
        REQUIRE(k.dim() == 3 && (k.size(0) == 1 || k.size(0) == n_seq));
        a.kv_nb1 = k.stride(1) * es; a.kv_nb3 = k.size(0) > 1 ? k.stride(0) * es : 0; a.n_kv = k.size(1);
    }
    if (mask) {
        REQUIRE(mask->scalar_type() == at::kHalf && mask->dim() == 2 && mask->stride(1) == 1 && mask->size(0) >= n_tok);
        a.mask = mask->data_ptr(); a.mask_nb1 = mask->stride(0) * 2; a.mask_ne0 = mask->size(1);
    }
    at::Tensor made;
    if (!outp) {
        made = at::empty({ n_seq, n_tok, n_head, 576 }, q.options());
        outp = &made;
    }
    const at::Tensor & out = *outp;
    REQUIRE(out.scalar_type() == at::kFloat && out.dim() == 4 && out.is_contiguous() && out.size(0) == n_seq && out.size(1) == n_tok && out.size(2) == n_head && out.size(3) >= a.dv);
    a.dst = (float *) out.data_ptr(); a.dst_nb1 = out.size(3) * 4;
    void * st;
    if (!stream_of(v[14], q, st)) return nullptr;
    THPObjectPtr ws = workspace(v[0], st, lib.workspace_size(&a), a);
    if (!ws) return nullptr;
    const int rc = unlocked([&] { return lib.attn(&a, st); });
    if (rc) return failed("mla_attn_launch", rc);
    if (made.defined()) return THPVariable_Wrap(made);
    Py_INCREF(v[10]);
    return v[10];
}

// The argument block of an op of a batch: kept as bytes by the batch until it is launched.
PyObject * add_to_batch(PyObject * batch, int kind, const void * args, size_t size, PyObject * result) {
    THPObjectPtr k(PyLong_FromLong(kind)), b(PyBytes_FromStringAndSize((const char *) args, (Py_ssize_t) size)), name(PyUnicode_InternFromString("add"));
    if (!k || !b || !name) return nullptr;
    THPObjectPtr r(PyObject_CallMethodObjArgs(batch, name.get(), k.get(), b.get(), nullptr));
    return r ? Py_NewRef(result) : nullptr;
}

// values: pos, n_dims, mode, n_ctx_orig, freq_base, freq_scale, ext_factor, attn_factor, beta_fast, beta_slow, freq_factors
constexpr int N_ROPE = 11;
PyObject * fill_rope(mla_rope_args & a, const at::Tensor & x, const at::Tensor & out, PyObject * const * v, int64_t n_pos) {
    const at::Tensor * pos = tensor(v[0]), * ff;
    if (!pos || !optional_tensor(v[10], ff)) return nullptr;
    a.n_dims = (int32_t) PyLong_AsLong(v[1]); a.mode = (int32_t) PyLong_AsLong(v[2]); a.n_ctx_orig = (int32_t) PyLong_AsLong(v[3]);
    a.freq_base = (float) PyFloat_AsDouble(v[4]); a.freq_scale = (float) PyFloat_AsDouble(v[5]); a.ext_factor = (float) PyFloat_AsDouble(v[6]);
    a.attn_factor = (float) PyFloat_AsDouble(v[7]); a.beta_fast = (float) PyFloat_AsDouble(v[8]); a.beta_slow = (float) PyFloat_AsDouble(v[9]);
    if (PyErr_Occurred()) return nullptr;
    REQUIRE(pos->scalar_type() == at::kInt && pos->is_contiguous() && pos->numel() == n_pos);
    int64_t ne_out[4];
    nb4(x, a.ne, a.src_nb);
    nb4(out, ne_out, a.dst_nb);
    a.src = x.data_ptr(); a.dst = out.data_ptr(); a.pos = (const int32_t *) pos->data_ptr();
    if (ff) {
        REQUIRE(ff->scalar_type() == at::kFloat && ff->is_contiguous() && ff->numel() >= a.n_dims / 2);
        a.freq_factors = (const float *) ff->data_ptr();
    }
    return Py_None;   // (borrowed: anything but nullptr)
}

// rope(x, out, stream, batch, *values) -> out
PyObject * rope(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 4 + N_ROPE)) return nullptr;
    const at::Tensor * xp = tensor(v[0]), * outp;
    if (!xp || !optional_tensor(v[1], outp)) return nullptr;
    const at::Tensor & x = *xp;
    if (!on_gpu(x)) return nullptr;
    REQUIRE(x.scalar_type() == at::kFloat && x.dim() == 3 && x.stride(2) == 1);
    at::Tensor made;
    if (!outp) { made = at::empty(x.sizes(), x.options()); outp = &made; }
    const at::Tensor & out = *outp;
    REQUIRE(out.sizes() == x.sizes() && out.scalar_type() == at::kFloat && out.stride(2) == 1);
    mla_rope_args a;
    memset(&a, 0, sizeof a);
    if (!fill_rope(a, x, out, v + 4, x.size(0))) return nullptr;
    THPObjectPtr result(made.defined() ? THPVariable_Wrap(made) : Py_NewRef(v[1]));
    if (!result) return nullptr;
    if (v[3] != Py_None) return add_to_batch(v[3], MLA_FRONT_ROPE, &a, sizeof a, result.get());
    void * st;
    if (!stream_of(v[2], x, st)) return nullptr;
    const int rc = unlocked([&] { return lib.rope(&a, st); });
    if (rc) return failed("mla_rope_launch", rc);
    return result.release();
}

// mul_mat(w, w_type, x, out, stream, batch) -> out
PyObject * mul_mat(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 6)) return nullptr;
    const at::Tensor * wp = tensor(v[0]), * xp = wp ? tensor(v[2]) : nullptr, * outp;
    if (!xp || !optional_tensor(v[3], outp)) return nullptr;
    const at::Tensor & w = *wp, & x = *xp;
    if (!on_gpu(x)) return nullptr;
    REQUIRE(w.dim() == 3 && x.dim() == 3 && w.element_size() == 2 && x.scalar_type() == at::kFloat);
    REQUIRE(w.stride(2) == 1 && x.stride(2) == 1 && w.size(2) == x.size(2));
    at::Tensor made;
    if (!outp) { made = at::empty({ x.size(0), x.size(1), w.size(1) }, x.options()); outp = &made; }
    const at::Tensor & out = *outp;
    REQUIRE(out.dim() == 3 && out.size(0) == x.size(0) && out.size(1) == x.size(1) && out.size(2) == w.size(1) && out.scalar_type() == at::kFloat && out.stride(2) == 1);
    mla_mul_mat_args a;
    memset(&a, 0, sizeof a);
    a.w_type = (int32_t) PyLong_AsLong(v[1]);
    if (PyErr_Occurred()) return nullptr;
    a.w = w.data_ptr(); a.x = x.data_ptr(); a.dst = out.data_ptr();
    a.K = w.size(2); a.N = w.size(1); a.w_ne2 = w.size(0); a.w_ne3 = 1;
    a.M = x.size(1); a.ne2 = x.size(0); a.ne3 = 1;
    a.w_nb1 = w.stride(1) * 2; a.w_nb2 = w.stride(0) * 2; a.w_nb3 = a.w_nb2 * a.w_ne2;
    a.x_nb1 = x.stride(1) * 4; a.x_nb2 = x.stride(0) * 4; a.x_nb3 = a.x_nb2 * a.ne2;
    a.d_nb1 = out.stride(1) * 4; a.d_nb2 = out.stride(0) * 4; a.d_nb3 = a.d_nb2 * a.ne2;
    THPObjectPtr result(made.defined() ? THPVariable_Wrap(made) : Py_NewRef(v[3]));
    if (!result) return nullptr;
    if (v[5] != Py_None) return add_to_batch(v[5], MLA_FRONT_MUL_MAT, &a, sizeof a, result.get());
    void * st;
    if (!stream_of(v[4], x, st)) return nullptr;
    const int rc = unlocked([&] { return lib.mul_mat(&a, st); });
    if (rc) return failed("mla_mul_mat_launch", rc);
    return result.release();
}

// copy(src, dst, stream, batch) -> dst
PyObject * copy(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 4)) return nullptr;
    const at::Tensor * sp = tensor(v[0]), * dp = sp ? tensor(v[1]) : nullptr;
    if (!dp) return nullptr;
    const at::Tensor & src = *sp, & dst = *dp;
    if (!on_gpu(src)) return nullptr;
    REQUIRE(src.scalar_type() == at::kFloat && dst.scalar_type() == at::kFloat && src.sizes() == dst.sizes() && src.dim() >= 1 && src.dim() <= 4);
    REQUIRE(src.stride(-1) == 1 && dst.stride(-1) == 1);
    mla_copy_args a;
    memset(&a, 0, sizeof a);
    int64_t ne_dst[4];
    nb4(src, a.ne, a.src_nb);
    nb4(dst, ne_dst, a.dst_nb);
    a.src = src.data_ptr(); a.dst = dst.data_ptr();
    if (v[3] != Py_None) return add_to_batch(v[3], MLA_FRONT_COPY, &a, sizeof a, v[1]);
    void * st;
    if (!stream_of(v[2], src, st)) return nullptr;
    const int rc = unlocked([&] { return lib.copy(&a, st); });
    if (rc) return failed("mla_copy_f32_launch", rc);
    return Py_NewRef(v[1]);
}

// kv_write(src, cache, kv_type, row0, rows, block_table, seq_ids, positions, stream, batch, k_pe[, *rope values]) -> cache
PyObject * kv_write(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (n != 11 && !arg_count(n, 11 + N_ROPE)) return nullptr;
    const at::Tensor * sp = tensor(v[0]), * cp = sp ? tensor(v[1]) : nullptr, * rows, * table, * ids, * positions, * k_pe;
    if (!cp || !optional_tensor(v[4], rows) || !optional_tensor(v[5], table) || !optional_tensor(v[6], ids) || !optional_tensor(v[7], positions) || !optional_tensor(v[10], k_pe)) return nullptr;
    const at::Tensor & src = *sp, & cache = *cp;
    if (!on_gpu(src)) return nullptr;
    const bool with_rope = k_pe != nullptr;
    REQUIRE(with_rope == (n > 11));
    mla_kv_write_rope_args ra;
    memset(&ra, 0, sizeof ra);
    mla_kv_write_args & a = ra.w;
    REQUIRE(src.dim() == 2 && src.stride(1) == 1 && cache.dim() == 2 && cache.stride(1) == 1);
    if (with_rope) {
        REQUIRE(k_pe->scalar_type() == at::kFloat && k_pe->dim() == 2 && k_pe->size(0) == src.size(0) && k_pe->size(1) == 64 && k_pe->stride(1) == 1);
        if (!fill_rope(ra.rope, *k_pe, *k_pe, v + 11, src.size(0))) return nullptr;
        // [tokens, 64] is [tokens, 1 head, 64]
        ra.rope.ne[2] = ra.rope.ne[1]; ra.rope.ne[1] = 1;
        ra.rope.src_nb[2] = ra.rope.dst_nb[2] = ra.rope.src_nb[1];
        ra.rope.src_nb[3] = ra.rope.dst_nb[3] = ra.rope.src_nb[2] * ra.rope.ne[2];
    }
    a.n_tok = (int32_t) src.size(0);
    a.kv_type = (int32_t) PyLong_AsLong(v[2]);
    if (PyErr_Occurred()) return nullptr;
    const int64_t row = row_bytes(a.kv_type);
    if (row < 0) { PyErr_SetObject(PyExc_KeyError, v[2]); return nullptr; }
    const bool f32 = src.scalar_type() == at::kFloat;
    a.src_type = f32 ? MLA_TYPE_F32 : a.kv_type;
    REQUIRE(cache.size(1) * (int64_t) cache.element_size() == row);
    if (f32) REQUIRE(src.size(1) == 576 || (with_rope && src.size(1) >= 512));
    else     REQUIRE(src.size(1) * (int64_t) src.element_size() == row);
    a.src = src.data_ptr(); a.src_nb1 = src.stride(0) * (int64_t) src.element_size();
    a.kv = cache.data_ptr(); a.kv_nb1 = cache.stride(0) * (int64_t) cache.element_size(); a.n_kv_rows = cache.size(0);
    REQUIRE((v[3] != Py_None) + (rows != nullptr) + (table != nullptr) == 1);
    if (v[3] != Py_None) {
        a.row0 = PyLong_AsLongLong(v[3]);
        if (PyErr_Occurred()) return nullptr;
    } else if (rows) {
        REQUIRE((rows->scalar_type() == at::kInt || rows->scalar_type() == at::kLong) && rows->is_contiguous() && rows->numel() == a.n_tok);
        a.rows = rows->data_ptr(); a.rows_type = rows->scalar_type() == at::kLong ? 1 : 0;
    } else {
        REQUIRE(ids && positions);
        for (const at::Tensor * t : { table, ids, positions }) REQUIRE(t->scalar_type() == at::kInt && t->is_contiguous());
        REQUIRE(table->dim() == 2 && ids->numel() == a.n_tok && positions->numel() == a.n_tok);
        a.block_table = (const int32_t *) table->data_ptr(); a.bt_stride = table->size(1);
        a.seq_ids = (const int32_t *) ids->data_ptr(); a.positions = (const int32_t *) positions->data_ptr();
    }
    if (v[9] != Py_None) return with_rope ? add_to_batch(v[9], MLA_FRONT_KV_WRITE_ROPE, &ra, sizeof ra, v[1]) : add_to_batch(v[9], MLA_FRONT_KV_WRITE, &a, sizeof a, v[1]);
    void * st;
    if (!stream_of(v[8], src, st)) return nullptr;
    const int rc = unlocked([&] { return with_rope ? lib.kv_write_rope(&ra, st) : lib.kv_write(&a, st); });
    if (rc) return failed(with_rope ? "mla_kv_write_rope_launch" : "mla_kv_write_launch", rc);
    return Py_NewRef(v[1]);
}

struct Buffers {
    std::vector<Py_buffer> held;
    ~Buffers() { for (Py_buffer & b : held) PyBuffer_Release(&b); }
};

// front_batch(ops, stream): ops = [(kind, argument block: bytes or anything with a buffer), ...]
PyObject * front_batch(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 2)) return nullptr;
    REQUIRE(PyList_Check(v[0]));
    const Py_ssize_t count = PyList_GET_SIZE(v[0]);
    std::vector<mla_front_op> ops((size_t) std::max<Py_ssize_t>(count, 1));
    Buffers b;
    b.held.reserve((size_t) count);
    for (Py_ssize_t i = 0; i < count; i++) {
        PyObject * op = PyList_GET_ITEM(v[0], i);
        Py_buffer  buf;
        if (!PyTuple_Check(op) || PyTuple_GET_SIZE(op) != 2) {
            PyErr_SetString(PyExc_TypeError, "front_batch: ops are (kind, argument block) pairs");
            return nullptr;
        }
        if (PyObject_GetBuffer(PyTuple_GET_ITEM(op, 1), &buf, PyBUF_SIMPLE) != 0) return nullptr;
        b.held.push_back(buf);
        ops[(size_t) i] = mla_front_op{ (int32_t) PyLong_AsLong(PyTuple_GET_ITEM(op, 0)), 0, buf.buf };
        if (PyErr_Occurred()) return nullptr;
    }
    void * st = PyLong_AsVoidPtr(v[1]);
    if (PyErr_Occurred()) return nullptr;
    const int rc = unlocked([&] { return lib.front_batch(ops.data(), (int32_t) count, st); });
    if (rc) return failed("mla_front_batch_launch", rc);
    Py_RETURN_NONE;
}

// bind(addresses of the eight entry points in Bound's order, workspace function, workspace table, torch's raw current stream)
PyObject * bind(PyObject *, PyObject * const * v, Py_ssize_t n) {
    if (!arg_count(n, 11)) return nullptr;
    void * p[8];
    for (int i = 0; i < 8; i++) p[i] = PyLong_AsVoidPtr(v[i]);
    if (PyErr_Occurred()) return nullptr;
    REQUIRE(PyCallable_Check(v[8]) && PyDict_Check(v[9]) && PyCallable_Check(v[10]));
    lib.workspace_size = (decltype(lib.workspace_size)) p[0]; lib.attn = (decltype(lib.attn)) p[1];
    lib.kv_write = (decltype(lib.kv_write)) p[2]; lib.kv_write_rope = (decltype(lib.kv_write_rope)) p[3];
    lib.rope = (decltype(lib.rope)) p[4]; lib.mul_mat = (decltype(lib.mul_mat)) p[5];
    lib.copy = (decltype(lib.copy)) p[6]; lib.front_batch = (decltype(lib.front_batch)) p[7];
    lib.workspace = Py_NewRef(v[8]); lib.workspaces = Py_NewRef(v[9]); lib.raw_stream = Py_NewRef(v[10]);
    Py_RETURN_NONE;
}

template <PyObject * (*F)(PyObject *, PyObject * const *, Py_ssize_t)> PyObject * entry(PyObject * self, PyObject * const * v, Py_ssize_t n) {
    try {
        return F(self, v, n);
    } catch (...) {   // (what HANDLE_TH_ERRORS does, without its buffer for torch's warnings: none arise here)
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

#define FAST(name) { #name, (PyCFunction) (void (*)(void)) entry<name>, METH_FASTCALL, nullptr }
PyMethodDef methods[] = { FAST(bind), FAST(attn), FAST(rope), FAST(mul_mat), FAST(copy), FAST(kv_write), FAST(front_batch), { nullptr, nullptr, 0, nullptr } };
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
