// Host side of the Python view (vesper_amd/api.py) in native code: tensor descriptors, output allocation, workspaces
// and the calls into libvsp_attn.so, one Python -> C crossing per operator.
//
// What bounds it: the small calls of the path (one generated token, a short prompt) take 3 to 12 us of GPU time, and
// building the ctypes descriptors in Python took 5 to 8 us per tensor: 36 us for a token step of two operators (append
// + decode), the GPU idle for two thirds of it.  torch is used for what it was used for there: device memory (its
// caching allocator) and the current stream.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/vsp_attn.h"

namespace {

PyObject* g_error;       // vesper_amd.VspError(status)
PyObject* g_workspaces;  // the dict of what streams keep between calls that api.py owns (stream_workspace)

struct PyFailed {};  // a Python exception is set

[[noreturn]] void raise_status(int rc) {
    PyObject* code = PyLong_FromLong(rc);
    PyObject* e = code ? PyObject_CallOneArg(g_error, code) : nullptr;
    Py_XDECREF(code);
    if (e) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    throw PyFailed{};
}
// Every call into the library: a launch waits for room when a hardware queue is full, and the program's other Python threads
// run meanwhile (as they do during a call through ctypes).  One of them may replace this stream's workspace before the launch is in
// the queue, so the caller holds a reference to every tensor whose address is among the arguments.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class... P, class... A>
void call(int (*f)(P...), A... args) {
    int rc;
    {
        Unlocked unlocked;
        rc = f(args...);
    }
    if (rc != VSP_OK) raise_status(rc);
}
[[noreturn]] void raise_text(PyObject* type, const char* text) {
    PyErr_SetString(type, text);
    throw PyFailed{};
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) raise_text(PyExc_TypeError, "vesper_amd: expected a torch.Tensor");
    return THPVariable_Unpack(o);
}
double as_double(PyObject* o) {
    const double x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) throw PyFailed{};
    return x;
}
long long as_int(PyObject* o) {  // int(o): a NaN or infinite float is an error
    PyObject* n = PyLong_CheckExact(o) ? Py_NewRef(o) : PyNumber_Long(o);
    if (!n) throw PyFailed{};
    const long long x = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (x == -1 && PyErr_Occurred()) throw PyFailed{};
    return x;
}
int as_bool(PyObject* o) {
    const int x = PyObject_IsTrue(o);
    if (x < 0) throw PyFailed{};
    return x;
}
vsp_kv_cache* as_cache(PyObject* o) { return reinterpret_cast<vsp_kv_cache*>(as_int(o)); }

int dtype_of(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return VSP_F32;
        case at::kBFloat16: return VSP_BF16;
        case at::kHalf: return VSP_F16;
        case at::kChar: return VSP_I8;
        case at::kInt: return VSP_I32;
        default: raise_status(VSP_ERR_UNSUPPORTED);
    }
}
// Kernels are handed addresses: one of ordinary host memory would fault the GPU (pinned memory they can read).
const at::Tensor& reachable(const at::Tensor& t) {
    if (!t.is_cuda() && t.numel() > 0 && !(t.device().is_cpu() && t.is_pinned())) raise_text(PyExc_RuntimeError, "vesper_amd: expected a tensor on the GPU");
    return t;
}
vsp_tensor desc(const at::Tensor& t) {
    vsp_tensor d;
    d.data = reachable(t).data_ptr();
    d.dtype = dtype_of(t.scalar_type());
    const int n = (int)t.dim();
    d.ndim = n;  // more than 4: rejected by the library with the reference's message
    for (int i = 0; i < 4; ++i) {
        d.shape[i] = i < n ? t.size(i) : 0;
        d.stride[i] = i < n ? t.stride(i) : 0;
    }
    return d;
}

at::Tensor new_tensor(at::IntArrayRef shape, at::ScalarType dtype, at::Device device) {
    return at::Tensor(at::detail::empty_cuda(shape, dtype, device, c10::nullopt));
}
at::Tensor new_like(const at::Tensor& t) {
    if (t.is_contiguous() && t.is_cuda()) return new_tensor(t.sizes(), t.scalar_type(), t.device());
    return at::empty_like(t);
}
at::Tensor empty_bytes(size_t n, at::Device device) {
    const int64_t shape[1] = {(int64_t)(n < 16 ? 16 : n)};
    return new_tensor(at::IntArrayRef(shape, 1), at::kByte, device);
}

void* stream_of(const at::Tensor& t) {
    if (!t.is_cuda()) raise_text(PyExc_RuntimeError, "vesper_amd: expected a tensor on the GPU");
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}
const int32_t* device_ints(PyObject* o) { return o == Py_None ? nullptr : (const int32_t*)reachable(tensor(o)).data_ptr(); }

PyObject* tuple_of(std::initializer_list<at::Tensor> ts) {
    PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
    if (!r) throw PyFailed{};
    Py_ssize_t i = 0;
    for (const at::Tensor& t : ts) {
        PyObject* o = THPVariable_Wrap(t);
        if (!o) {
            Py_DECREF(r);
            throw PyFailed{};
        }
        PyTuple_SET_ITEM(r, i++, o);
    }
    return r;
}
// What a (device, stream) keeps between calls, in the dict that api.py owns; calls on different streams never share any.
//   ("cuda", device, stream) -> (workspace, counters).  The workspace is grow-only.  A captured graph keeps its address, so growth
//     during capture is refused, and a block that a capture was given outlives its replacement under ("held", device, address).  The
//     counters of the one-launch decode step are zero between calls.  Partials are written before they are read, wherever they
//     lie; counters are not, so they are never replaced.
constexpr size_t kCounters = 16384;
struct Workspace {
    at::Tensor block, counts;
    void* data() const { return block.data_ptr(); }
    size_t bytes() const { return (size_t)block.numel(); }
    uint32_t* counters() const { return (uint32_t*)counts.data_ptr(); }
};
PyObject* state_key(const char* what, at::Device device, const void* p) {
    PyObject* key = Py_BuildValue("(siK)", what, (int)device.index(), (unsigned long long)(uintptr_t)p);
    if (!key) throw PyFailed{};
    return key;
}
void state_set(PyObject* key, PyObject* value) {  // takes both references
    const int rc = value ? PyDict_SetItem(g_workspaces, key, value) : -1;
    Py_XDECREF(value);
    Py_DECREF(key);
    if (rc < 0) throw PyFailed{};
}
// optional: room that a call can do without; in a capture that it would have to grow for, none is given (the returned block is not defined)
Workspace stream_workspace(at::Device device, void* stream, size_t nbytes, bool optional = false) {
    PyObject* key = state_key("cuda", device, stream);
    PyObject* have = PyDict_GetItemWithError(g_workspaces, key);  // borrowed
    Py_DECREF(key);
    if (!have && PyErr_Occurred()) throw PyFailed{};
    Workspace w;
    if (have) w.block = tensor(PyTuple_GET_ITEM(have, 0)), w.counts = tensor(PyTuple_GET_ITEM(have, 1));
    const bool fits = have && w.bytes() >= nbytes;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;  // the null stream cannot be captured
    if (stream && hipStreamIsCapturing((hipStream_t)stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone) {
        if (!fits && optional) return Workspace{};
        if (!fits)
            raise_text(PyExc_RuntimeError,
                       "decode_attention: the workspace would have to grow during stream capture; "
                       "run one eager call of this size first, or pass workspace=");
        state_set(state_key("held", device, w.data()), THPVariable_Wrap(w.block));
    } else if (!fits) {
        if (!have) {
            const int64_t n[1] = {(int64_t)kCounters};
            w.counts = new_tensor(at::IntArrayRef(n, 1), at::kInt, device);
            w.counts.zero_();
        }
        w.block = empty_bytes(nbytes, device);
        state_set(state_key("cuda", device, stream), tuple_of({w.block, w.counts}));
    }
    return w;
}

PyObject* out_and_lse(const at::Tensor& out, const at::Tensor& lse, bool both) {
    return both ? tuple_of({out, lse}) : THPVariable_Wrap(out);
}
// Workspace of n bytes for the attention of several tokens over a cache.  Partials of a split context alone go to the per-stream block the decode step uses, or
// nowhere: a capture that the block would have to grow for records the call unsplit.  A quantised cache's dequantised rows are needed, grow with the batch's
// contexts and are given back after the call.
at::Tensor context_workspace(const vsp_kv_cache* c, const at::Tensor& q, void* st, size_t n) {
    if (!n) return at::Tensor();
    return c->format == VSP_KV_Q8_0 ? empty_bytes(n, q.device()) : stream_workspace(q.device(), st, n, true).block;
}
at::Tensor lse_for(const at::Tensor& q) { return new_tensor(q.sizes().slice(0, 3), at::kFloat, q.device()); }

// ---- operators: arguments are positional, defaults and keyword handling live in api.py -------------------------------

// flash(q, k, v, scale, is_causal, dropout_p, training, return_lse)
PyObject* flash(PyObject* const* a) {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    if (!(q.is_cuda() && k.is_cuda() && v.is_cuda()))
        raise_text(PyExc_RuntimeError, "flash_attention: unsupported device");  // src/ops/flash_attention.cpp:111-112
    const bool want_lse = as_bool(a[7]);
    vsp_tensor dq = desc(q), dk = desc(k), dv = desc(v);
    at::Tensor out = new_tensor(q.sizes(), q.scalar_type(), q.device()), lse;
    vsp_tensor dout = desc(out), dl;
    if (want_lse && q.dim() == 4) {
        lse = lse_for(q);
        dl = desc(lse);
    }
    call(vsp_attn_prefill, &dq, &dk, &dv, &dout, lse.defined() ? &dl : nullptr, (float)as_double(a[3]), as_bool(a[4]),
         (float)as_double(a[5]), as_bool(a[6]), stream_of(q));
    return out_and_lse(out, lse, want_lse);
}

// flash_split(q, k, v, scale, is_causal, return_lse, workspace | None)
PyObject* flash_split(PyObject* const* a) {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const bool want_lse = as_bool(a[5]);
    vsp_tensor dq = desc(q), dk = desc(k), dv = desc(v);
    void* st = stream_of(q);
    at::Tensor out = new_tensor(q.sizes(), q.scalar_type(), q.device()), lse, ws;
    vsp_tensor dout = desc(out), dl;
    if (want_lse && q.dim() == 4) {
        lse = lse_for(q);
        dl = desc(lse);
    }
    if (a[6] != Py_None) ws = reachable(tensor(a[6]));
    else
        ws = empty_bytes(q.dim() == 4 && k.dim() == 4
                             ? vsp_attn_prefill_split_workspace_bytes((int)q.size(0), (int)q.size(1), (int)k.size(1), (int)q.size(2),
                                                                      (int)k.size(2), (int)q.size(3))
                             : 0,
                         q.device());
    call(vsp_attn_prefill_split, &dq, &dk, &dv, &dout, lse.defined() ? &dl : nullptr, (float)as_double(a[3]), as_bool(a[4]),
         ws.data_ptr(), (size_t)ws.numel(), st);
    return out_and_lse(out, lse, want_lse);
}

// backward(dout, q, k, v, out, lse, scale, is_causal, workspace | None, split)
PyObject* backward(PyObject* const* a) {
    const at::Tensor &q = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]);
    const bool split = as_bool(a[9]);
    void* st = stream_of(q);
    at::Tensor dq = new_like(q), dk = new_like(k), dv = new_like(v), ws;
    vsp_tensor d[9];
    for (int i = 0; i < 6; ++i) d[i] = desc(tensor(a[i]));
    d[6] = desc(dq), d[7] = desc(dk), d[8] = desc(dv);
    if (a[8] != Py_None) ws = reachable(tensor(a[8]));
    else {
        size_t n = 0;
        if (q.dim() == 4 && k.dim() == 4) {
            const int B = (int)q.size(0), Hq = (int)q.size(1), Hkv = (int)k.size(1), N = (int)q.size(2), D = (int)q.size(3);
            n = split ? vsp_attn_backward_split_workspace_bytes(B, Hq, Hkv, N, D) : vsp_attn_backward_workspace_bytes(B, Hq, N);
            if (split || q.scalar_type() == at::kBFloat16) n = std::max(n, vsp_attn_backward_parts_workspace_bytes(B, Hq, Hkv, N, D, as_bool(a[7]), split));
        }
        ws = empty_bytes(n, q.device());
    }
    // a caller's workspace selects the bf16 path by its size
    auto f = split ? vsp_attn_prefill_backward_split : a[8] != Py_None ? vsp_attn_prefill_backward : vsp_attn_prefill_backward_parts;
    call(f, &d[0], &d[1], &d[2], &d[3], &d[4], &d[5], &d[6], &d[7], &d[8], (float)as_double(a[6]), as_bool(a[7]), ws.data_ptr(),
         (size_t)ws.numel(), st);
    return tuple_of({dq, dk, dv});
}

// update(cache, new_k, new_v, start_pos, start_pos_dev | None)
PyObject* update(PyObject* const* a) {
    const at::Tensor &k = tensor(a[1]), &v = tensor(a[2]);
    vsp_tensor dk = desc(k), dv = desc(v);
    call(vsp_kv_append, as_cache(a[0]), &dk, &dv, as_int(a[3]), device_ints(a[4]), stream_of(k));
    Py_RETURN_NONE;
}

// rope_update(cache, q, new_k, new_v, start_pos, table, table_len, out | None, out_dtype | None, start_pos_dev | None)
PyObject* rope_update(PyObject* const* a) {
    const at::Tensor &q = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]), &table = reachable(tensor(a[5]));
    void* st = stream_of(q);
    at::Tensor out;
    if (a[7] != Py_None) out = tensor(a[7]);
    else {
        at::ScalarType dt = q.scalar_type();
        if (a[8] != Py_None) {
            if (!THPDtype_Check(a[8])) raise_text(PyExc_TypeError, "vesper_amd: expected a torch.dtype");
            dt = ((THPDtype*)a[8])->scalar_type;
        }
        out = new_tensor(q.sizes(), dt, q.device());
    }
    vsp_tensor dq = desc(q), dk = desc(k), dv = desc(v), dout = desc(out);
    call(vsp_rope_kv_append, as_cache(a[0]), &dq, &dk, &dv, &dout, (const float*)table.data_ptr(), as_int(a[6]), as_int(a[4]),
         device_ints(a[9]), st);
    return THPVariable_Wrap(out);
}

// prefill(cache, q, seq_lens | None, max_len, chunk_lens | None, scale, is_causal, return_lse, split)
PyObject* prefill(PyObject* const* a) {
    vsp_kv_cache* c = as_cache(a[0]);
    const at::Tensor& q = tensor(a[1]);
    const int32_t *lens = device_ints(a[2]), *chunks = device_ints(a[4]);
    const int max_len = (int)as_int(a[3]);
    const bool want_lse = as_bool(a[7]);
    void* st = stream_of(q);
    vsp_tensor dq = desc(q), dl;
    at::Tensor out = new_like(q), lse, ws;
    vsp_tensor dout = desc(out);
    if (want_lse) {
        lse = lse_for(q);
        dl = desc(lse);
    }
    // a few queries over a long context: with room for partials the context is split over workgroups
    const size_t n = as_bool(a[8]) && q.dim() == 4 ? vsp_attn_prefill_cached_best_workspace_bytes(c, lens != nullptr, max_len, (int)q.size(1), (int)q.size(2))
                                                   : vsp_attn_prefill_cached_workspace_bytes(c, lens != nullptr, max_len);
    ws = context_workspace(c, q, st, n);
    call(vsp_attn_prefill_cached, &dq, c, lens, max_len, chunks, &dout, want_lse ? &dl : nullptr, (float)as_double(a[5]), as_bool(a[6]),
         ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? n : 0, st);
    return out_and_lse(out, lse, want_lse);
}

// decode(cache, q, seq_lens | None, max_len, scale, out | None, workspace | None, kind): kind 0 one token per sequence,
// 1 several, 2 one token with the library's own scratch
PyObject* decode(PyObject* const* a) {
    vsp_kv_cache* c = as_cache(a[0]);
    const at::Tensor& q = tensor(a[1]);
    const int32_t* lens = device_ints(a[2]);
    const int max_len = (int)as_int(a[3]);
    const long kind = (long)as_int(a[7]);
    void* st = stream_of(q);
    at::Tensor out = a[5] != Py_None ? tensor(a[5]) : new_like(q);
    vsp_tensor dq = desc(q), dout = desc(out);
    const float scale = (float)as_double(a[4]);
    if (kind == 2) {
        call(vsp_attn_decode_noalloc, &dq, c, lens, max_len, &dout, scale, st);
        return THPVariable_Wrap(out);
    }
    if (a[6] != Py_None || q.dim() != 4) {
        at::Tensor ws;
        if (a[6] != Py_None) ws = reachable(tensor(a[6]));
        auto f = kind == 1 ? vsp_attn_decode_multi : vsp_attn_decode;
        call(f, &dq, c, lens, max_len, &dout, scale, ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? (size_t)ws.numel() : 0, st);
        return THPVariable_Wrap(out);
    }
    if (kind == 0 && q.size(2) != 1) raise_status(VSP_ERR_SHAPE);
    const int bound = max_len ? max_len : (lens ? c->S_max : c->len);
    const Workspace ws = stream_workspace(
        q.device(), st, vsp_attn_decode_workspace_bytes((int)(q.size(0) * q.size(2)), (int)q.size(1), (int)q.size(3), bound > 1 ? bound : 1));
    call(vsp_attn_decode_counted, &dq, c, lens, max_len, &dout, scale, ws.data(), ws.bytes(), ws.counters(), kCounters, st);
    return THPVariable_Wrap(out);
}

// What the one-call steps take: everything where q is.  Other operands go through rope_update / update, which take or refuse them.
bool beside(const at::Tensor& q, std::initializer_list<const at::Tensor*> ts) {
    if (!q.is_cuda()) return false;
    for (const at::Tensor* t : ts)
        if (t->defined() && t->device() != q.device()) return false;
    return true;
}

// token_step(cache, q, new_k, new_v, start_pos, table | None, table_len, scale): append and attention of one token per sequence in one
// launch; None, with nothing done, where the library leaves the call to rope_update / update and decode
PyObject* token_step(PyObject* const* a) {
    vsp_kv_cache* c = as_cache(a[0]);
    const at::Tensor &q = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]);
    const long long start = as_int(a[4]);
    const at::Tensor table = a[5] != Py_None ? tensor(a[5]) : at::Tensor();
    if (q.dim() != 4 || q.numel() == 0 || !beside(q, {&k, &v, &table}) || start < 0 || start >= c->S_max) Py_RETURN_NONE;
    void* st = stream_of(q);
    at::Tensor out = new_tensor(q.sizes(), q.scalar_type(), q.device());
    vsp_tensor dq = desc(q), dk = desc(k), dv = desc(v), dout = desc(out);
    const Workspace ws = stream_workspace(
        q.device(), st, vsp_attn_token_step_workspace_bytes((int)q.size(0), (int)q.size(1), (int)q.size(3), (int)start));
    const long long table_len = as_int(a[6]);
    const float scale = (float)as_double(a[7]);
    int rc;
    {
        Unlocked unlocked;
        rc = vsp_attn_token_step(c, &dq, &dk, &dv, table.defined() ? (const float*)table.data_ptr() : nullptr, table_len, start, &dout, scale,
                                 ws.data(), ws.bytes(), ws.counters(), kCounters, st);
    }
    if (rc == VSP_ERR_LAUNCH) raise_status(rc);
    if (rc != VSP_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
}

// prompt_step(cache, q, new_k, new_v, start_pos, table, table_len, scale): a prompt's rows into an empty cache and its attention, Q rotated
// in the attention (fp32 caches: in the append); None, with nothing done, where the library leaves the call to rope_update and prefill
PyObject* prompt_step(PyObject* const* a) {
    vsp_kv_cache* c = as_cache(a[0]);
    const at::Tensor &q = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]), &table = tensor(a[5]);
    if (q.dim() != 4 || q.numel() == 0 || !beside(q, {&k, &v, &table}) || as_int(a[4]) != 0 || q.size(2) > c->S_max) Py_RETURN_NONE;
    void* st = stream_of(q);
    at::Tensor out = new_tensor(q.sizes(), q.scalar_type(), q.device()), ws;
    vsp_tensor dq = desc(q), dk = desc(k), dv = desc(v), dout = desc(out);
    if (c->format == VSP_KV_F32) {
        // append with Q rotated, then the attention over the planes: the launches of rope_update and flash_attention over views(), without the views and their
        // descriptors.  Short fp32 prompts wait for the host: 32 / 8 heads, 16 tokens 13.9 -> 9.1 us
        if (q.scalar_type() != at::kFloat || c->len > q.size(2) || q.size(0) != c->B || q.size(3) != c->D || c->D > 256 || c->Hkv <= 0 || q.size(1) % c->Hkv != 0 || c->page_table)
            Py_RETURN_NONE;
        at::Tensor rotated = new_tensor(q.sizes(), at::kFloat, q.device());
        vsp_tensor dr = desc(rotated);
        const long long table_len = as_int(a[6]);
        const float scale = (float)as_double(a[7]);
        int rc;
        {
            Unlocked unlocked;
            rc = vsp_rope_kv_append(c, &dq, &dk, &dv, &dr, (const float*)table.data_ptr(), table_len, 0, nullptr, st);
            if (rc == VSP_OK) rc = vsp_attn_prefill_cached(&dr, c, nullptr, 0, nullptr, &dout, nullptr, scale, 1, nullptr, 0, st);
        }
        if (rc != VSP_OK) raise_status(rc);
        return THPVariable_Wrap(out);
    }
    const size_t n = vsp_attn_prefill_cached_best_workspace_bytes(c, 0, (int)q.size(2), (int)q.size(1), (int)q.size(2));
    ws = context_workspace(c, q, st, n);
    const long long table_len = as_int(a[6]);
    const float scale = (float)as_double(a[7]);
    int rc;
    {
        Unlocked unlocked;
        rc = vsp_attn_prompt_step(c, &dq, &dk, &dv, (const float*)table.data_ptr(), table_len, &dout, scale, ws.defined() ? ws.data_ptr() : nullptr,
                                  ws.defined() ? n : 0, st);
    }
    if (rc == VSP_ERR_UNSUPPORTED) Py_RETURN_NONE;
    if (rc != VSP_OK) raise_status(rc);
    return THPVariable_Wrap(out);
}

// decode_proj(cache, q, wo, bias | None, seq_lens | None, max_len, scale, out | None, workspace | None)
PyObject* decode_proj(PyObject* const* a) {
    vsp_kv_cache* c = as_cache(a[0]);
    const at::Tensor &q = tensor(a[1]), &wo = tensor(a[2]);
    const int32_t* lens = device_ints(a[4]);
    const int max_len = (int)as_int(a[5]);
    void* st = stream_of(q);
    at::Tensor out, ws;
    if (a[7] != Py_None) out = tensor(a[7]);
    else {
        const int64_t shape[3] = {q.size(0), 1, wo.size(0)};
        out = new_tensor(at::IntArrayRef(shape, 3), q.scalar_type(), q.device());
    }
    if (a[8] != Py_None) ws = reachable(tensor(a[8]));
    else {
        const int bound = max_len ? max_len : (lens ? c->S_max : c->len);
        ws = stream_workspace(q.device(), st,
                              vsp_attn_decode_proj_workspace_bytes((int)q.size(0), (int)q.size(1), (int)q.size(3), bound > 1 ? bound : 1,
                                                                   (int)wo.size(0))).block;
    }
    vsp_tensor dq = desc(q), dw = desc(wo), dy = desc(out), db;
    if (a[3] != Py_None) db = desc(tensor(a[3]));
    call(vsp_attn_decode_proj, &dq, c, lens, max_len, &dw, a[3] != Py_None ? &db : nullptr, &dy, (float)as_double(a[6]), ws.data_ptr(),
         (size_t)ws.numel(), st);
    return THPVariable_Wrap(out);
}

// advance(seq_lens, n_new | None, T, B, S_max)
PyObject* advance(PyObject* const* a) {
    const at::Tensor& lens = tensor(a[0]);
    call(vsp_seq_lens_advance, (int32_t*)lens.data_ptr(), device_ints(a[1]), (int)as_int(a[2]), (int)as_int(a[3]), (int)as_int(a[4]),
         stream_of(lens));
    Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    try {
        return F(args);
    } catch (const PyFailed&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// bind(VspError, workspaces dict)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2 || !PyDict_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "bind(error class, dict)");
        return nullptr;
    }
    Py_INCREF(args[0]);
    Py_INCREF(args[1]);
    Py_XDECREF(g_error);
    Py_XDECREF(g_workspaces);
    g_error = args[0];
    g_workspaces = args[1];
    Py_RETURN_NONE;
}

#define VSP_ENTRY(f, n) {#f, (PyCFunction)(void (*)(void))entry<f, n>, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                          VSP_ENTRY(flash, 8),
                          VSP_ENTRY(flash_split, 7),
                          VSP_ENTRY(backward, 10),
                          VSP_ENTRY(update, 5),
                          VSP_ENTRY(rope_update, 10),
                          VSP_ENTRY(prefill, 9),
                          VSP_ENTRY(decode, 8),
                          VSP_ENTRY(token_step, 8),
                          VSP_ENTRY(prompt_step, 8),
                          VSP_ENTRY(decode_proj, 9),
                          VSP_ENTRY(advance, 5),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }
