// ops_binding.cpp - the torch-facing calls of ops.py in native code: a CPython module over the C ABI.
//
// Each function takes the tensors of a well-formed call straight to the C entry: the same checks as ops.py's Python
// path, which stays the one that reports an ill-formed call. A function returns None when any check fails or a tensor
// is not a plain torch.Tensor (subclasses, tracing and fake tensors); ops.py then runs its Python path, which raises the
// error or serves the call. Building the ctypes structures and reading the tensors from Python cost 17 us per attention
// call and ~12 us per quantiser call, more than most kernels take; here a call costs its launches.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/hip/HIPFunctions.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <map>
#include <optional>
#include <utility>

#include "../../include/fmha_mxfp8.h"
#include "../../include/mxfp8_quant.h"

namespace {

constexpr int64_t kD = 128;

// A plain device tensor, or nullptr.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg()) return nullptr;
    return &t;
}

uint64_t cap(const at::Tensor& t) { return t.storage().nbytes() - (uint64_t)t.storage_offset() * t.element_size(); }

bool is4(const at::Tensor& t, int64_t a, int64_t b, int64_t c, int64_t d, int64_t esize, uintptr_t align = 1) {
    return t.dim() == 4 && t.size(0) == a && t.size(1) == b && t.size(2) == c && t.size(3) == d && t.element_size() == esize &&
           t.is_contiguous() && (uintptr_t)t.data_ptr() % align == 0;
}

// Makes a device current for the calls of the library (which act on the current device).
struct OnDevice {
    explicit OnDevice(int dev) : prev(c10::hip::current_device()), dev(dev) {
        if (prev != dev) c10::hip::set_device((c10::DeviceIndex)dev);
    }
    ~OnDevice() {
        if (prev != dev) (void)hipSetDevice(prev);
    }
    int prev, dev;
};

// An allocation by this thread is no part of any capture, and does not disturb one that another thread has under way.
struct RelaxedCapture {
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
};

// Whether the allocation lies in a pool that torch keeps apart from the ordinary ones (a graph's, while torch captures it).
// Allocators that cannot tell have none that is known here.
bool in_private_pool(const void* ptr) {
    const size_t a = (size_t)(uintptr_t)ptr;
    try {
        for (const auto& s : c10::hip::HIPCachingAllocator::get()->snapshot().segments)
            if (a >= s.address && a < s.address + s.total_size) return s.owner_private_pool_id.first != 0 || s.owner_private_pool_id.second != 0;
    } catch (const std::exception&) {
    }
    return false;
}

// The attention's workspace: memory of one call, from torch's caching allocator by the call's stream, so that its earlier users are
// work on that stream, and so are its next ones. Nothing is kept between calls and no two callers share a buffer. (The
// allocator hands consecutive calls of a stream the same block, whose slots they then take in turn.)
// Under a capture by torch the block is the graph's own, from its pool. Under any other capture nobody owns the memory that
// the graph will use on each replay, so it is allocated for that capture and stream, and stays allocated.
// hipStreamPerThread is one handle for a stream of each thread, which the allocator cannot tell apart. Its calls take memory
// of torch's current stream and wait for the work queued there, and the allocator hands the block out again behind this
// thread's stream.
class Scratch {
  public:
    // Throws torch's out-of-memory error.
    Scratch(size_t bytes, hipStream_t stream, int dev) {
        RelaxedCapture relaxed;
        unsigned long long id = capture_of(stream);
        if (stream == hipStreamPerThread) {
            const c10::hip::HIPStream cur = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev);
            if (!id) id = capture_of(cur.stream());   // (nothing of the current stream's can be waited for then)
            if (id) {
                ptr = of_capture(id, stream, bytes);
                return;
            }
            data_ = c10::hip::HIPCachingAllocator::get()->allocate(bytes);
            ptr = data_.get();
            c10::hip::HIPCachingAllocator::recordStream(data_, c10::hip::getStreamFromExternal(stream, (c10::DeviceIndex)dev));
            hipEvent_t ev;
            C10_HIP_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
            const hipError_t e0 = hipEventRecord(ev, cur.stream()), e1 = hipStreamWaitEvent(stream, ev, 0);
            (void)hipEventDestroy(ev);
            C10_HIP_CHECK(e0);
            C10_HIP_CHECK(e1);
            return;
        }
        own_ = c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, stream);
        ptr = own_;
        if (id && !in_private_pool(own_)) {
            release();
            ptr = of_capture(id, stream, bytes);
        }
    }
    ~Scratch() { release(); }
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    void* ptr = nullptr;

  private:
    // One more than the id of the capture that the stream takes part in, or 0.
    static unsigned long long capture_of(hipStream_t stream) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        if (hipStreamGetCaptureInfo(stream, &st, &id) != hipSuccess) (void)hipGetLastError();   // (the legacy stream, while another captures)
        else if (st == hipStreamCaptureStatusActive) return id + 1u;
        return 0;
    }
    void release() {
        if (own_) c10::hip::HIPCachingAllocator::raw_delete(own_);
        own_ = nullptr;
    }
    // Called with the GIL held (which guards the map).
    static void* of_capture(unsigned long long id, hipStream_t stream, size_t bytes) {
        static auto* held = new std::map<std::pair<unsigned long long, hipStream_t>, std::pair<void*, size_t>>;
        auto& h = (*held)[{id, stream}];
        if (h.second < bytes) {
            void* p = nullptr;
            if (hipMalloc(&p, bytes) != hipSuccess) {
                (void)hipGetLastError();
                TORCH_CHECK_WITH(OutOfMemoryError, false, "no memory for a captured call's workspace (", bytes, " bytes)");
            }
            h = {p, bytes};
        }
        return h.first;
    }
    void* own_ = nullptr;
    at::DataPtr data_;
};

void* stream_of(PyObject* o, int dev, bool& ok) {
    if (o == Py_None) return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA((c10::DeviceIndex)dev).stream();
    if (!PyLong_Check(o)) {
        ok = false;
        return nullptr;
    }
    void* s = PyLong_AsVoidPtr(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        ok = false;
    }
    return s;
}

PyObject* fmha_error = nullptr;   // lib.FmhaError

PyObject* raise_code(int rc, const char* msg) {
    PyObject* e = PyObject_CallFunction(fmha_error, "is", rc, msg);
    if (e) {
        PyErr_SetObject(fmha_error, e);
        Py_DECREF(e);
    }
    return nullptr;
}

PyObject* decline() { Py_RETURN_NONE; }

// The one-call entry with its workspace -> (path, splits, partials). Called with the GIL held.
PyObject* run_params(fmha_mxfp8_params& p, int dev, void* stream) {
    static thread_local uint32_t turn = 0;   // which slots: any will do
    int32_t parts = 0;
    int path = -1, splits = 0, rc;
    p.partials_out = &parts;
    p.ws_turn = &turn;
    char err[512] = "";
    {
        OnDevice on(dev);
        // room for the entry's workspace slots (consecutive calls then write partials the previous combine did not just
        // read), unless that would take more than 512 MiB
        const size_t one = fmha_mxfp8_auto_workspace_bytes(&p);
        size_t bytes = one;
        const size_t slotted = FMHA_WORKSPACE_SLOTS * ((bytes + 255) / 256 * 256);
        if (slotted <= (512u << 20)) bytes = slotted;
        std::optional<Scratch> ws;
        std::exception_ptr oom;
        for (const size_t n : {bytes, one}) {
            if (ws || !n || (oom && n == bytes)) continue;
            try {
                ws.emplace(n, (hipStream_t)stream, dev);
                bytes = n;
            } catch (const c10::OutOfMemoryError&) {
                oom = std::current_exception();
            }
        }
        if (!ws) bytes = 0;   // the full-sequence paths then run their own kernels, which take none
        Py_BEGIN_ALLOW_THREADS
        rc = fmha_fwd_hd128_mxfp8_auto_ws(&p, ws ? ws->ptr : nullptr, bytes, stream, &path, &splits, err, sizeof(err));
        Py_END_ALLOW_THREADS
        if (rc == FMHA_ERR_WORKSPACE && oom) std::rethrow_exception(oom);
    }
    if (rc != FMHA_OK) return raise_code(rc, err);
    PyObject* r = PyTuple_New(3);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, PyLong_FromLong(path));
    PyTuple_SET_ITEM(r, 1, PyLong_FromLong(splits));
    PyTuple_SET_ITEM(r, 2, PyLong_FromLong(parts));
    return r;
}

// attend(q, k, v, q_scale, k_scale, v_scale, out, lse, path, splits, causal, f32_partials, softmax_scale, no_check,
//        causal_pair, kv_fill, stream) -> (path, splits, partials), or None
PyObject* attend_impl(PyObject* const* a, Py_ssize_t n) {
    if (n != 17) return decline();
    const at::Tensor* t[8] = {};
    for (int i = 0; i < 8; ++i) {
        if (i == 7 && a[7] == Py_None) break;
        if (!(t[i] = plain(a[i]))) return decline();
    }
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &qs = *t[3], &ks = *t[4], &vs = *t[5], &out = *t[6];
    if (q.dim() != 4 || k.dim() != 4) return decline();
    const int64_t B = q.size(0), S = q.size(1), H = q.size(2), SK = k.size(1), HK = k.size(2);
    if (q.size(3) != kD || k.size(3) != kD || HK < 1 || H < 1 || H % HK || ((H / HK) & (H / HK - 1)) || H / HK > 16) return decline();
    if (B > INT32_MAX || S > INT32_MAX || H > INT32_MAX || SK > INT32_MAX) return decline();
    const bool seq32 = vs.scalar_type() == at::kByte && vs.dim() == 4;
    if (!is4(q, B, S, H, kD, 1) || !is4(k, B, SK, HK, kD, 1) || !is4(v, B, SK, HK, kD, 1) || !is4(qs, B, S, H, 4, 1, 4) ||
        !is4(ks, B, SK, HK, 4, 1, 4) || !is4(out, B, S, H, kD, 2))
        return decline();
    if (seq32 ? !is4(vs, B, (SK + 31) / 32, HK, kD, 1) : cap(vs) < 4) return decline();
    if (t[7]) {
        const at::Tensor& l = *t[7];
        if (l.dim() != 3 || l.size(0) != B || l.size(1) != H || l.size(2) != S || l.element_size() != 4 || !l.is_contiguous()) return decline();
    }
    fmha_mxfp8_params p;
    std::memset(&p, 0, sizeof(p));
    const int dev = q.device().index();
    bool ok = true;
    void* stream = stream_of(a[16], dev, ok);
    const double scale = PyFloat_AsDouble(a[12]);
    int32_t iv[16] = {};
    for (int i : {8, 9, 10, 11, 13, 14, 15}) iv[i] = (int32_t)PyLong_AsLong(a[i]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return decline();
    }
    if (!ok) return decline();
    p.o = out.data_ptr(); p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr();
    p.q_descale = qs.data_ptr(); p.k_descale = ks.data_ptr(); p.v_descale = vs.data_ptr();
    p.lse = t[7] ? t[7]->data_ptr() : nullptr;
    p.bytes_q = cap(q); p.bytes_k = cap(k); p.bytes_v = cap(v); p.bytes_o = cap(out);
    p.bytes_q_descale = cap(qs); p.bytes_k_descale = cap(ks); p.bytes_v_descale = cap(vs);
    p.B = (int32_t)B; p.H = (int32_t)H; p.HK = (int32_t)HK; p.S = (int32_t)S; p.SK = (int32_t)SK;
    p.path = iv[8]; p.splits = iv[9]; p.causal = iv[10]; p.f32_partials = iv[11];
    p.v_seq32 = seq32 ? 1 : 0;
    p.softmax_scale = (float)scale;
    p.no_check = iv[13]; p.causal_pair = iv[14]; p.kv_fill = iv[15];
    return run_params(p, dev, stream);
}

// A bf16 tensor the quantisers can read as it is.
const at::Tensor* plain_bf16(PyObject* o) {
    const at::Tensor* x = plain(o);
    return x && x->scalar_type() == at::kBFloat16 && x->is_contiguous() && x->numel() > 0 ? x : nullptr;
}

// quantize_rows(x, scale_out, mul, stream) -> q, or None
PyObject* quantize_rows_impl(PyObject* const* a, Py_ssize_t n) {
    if (n != 4) return decline();
    const at::Tensor *x = plain_bf16(a[0]), *sc = x ? plain(a[1]) : nullptr;
    if (!x || !sc || x->dim() < 1 || x->size(-1) != kD || sc->dim() != x->dim() || sc->size(-1) != 4 || sc->element_size() != 1 ||
        !sc->is_contiguous() || (uintptr_t)sc->data_ptr() % 4)
        return decline();
    for (int64_t i = 0; i + 1 < x->dim(); ++i)
        if (x->size(i) != sc->size(i)) return decline();
    const int dev = x->device().index();
    bool ok = true;
    void* stream = stream_of(a[3], dev, ok);
    const double mul = PyFloat_AsDouble(a[2]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return decline();
    }
    if (!ok) return decline();
    char err[512] = "";
    int rc;
    at::Tensor q;
    {
        OnDevice on(dev);
        q = at::empty(x->sizes(), x->options().dtype(at::kByte));
        Py_BEGIN_ALLOW_THREADS
        rc = fmha_mxfp8_quantize_rows(x->data_ptr(), q.data_ptr(), sc->data_ptr(), x->numel() / kD, (float)mul, cap(*x), cap(q), cap(*sc), stream,
                                      err, sizeof(err));
        Py_END_ALLOW_THREADS
    }
    return rc != FMHA_OK ? raise_code(rc, err) : THPVariable_Wrap(q);
}

// quantize_v(x, seq32, stream) -> (q, scale), or None
PyObject* quantize_v_impl(PyObject* const* a, Py_ssize_t n) {
    if (n != 3) return decline();
    const at::Tensor* x = plain_bf16(a[0]);
    const bool seq32 = a[1] == Py_True;
    if (!x || (seq32 && (x->dim() != 4 || x->size(3) != kD || x->numel() > INT32_MAX * kD))) return decline();
    const int dev = x->device().index();
    bool ok = true;
    void* stream = stream_of(a[2], dev, ok);
    if (!ok) return decline();
    char err[512] = "";
    int rc;
    at::Tensor q, sc;
    {
        OnDevice on(dev);
        q = at::empty(x->sizes(), x->options().dtype(at::kByte));
        sc = seq32 ? at::empty({x->size(0), (x->size(1) + 31) / 32, x->size(2), kD}, x->options().dtype(at::kByte))
                   : at::empty({1024}, x->options().dtype(at::kFloat));
        Py_BEGIN_ALLOW_THREADS
        rc = seq32 ? fmha_mxfp8_quantize_seq32(x->data_ptr(), q.data_ptr(), sc.data_ptr(), (int32_t)x->size(0), (int32_t)x->size(1),
                                               (int32_t)x->size(2), cap(*x), cap(q), cap(sc), stream, err, sizeof(err))
                   : fmha_mxfp8_quantize_v(x->data_ptr(), q.data_ptr(), sc.data_ptr(), x->numel(), cap(*x), cap(q), cap(sc), stream, err,
                                           sizeof(err));
        Py_END_ALLOW_THREADS
    }
    if (rc != FMHA_OK) return raise_code(rc, err);
    PyObject *pq = THPVariable_Wrap(q), *ps = THPVariable_Wrap(sc);
    PyObject* r = pq && ps ? PyTuple_Pack(2, pq, ps) : nullptr;
    Py_XDECREF(pq);
    Py_XDECREF(ps);
    return r;
}

// quantize_qkv(q, k, v, mul, seq32, stream) -> (q8, k8, v8, q_scale, k_scale, v_scale), or None. The scales lie
// at the front of allocations with the (cleared) slack that the attention requires behind them.
PyObject* quantize_qkv_impl(PyObject* const* a, Py_ssize_t n) {
    if (n != 6) return decline();
    const at::Tensor *q = plain_bf16(a[0]), *k = plain_bf16(a[1]), *v = plain_bf16(a[2]);
    if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || q->device() != k->device() || q->device() != v->device()) return decline();
    const int64_t B = q->size(0), S = q->size(1), H = q->size(2), SK = k->size(1), HK = k->size(2);
    if (!is4(*q, B, S, H, kD, 2, 16) || !is4(*k, B, SK, HK, kD, 2, 16) || !is4(*v, B, SK, HK, kD, 2, 16)) return decline();
    if (B > INT32_MAX || S > INT32_MAX || H > INT32_MAX || SK > INT32_MAX || HK > INT32_MAX) return decline();
    const bool seq32 = a[4] == Py_True;
    const int dev = q->device().index();
    bool ok = true;
    void* stream = stream_of(a[5], dev, ok);
    const double mul = PyFloat_AsDouble(a[3]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return decline();
    }
    if (!ok) return decline();
    const int64_t nq = B * S * H, nk = B * SK * HK, nb = (SK + 31) / 32;
    char err[512] = "";
    int rc;
    at::Tensor o[6];
    {
        OnDevice on(dev);
        const auto bytes = q->options().dtype(at::kByte);
        o[0] = at::empty(q->sizes(), bytes);
        o[1] = at::empty(k->sizes(), bytes);
        o[2] = at::empty(v->sizes(), bytes);
        const at::Tensor qs = at::empty({nq * 4 + 640 * H * 4}, bytes), ks = at::empty({nk * 4 + 640 * HK * 4}, bytes);
        o[3] = qs.narrow(0, 0, nq * 4).view({B, S, H, 4});
        o[4] = ks.narrow(0, 0, nk * 4).view({B, SK, HK, 4});
        o[5] = seq32 ? at::empty({B, nb, HK, kD}, bytes) : at::empty({1024}, q->options().dtype(at::kFloat));
        fmha_mxfp8_qkv_params p;
        std::memset(&p, 0, sizeof(p));
        p.q = q->data_ptr(); p.k = k->data_ptr(); p.v = v->data_ptr();
        p.q8 = o[0].data_ptr(); p.k8 = o[1].data_ptr(); p.v8 = o[2].data_ptr();
        p.q_scale = qs.data_ptr(); p.k_scale = ks.data_ptr(); p.v_scale = o[5].data_ptr();
        p.bytes_q = cap(*q); p.bytes_k = cap(*k); p.bytes_v = cap(*v);
        p.bytes_q8 = cap(o[0]); p.bytes_k8 = cap(o[1]); p.bytes_v8 = cap(o[2]);
        p.bytes_q_scale = (uint64_t)qs.numel(); p.bytes_k_scale = (uint64_t)ks.numel(); p.bytes_v_scale = cap(o[5]);
        p.B = (int32_t)B; p.S = (int32_t)S; p.H = (int32_t)H; p.SK = (int32_t)SK; p.HK = (int32_t)HK;
        p.v_seq32 = seq32 ? 1 : 0;
        p.q_mul = (float)mul;
        Py_BEGIN_ALLOW_THREADS
        rc = fmha_mxfp8_quantize_qkv(&p, stream, err, sizeof(err));
        Py_END_ALLOW_THREADS
    }
    if (rc != FMHA_OK) return raise_code(rc, err);
    PyObject* r = PyTuple_New(6);
    for (int i = 0; r && i < 6; ++i) {
        PyObject* t = THPVariable_Wrap(o[i]);
        if (!t) {
            Py_DECREF(r);
            return nullptr;
        }
        PyTuple_SET_ITEM(r, i, t);
    }
    return r;
}

// No C++ exception leaves a call: tensors without storage (vmap's, functional ones) throw where their memory is asked for.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* a, Py_ssize_t n) {
    try {
        return F(a, n);
    } catch (const std::exception&) {
        return decline();
    }
}

// run(params address, device, stream) -> (path, splits, partials): attend's call for params that Python filled
PyObject* run_impl(PyObject* const* a, Py_ssize_t n) {
    if (n != 3) return decline();
    bool ok = true;
    const int dev = (int)PyLong_AsLong(a[1]);
    fmha_mxfp8_params p;
    const void* src = PyLong_AsVoidPtr(a[0]);
    if (PyErr_Occurred()) return nullptr;
    std::memcpy(&p, src, sizeof(p));
    void* stream = stream_of(a[2], dev, ok);
    if (!ok) {
        PyErr_SetString(PyExc_TypeError, "stream: expected a hipStream_t handle");
        return nullptr;
    }
    try {
        return run_params(p, dev, stream);
    } catch (const std::exception&) {   // (out of memory)
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// set_error(cls): the exception class of failing C calls (lib.FmhaError: code, message)
PyObject* set_error(PyObject*, PyObject* cls) {
    Py_INCREF(cls);
    Py_XSETREF(fmha_error, cls);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"attend", (PyCFunction)(void*)guarded<attend_impl>, METH_FASTCALL, nullptr},
    {"quantize_rows", (PyCFunction)(void*)guarded<quantize_rows_impl>, METH_FASTCALL, nullptr},
    {"quantize_v", (PyCFunction)(void*)guarded<quantize_v_impl>, METH_FASTCALL, nullptr},
    {"quantize_qkv", (PyCFunction)(void*)guarded<quantize_qkv_impl>, METH_FASTCALL, nullptr},
    {"run", (PyCFunction)(void*)guarded<run_impl>, METH_FASTCALL, nullptr},
    {"set_error", set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fmha_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fmha_ops() { return PyModule_Create(&module); }
