// The native call path between Python and libsqhip.so: argument checks, workspace lookup, output allocation and the call
// itself, on torch tensors, in one C function per entry point.
//
// A decode-time product takes the GPU 5 to 20 us.  The same steps in Python (a ctypes struct per piece, a device context, the
// stream, the workspace, a ctypes call) took 18 us for one piece and 24 for three, 6 more through a Python custom op, so a
// program without a graph waited for its host on every call; here they take 4 to 6 us, of which the launch is 3.5.
//
// Every function answers 0 (done), a negative SQ_E* code (sq_last_error has the text), or 1: not a call this path covers (an
// unusual dtype or stride, a workspace that has to grow, a stream under capture), and the caller goes on in Python, which
// also words the errors.  Nothing is kept between calls but what a matrix is (its tensors and sizes, dropped by PackedLinear
// whenever one of its attributes is set).
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>
#include "../../include/sqhip.h"

namespace {

constexpr int MAX_PIECES = 8;
constexpr int NOT_COVERED = 1;

struct Native {                      // one packed matrix: its tensors and what the library wants to know about them
    PyObject_HEAD
    sq_matrix m;
    at::Tensor* t;                   // words, table, row_scale, row_book, row_mask, perms, row_order, stream
};

PyObject *s_native, *s_make_native, *s_rls, *s_cross, *s_large, *s_dequant_from, *s_enabled, *s_forward, *s_trace, *s_fused;
PyObject *g_bufs;                    // kernels._Workspace.bufs
PyObject *g_registry, *g_core;       // vllm_ext.core._REGISTRY and the module itself (its _trace is looked up per call)
PyTypeObject* g_shards_type;         // vllm_ext.core.PackedShards
PyObject* g_keys[64];                // (str(device), "kernels") per device

void native_dealloc(PyObject* self) {
    delete[] reinterpret_cast<Native*>(self)->t;
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject NativeType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// native(words, table, row_scale, row_book, row_mask, perms, row_order, stream, R, C, d, bits, G, M, W, stream_runs, stream_groups)
PyObject* make_native(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 17) { PyErr_SetString(PyExc_TypeError, "native: 17 arguments"); return nullptr; }
    Native* o = reinterpret_cast<Native*>(NativeType.tp_alloc(&NativeType, 0));
    if (!o) return nullptr;
    o->t = new at::Tensor[8];
    for (int i = 0; i < 8; ++i)
        if (THPVariable_Check(a[i])) o->t[i] = THPVariable_Unpack(a[i]);
    int32_t v[9];
    for (int i = 0; i < 9; ++i) v[i] = (int32_t)PyLong_AsLong(a[8 + i]);
    if (PyErr_Occurred()) { Py_DECREF(o); return nullptr; }
    sq_matrix& m = o->m;
    m.R = v[0]; m.C = v[1]; m.d = v[2]; m.bits = v[3]; m.G = v[4]; m.M = v[5]; m.W = v[6]; m.y_off = 0;
    m.stream_runs = v[7]; m.stream_groups = v[8];
    return reinterpret_cast<PyObject*>(o);
}

// The pieces of a call as the library takes them, and what owns their tensors: the library runs without the GIL, so another
// thread may set an attribute of a piece (which drops its Native) before the kernels are launched.
// 0, NOT_COVERED, or -1 with a Python error set.
struct Pieces { sq_matrix m[MAX_PIECES]; int n = 0, dev = -1; int64_t rows = 0; pybind11::object held[MAX_PIECES]; };
int unpack_pieces(PyObject* seq, Pieces& p) {
    if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) return NOT_COVERED;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    if (n < 1 || n > MAX_PIECES) return NOT_COVERED;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* piece = PySequence_Fast_GET_ITEM(seq, i);
        PyObject* o = PyObject_GetAttr(piece, s_native);
        if (!o) { PyErr_Clear(); return NOT_COVERED; }
        if (o == Py_None) {
            Py_DECREF(o);
            o = PyObject_CallMethodObjArgs(piece, s_make_native, nullptr);
            if (!o) return -1;
        }
        p.held[i] = pybind11::reinterpret_steal<pybind11::object>(o);
        if (Py_TYPE(o) != &NativeType) return NOT_COVERED;
        const Native* nat = reinterpret_cast<Native*>(o);
        sq_matrix& m = p.m[i];
        m = nat->m;
        const at::Tensor* t = nat->t;
        auto ptr = [](const at::Tensor& x) { return x.defined() ? x.data_ptr() : nullptr; };
        m.tags = (const int32_t*)ptr(t[0]); m.table = (const uint16_t*)ptr(t[1]); m.row_scale = (const uint16_t*)ptr(t[2]);
        m.row_book = (const uint8_t*)ptr(t[3]); m.row_mask = (const uint8_t*)ptr(t[4]); m.perms = (const int32_t*)ptr(t[5]);
        m.row_order = (const int32_t*)ptr(t[6]); m.stream = ptr(t[7]);
        m.y_off = (int32_t)p.rows;
        p.rows += m.R;
        const int dev = t[1].is_cuda() ? t[1].get_device() : -1;
        if (dev < 0 || dev >= 64 || (i > 0 && dev != p.dev) || m.C != p.m[0].C) return NOT_COVERED;
        p.dev = dev;
    }
    p.n = (int)n;
    return 0;
}

int dtype_of(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return SQ_F32;
        case at::kHalf: return SQ_F16;
        case at::kBFloat16: return SQ_BF16;
        default: return -1;
    }
}
bool is16(int dt) { return dt == SQ_F16 || dt == SQ_BF16; }

// a [rows, cols] matrix on device `dev` with unit column stride; a subclass or a tensor that needs Python dispatch is left alone
bool matrix_on(const at::Tensor& t, int dev) {
    return t.dim() == 2 && t.is_cuda() && t.get_device() == dev && t.layout() == at::kStrided && !t.unsafeGetTensorImpl()->is_python_dispatch() &&
           (t.stride(1) == 1 || t.size(1) == 1);
}
int64_t row_ld(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max(t.stride(0), t.size(1)); }
bool vec16(const at::Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

// The device as it was, and the current stream of `dev`.
struct OnDevice {
    int prev = -1;
    hipStream_t stream;
    explicit OnDevice(int dev) {
        const int cur = c10::hip::current_device();
        if (cur != dev) { prev = cur; c10::hip::set_device((c10::DeviceIndex)dev); }
        stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    }
    ~OnDevice() { if (prev >= 0) c10::hip::set_device((c10::DeviceIndex)prev); }
};

// The shared workspace of a device (kernels._Workspace), held for as long as the call uses it: the library runs without the
// GIL, and a call of another thread may meanwhile replace the buffer by a larger one.  (Its kernels are enqueued when the call
// returns; what is freed after that is given out again behind them on this stream.)
struct Workspace { at::Tensor held; void* p = nullptr; size_t bytes = 0; };
// It if it holds `need` bytes and the stream is not being captured (who was captured with which buffer is recorded in Python).
bool workspace(int dev, size_t need, hipStream_t s, Workspace& ws) {
    if (need == 0) return true;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone) { (void)hipGetLastError(); return false; }
    if (!g_keys[dev]) g_keys[dev] = Py_BuildValue("(Ns)", PyUnicode_FromFormat("cuda:%d", dev), "kernels");
    PyObject* b = g_bufs && g_keys[dev] ? PyDict_GetItem(g_bufs, g_keys[dev]) : nullptr;
    if (!b || !THPVariable_Check(b)) return false;
    const at::Tensor& t = THPVariable_Unpack(b);
    if ((size_t)t.numel() < need) return false;
    ws.held = t;
    ws.p = t.data_ptr();
    ws.bytes = (size_t)t.numel();
    return true;
}

// The workspace of a product: the shared one; a buffer of the call's own where the pieces could run without any (their partial sums
// only make them faster), so that streams may run them side by side.
bool product_workspace(const Pieces& p, int rows, int which, const at::Tensor& like, hipStream_t s, Workspace& ws) {
    const size_t need = sq_workspace_bytes(p.m, p.n, rows, which);
    if (need == 0 || rows > SQ_SMALL_BMAX || sq_workspace_bytes(p.m, p.n, rows, which | 4) != 0) return workspace(p.dev, need, s, ws);
    ws.bytes = sq_workspace_bytes(p.m, p.n, rows, which | 2);
    ws.held = at::empty({(int64_t)ws.bytes}, like.options().dtype(at::kByte));
    ws.p = ws.held.data_ptr();
    return true;
}

int linear_into(const Pieces& p, const at::Tensor& x, const at::Tensor& y, bool gemm) {
    const int xd = dtype_of(x), yd = dtype_of(y);
    if (!is16(xd) || yd < 0 || !matrix_on(x, p.dev) || !matrix_on(y, p.dev) || x.size(0) != y.size(0) || y.size(1) != p.rows || x.size(1) != p.m[0].C ||
        x.size(0) < 1)
        return NOT_COVERED;
    const int B = (int)x.size(0);
    OnDevice on(p.dev);
    Workspace ws;
    if (!product_workspace(p, B, gemm, x, on.stream, ws)) return NOT_COVERED;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = (gemm ? sq_linear_gemm : sq_linear_small)(p.m, p.n, x.data_ptr(), xd, row_ld(x), y.data_ptr(), yd, row_ld(y), B, ws.p, ws.bytes, on.stream);
    Py_END_ALLOW_THREADS
    return rc;
}

PyObject* answer(int rc) { return rc == -1 && PyErr_Occurred() ? nullptr : PyLong_FromLong(rc); }
bool tensors(PyObject* const* a, int n) {
    for (int i = 0; i < n; ++i) if (!THPVariable_Check(a[i])) return false;
    return true;
}

// (torch's own translation: an allocation that fails is a torch.OutOfMemoryError here too)
#define SQ_GUARD(...) try { __VA_ARGS__ } catch (...) { if (!PyErr_Occurred()) torch::translate_exception_to_python(std::current_exception()); return nullptr; }

// linear(pieces, x, y, gemm)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 4 || !tensors(a + 1, 2)) return answer(NOT_COVERED);
    SQ_GUARD(
        Pieces p;
        if (int rc = unpack_pieces(a[0], p)) return answer(rc);
        return answer(linear_into(p, THPVariable_Unpack(a[1]), THPVariable_Unpack(a[2]), a[3] == Py_True));
    )
}

// The forward of a PackedShards: a tensor, an undefined tensor (not covered), or a Python error.
bool shards_forward(PyObject* ps, const at::Tensor& x, at::Tensor& out, int* rc) {
    *rc = NOT_COVERED;
    if (x.dim() < 1 || !x.is_cuda() || !is16(dtype_of(x)) || !x.is_contiguous() || x.unsafeGetTensorImpl()->is_python_dispatch()) return true;
    auto get = [&](PyObject* name) { return pybind11::reinterpret_steal<pybind11::object>(PyObject_GetAttr(ps, name)); };
    pybind11::object rls = get(s_rls), cross = get(s_cross);
    if (!rls || !cross) return false;
    Pieces p;
    if (int r = unpack_pieces(rls.ptr(), p)) { *rc = r; return r >= 0 || !PyErr_Occurred(); }
    const int64_t C = p.m[0].C;
    if (x.size(-1) != C || x.numel() == 0 || x.get_device() != p.dev || C % 8 || !vec16(x)) return true;
    const int64_t M = x.numel() / C;
    const long cr = PyLong_AsLong(cross.ptr());
    if (cr == -1 && PyErr_Occurred()) { PyErr_Clear(); return true; }
    bool gemm = false;
    if (M > cr) {
        pybind11::object large = get(s_large), from = get(s_dequant_from);
        if (!large || !from) return false;
        if (PyUnicode_Compare(large.ptr(), s_fused) != 0) return true;
        const long f = PyLong_AsLong(from.ptr());
        if ((f == -1 && PyErr_Occurred()) || M >= f || M > INT32_MAX) { PyErr_Clear(); return true; }
        gemm = true;
    }
    const at::Tensor x2 = x.dim() == 2 ? x : x.view({M, C});
    at::Tensor y = at::empty({M, p.rows}, x.options());
    *rc = linear_into(p, x2, y, gemm);
    if (*rc) return true;
    if (x.dim() == 2) { out = std::move(y); return true; }
    auto sizes = x.sizes().vec();
    sizes.back() = p.rows;
    out = y.view(sizes);
    return true;
}

// forward(shards, x) -> tensor or a code
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2 || !THPVariable_Check(a[1])) return answer(NOT_COVERED);
    SQ_GUARD(
        at::Tensor out;
        int rc;
        if (!shards_forward(a[0], THPVariable_Unpack(a[1]), out, &rc)) return nullptr;
        return rc ? answer(rc) : THPVariable_Wrap(std::move(out));
    )
}

// addnorm operands as the library takes them; `C` columns, `B` rows, the 16-bit operands of type `dt` (dt < 0: their own)
struct Norm { const float* h_in; float* h_out; const void* add; const void* w; int add_dt = 0, w_dt = 0; int64_t ld_h = 0, ld_add = 0; };
bool norm_operands(PyObject* h_in, PyObject* add, PyObject* w, PyObject* h_out, int dev, int64_t B, int64_t C, int dt, Norm& o) {
    if (!THPVariable_Check(h_in) || !THPVariable_Check(w)) return false;
    const at::Tensor& h = THPVariable_Unpack(h_in);
    const at::Tensor& wt = THPVariable_Unpack(w);
    if (h.scalar_type() != at::kFloat || !matrix_on(h, dev) || h.size(0) != B || h.size(1) != C) return false;
    o.w_dt = dtype_of(wt);
    if (!wt.is_cuda() || wt.get_device() != dev || wt.numel() != C || !wt.is_contiguous() || !is16(o.w_dt) || (dt >= 0 && o.w_dt != dt)) return false;
    o.h_in = (const float*)h.data_ptr(); o.ld_h = row_ld(h); o.w = wt.data_ptr();
    o.add = nullptr; o.h_out = nullptr;
    if (add != Py_None) {
        if (!THPVariable_Check(add)) return false;
        const at::Tensor& t = THPVariable_Unpack(add);
        o.add_dt = dtype_of(t);
        if (!is16(o.add_dt) || (dt >= 0 && o.add_dt != dt) || !matrix_on(t, dev) || t.size(0) != B || t.size(1) != C) return false;
        o.add = t.data_ptr(); o.ld_add = row_ld(t);
    }
    if (h_out != Py_None) {
        if (!THPVariable_Check(h_out)) return false;
        const at::Tensor& t = THPVariable_Unpack(h_out);
        if (t.scalar_type() != at::kFloat || !matrix_on(t, dev) || t.sizes() != h.sizes() || t.strides() != h.strides()) return false;
        o.h_out = (float*)t.data_ptr();
    }
    return true;
}
bool perm_operand(PyObject* perms, int dev, int64_t C, const int32_t** pp, int* M) {
    *pp = nullptr; *M = 1;
    if (perms == Py_None) return true;
    if (!THPVariable_Check(perms)) return false;
    const at::Tensor& t = THPVariable_Unpack(perms);
    if (t.scalar_type() != at::kInt || t.dim() != 2 || t.size(1) != C || !t.is_contiguous() || !t.is_cuda() || t.get_device() != dev) return false;
    *pp = (const int32_t*)t.data_ptr(); *M = (int)t.size(0);
    return true;
}

// addnorm(h_in, add, w, eps, out, h_out, perms)
PyObject* addnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 7 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[4])) return answer(NOT_COVERED);
    SQ_GUARD(
        const at::Tensor& h = THPVariable_Unpack(a[0]);
        const at::Tensor& out = THPVariable_Unpack(a[4]);
        if (h.dim() != 2 || !h.is_cuda()) return answer(NOT_COVERED);
        const int dev = h.get_device();
        const int64_t B = h.size(0); const int64_t C = h.size(1);
        Norm o; const int32_t* pp; int M;
        const double eps = PyFloat_AsDouble(a[3]);
        if (PyErr_Occurred()) return nullptr;
        if (B < 1 || !norm_operands(a[0], a[1], a[2], a[5], dev, B, C, -1, o) || !perm_operand(a[6], dev, C, &pp, &M) || !is16(dtype_of(out)) ||
            !out.is_cuda() || out.get_device() != dev || !out.is_contiguous() || out.numel() != B * M * C)
            return answer(NOT_COVERED);
        OnDevice on(dev);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_addnorm(o.h_in, o.h_out, h.stride(0), o.add, o.add_dt, o.ld_add, o.w, o.w_dt, pp, M, (int)B, (int)C, (float)eps, out.data_ptr(), dtype_of(out), on.stream);
        Py_END_ALLOW_THREADS
        return answer(rc);
    )
}

// silu_mul(gate, up, out, perms)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 4 || !tensors(a, 3)) return answer(NOT_COVERED);
    SQ_GUARD(
        const at::Tensor& g = THPVariable_Unpack(a[0]);
        const at::Tensor& u = THPVariable_Unpack(a[1]);
        const at::Tensor& out = THPVariable_Unpack(a[2]);
        if (g.dim() != 2 || !g.is_cuda()) return answer(NOT_COVERED);
        const int dev = g.get_device(); const int dt = dtype_of(g);
        const int64_t B = g.size(0); const int64_t C = g.size(1);
        const int32_t* pp; int M;
        if (B < 1 || !is16(dt) || !matrix_on(g, dev) || !matrix_on(u, dev) || dtype_of(u) != dt || u.sizes() != g.sizes() || u.strides() != g.strides() ||
            !perm_operand(a[3], dev, C, &pp, &M) || dtype_of(out) != dt || !out.is_cuda() || out.get_device() != dev || !out.is_contiguous() || out.numel() != B * M * C)
            return answer(NOT_COVERED);
        OnDevice on(dev);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_silu_mul(g.data_ptr(), u.data_ptr(), dt, g.stride(0), pp, M, (int)B, (int)C, out.data_ptr(), on.stream);
        Py_END_ALLOW_THREADS
        return answer(rc);
    )
}

// linear_from(pieces, y, x_out, h_in, add, w, eps, h_out, gate, up)
PyObject* linear_from(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 10 || !tensors(a + 1, 2) || (a[3] == Py_None) == (a[8] == Py_None)) return answer(NOT_COVERED);
    SQ_GUARD(
        Pieces p;
        if (int rc = unpack_pieces(a[0], p)) return answer(rc);
        const at::Tensor& y = THPVariable_Unpack(a[1]);
        const at::Tensor& x = THPVariable_Unpack(a[2]);
        const int dt = dtype_of(x); const int yd = dtype_of(y);
        if (!is16(dt) || yd < 0 || !matrix_on(x, p.dev) || !x.is_contiguous() || !matrix_on(y, p.dev) || x.size(0) != y.size(0) || x.size(0) < 1 ||
            y.size(1) != p.rows || x.size(1) != p.m[0].C)
            return answer(NOT_COVERED);
        const int64_t B = x.size(0); const int64_t C = x.size(1);
        sq_producer pr{};
        pr.x_out = x.data_ptr();
        pr.eps = (float)PyFloat_AsDouble(a[6]);
        if (PyErr_Occurred()) return nullptr;
        if (a[3] != Py_None) {
            Norm o;
            if (!norm_operands(a[3], a[4], a[5], a[7], p.dev, B, C, dt, o)) return answer(NOT_COVERED);
            pr.mode = SQ_FROM_ADDNORM; pr.h_in = o.h_in; pr.h_out = o.h_out; pr.add = o.add; pr.w = o.w; pr.ld_h = o.ld_h; pr.ld_in = o.ld_add;
        } else {
            if (!tensors(a + 8, 2)) return answer(NOT_COVERED);
            const at::Tensor& g = THPVariable_Unpack(a[8]);
            const at::Tensor& u = THPVariable_Unpack(a[9]);
            if (dtype_of(g) != dt || dtype_of(u) != dt || !matrix_on(g, p.dev) || !matrix_on(u, p.dev) || g.sizes() != x.sizes() || u.sizes() != g.sizes() ||
                u.strides() != g.strides())
                return answer(NOT_COVERED);
            pr.mode = SQ_FROM_SILU_MUL; pr.add = g.data_ptr(); pr.up = u.data_ptr(); pr.ld_in = row_ld(g);
        }
        OnDevice on(p.dev);
        Workspace ws;
        if (!product_workspace(p, (int)B, 0, y, on.stream, ws)) return answer(NOT_COVERED);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_linear_small_from(p.m, p.n, &pr, dt, y.data_ptr(), yd, row_ld(y), (int)B, ws.p, ws.bytes, on.stream);
        Py_END_ALLOW_THREADS
        return answer(rc);
    )
}

// linear_silu(pieces, x, out, x_out, h_in, add, w, eps, h_out)
PyObject* linear_silu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    const bool norm = n == 9 && a[4] != Py_None;
    if (n != 9 || !THPVariable_Check(a[norm ? 3 : 1]) || !THPVariable_Check(a[2])) return answer(NOT_COVERED);
    SQ_GUARD(
        Pieces p;
        if (int rc = unpack_pieces(a[0], p)) return answer(rc);
        const at::Tensor& x = THPVariable_Unpack(a[norm ? 3 : 1]);
        const at::Tensor& out = THPVariable_Unpack(a[2]);
        const int dt = dtype_of(x);
        if (p.n != 2 || p.m[0].R != p.m[1].R || !is16(dt) || dtype_of(out) != dt || !matrix_on(x, p.dev) || !matrix_on(out, p.dev) || x.size(0) < 1 ||
            out.size(0) != x.size(0) || out.size(1) != p.m[0].R || x.size(1) != p.m[0].C)
            return answer(NOT_COVERED);
        const int64_t B = x.size(0);
        sq_producer pr{};
        if (norm) {
            Norm o;
            pr.eps = (float)PyFloat_AsDouble(a[7]);
            if (PyErr_Occurred()) return nullptr;
            if (B != 1 || !x.is_contiguous() || !norm_operands(a[4], a[5], a[6], a[8], p.dev, B, x.size(1), dt, o)) return answer(NOT_COVERED);
            pr.mode = SQ_FROM_ADDNORM; pr.x_out = x.data_ptr();
            pr.h_in = o.h_in; pr.h_out = o.h_out; pr.add = o.add; pr.w = o.w; pr.ld_h = o.ld_h; pr.ld_in = o.ld_add;
        }
        OnDevice on(p.dev);
        Workspace ws;
        if (!product_workspace(p, (int)B, 0, out, on.stream, ws)) return answer(NOT_COVERED);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_linear_small_silu(p.m, 2, norm ? &pr : nullptr, norm ? nullptr : x.data_ptr(), dt, norm ? 0 : row_ld(x), out.data_ptr(), row_ld(out), (int)B,
                                  ws.p, ws.bytes, on.stream);
        Py_END_ALLOW_THREADS
        if (rc != SQ_EUNSUPPORTED) return answer(rc);
        // no fused kernel for this stack: the product into a temporary, then SiLU * up (which writes whole rows)
        if (!out.is_contiguous()) return answer(NOT_COVERED);
        const at::Tensor y = at::empty({B, p.rows}, x.options());
        uint16_t* yp = (uint16_t*)y.data_ptr();
        Py_BEGIN_ALLOW_THREADS
        rc = norm ? sq_linear_small_from(p.m, 2, &pr, dt, yp, dt, p.rows, (int)B, ws.p, ws.bytes, on.stream)
                  : sq_linear_small(p.m, 2, x.data_ptr(), dt, row_ld(x), yp, dt, p.rows, (int)B, ws.p, ws.bytes, on.stream);
        if (rc == SQ_OK) rc = sq_silu_mul(yp, yp + p.m[0].R, dt, p.rows, nullptr, 1, (int)B, p.m[0].R, out.data_ptr(), on.stream);
        Py_END_ALLOW_THREADS
        return answer(rc);
    )
}

// q8_linear(q, scale, x, y)
PyObject* q8_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 4 || !tensors(a, 4)) return answer(NOT_COVERED);
    SQ_GUARD(
        const at::Tensor& q = THPVariable_Unpack(a[0]);
        const at::Tensor& sc = THPVariable_Unpack(a[1]);
        const at::Tensor& x = THPVariable_Unpack(a[2]);
        const at::Tensor& y = THPVariable_Unpack(a[3]);
        if (!q.is_cuda() || q.dim() != 2 || q.scalar_type() != at::kChar || !q.is_contiguous()) return answer(NOT_COVERED);
        const int dev = q.get_device(); const int xd = dtype_of(x); const int yd = dtype_of(y);
        const int64_t V = q.size(0); const int64_t C = q.size(1);
        if (C % 32 || !sc.is_cuda() || sc.get_device() != dev || sc.scalar_type() != at::kHalf || !sc.is_contiguous() || sc.dim() != 2 || sc.size(0) != V ||
            sc.size(1) != C / 32 || !is16(xd) || yd < 0 || !matrix_on(x, dev) || !matrix_on(y, dev) || x.size(1) != C || x.size(0) < 1 || y.size(0) != x.size(0) ||
            y.size(1) < V)
            return answer(NOT_COVERED);
        OnDevice on(dev);
        Workspace ws;
        const size_t need = sq_q8_workspace_bytes((int)V, (int)C, (int)x.size(0));
        if (need && C % 256 && x.size(0) <= SQ_SMALL_BMAX) {     // (a buffer of its own: see kernels.q8_linear)
            ws.held = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
            ws.p = ws.held.data_ptr();
            ws.bytes = need;
        } else if (!workspace(dev, need, on.stream, ws)) {
            return answer(NOT_COVERED);
        }
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_q8_linear((const int8_t*)q.data_ptr(), (const uint16_t*)sc.data_ptr(), (int)V, (int)C, x.data_ptr(), xd, x.stride(0), y.data_ptr(), yd, y.stride(0),
                          (int)x.size(0), ws.p, ws.bytes, on.stream);
        Py_END_ALLOW_THREADS
        return answer(rc);
    )
}

// q4_rows(q, scale, ids, dtype code) -> [len(ids), C], or a code; tables on the GPU (pinned host tables: Python)
PyObject* q4_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 4 || !tensors(a, 3)) return answer(NOT_COVERED);
    SQ_GUARD(
        const at::Tensor& q = THPVariable_Unpack(a[0]);
        const at::Tensor& sc = THPVariable_Unpack(a[1]);
        const at::Tensor& ids = THPVariable_Unpack(a[2]);
        const long dt = PyLong_AsLong(a[3]);
        if (PyErr_Occurred()) return nullptr;
        if (!q.is_cuda() || q.dim() != 2 || q.scalar_type() != at::kByte || !q.is_contiguous() || !ids.is_cuda() || ids.get_device() != q.get_device() ||
            ids.dim() != 1 || ids.scalar_type() != at::kLong || !ids.is_contiguous() || ids.unsafeGetTensorImpl()->is_python_dispatch() || dt < SQ_F32 || dt > SQ_BF16)
            return answer(NOT_COVERED);
        const int dev = q.get_device();
        const int64_t V = q.size(0); const int64_t C = q.size(1) * 2;
        if (C % 32 || !sc.is_cuda() || sc.get_device() != dev || sc.scalar_type() != at::kHalf || !sc.is_contiguous() || sc.dim() != 2 || sc.size(0) != V ||
            sc.size(1) != C / 32)
            return answer(NOT_COVERED);
        OnDevice on(dev);
        at::Tensor out = at::empty({ids.numel(), C}, q.options().dtype(dt == SQ_F32 ? at::kFloat : dt == SQ_F16 ? at::kHalf : at::kBFloat16));
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = sq_q4_embed((const uint8_t*)q.data_ptr(), (const uint16_t*)sc.data_ptr(), (int)V, (int)C, (const int64_t*)ids.data_ptr(), ids.numel(), out.data_ptr(),
                         (int)dt, C, on.stream);
        Py_END_ALLOW_THREADS
        return rc ? answer(rc) : THPVariable_Wrap(std::move(out));
    )
}

// ------------------------------------------------------------------------------------------ torch.ops.shapequant.linear

at::Tensor linear_op(const at::Tensor& x, int64_t handle) {
    pybind11::gil_scoped_acquire gil;
    if (!g_core) throw std::runtime_error("shapequant::linear: quantexperiments_amd.vllm_ext.core is not loaded");
    auto own = [](PyObject* o) { if (!o) throw pybind11::error_already_set(); return pybind11::reinterpret_steal<pybind11::object>(o); };
    pybind11::object obj = own(PySequence_GetItem(g_registry, (Py_ssize_t)handle));
    pybind11::object trace = own(PyObject_GetAttr(g_core, s_trace)), on = own(PyObject_GetAttr(trace.ptr(), s_enabled));
    if (on.ptr() == Py_False && Py_TYPE(obj.ptr()) == g_shards_type) {
        at::Tensor out;
        int rc;
        if (!shards_forward(obj.ptr(), x, out, &rc)) throw pybind11::error_already_set();
        if (rc == 0) return out;
    }
    pybind11::object fn = own(PyObject_GetAttr(g_core, s_forward)), h = own(PyLong_FromLongLong(handle)), xo = own(THPVariable_Wrap(x));
    pybind11::object y = own(PyObject_CallFunctionObjArgs(fn.ptr(), xo.ptr(), h.ptr(), nullptr));
    if (!THPVariable_Check(y.ptr())) throw std::runtime_error("shapequant::linear: forward did not return a tensor");
    return THPVariable_Unpack(y.ptr());
}

const c10::TypedOperatorHandle<at::Tensor(const at::Tensor&, int64_t)>& linear_handle() {
    static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow("shapequant::linear", "").typed<at::Tensor(const at::Tensor&, int64_t)>();
    return h;
}

// inference only: the forward runs on inputs that require a gradient, its backward raises
struct NoBackward : torch::autograd::Function<NoBackward> {
    static at::Tensor forward(torch::autograd::AutogradContext*, const at::Tensor& x, int64_t handle) {
        at::AutoDispatchBelowADInplaceOrView below;
        return linear_handle().call(x, handle);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext*, torch::autograd::variable_list) {
        C10_THROW_ERROR(NotImplementedError, "shapequant::linear has no autograd formula");
    }
};

at::Tensor linear_autograd(const at::Tensor& x, int64_t handle) {
    if (at::GradMode::is_enabled() && x.requires_grad()) return NoBackward::apply(x, handle);
    at::AutoDispatchBelowADInplaceOrView below;
    return linear_handle().call(x, handle);
}

// install(bufs): where the workspaces are;  install_op(core module, registry, PackedShards)
PyObject* install(PyObject*, PyObject* bufs) {
    Py_INCREF(bufs);
    Py_XDECREF(g_bufs);
    g_bufs = bufs;
    Py_RETURN_NONE;
}
PyObject* install_op(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 3 || !PyType_Check(a[2])) { PyErr_SetString(PyExc_TypeError, "install_op(core, registry, shards type)"); return nullptr; }
    for (int i = 0; i < 3; ++i) Py_INCREF(a[i]);
    g_core = a[0];
    g_registry = a[1];
    g_shards_type = reinterpret_cast<PyTypeObject*>(a[2]);
    Py_RETURN_NONE;
}

#define SQ_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"native", (PyCFunction)(void (*)(void))make_native, METH_FASTCALL, nullptr}, {"install", install, METH_O, nullptr}, SQ_FAST(install_op),
                         SQ_FAST(linear), SQ_FAST(forward), SQ_FAST(linear_from), SQ_FAST(linear_silu), SQ_FAST(addnorm), SQ_FAST(silu_mul), SQ_FAST(q8_linear), SQ_FAST(q4_rows),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

TORCH_LIBRARY_IMPL(shapequant, CUDA, m) { m.impl("linear", linear_op); }
TORCH_LIBRARY_IMPL(shapequant, AutogradCUDA, m) { m.impl("linear", linear_autograd); }

PyMODINIT_FUNC PyInit__native() {
    NativeType.tp_name = "quantexperiments_amd._native.Native";
    NativeType.tp_basicsize = sizeof(Native);
    NativeType.tp_flags = Py_TPFLAGS_DEFAULT;
    NativeType.tp_dealloc = native_dealloc;
    if (PyType_Ready(&NativeType) < 0) return nullptr;
    struct { PyObject** at; const char* s; } names[] = {{&s_native, "_native"}, {&s_make_native, "_make_native"}, {&s_rls, "rls"}, {&s_cross, "cross"},
        {&s_large, "large"}, {&s_dequant_from, "dequant_from"}, {&s_enabled, "enabled"}, {&s_forward, "_linear_in_python"}, {&s_trace, "_trace"},
        {&s_fused, "fused"}};
    for (auto& nm : names) if (!(*nm.at = PyUnicode_InternFromString(nm.s))) return nullptr;
    return PyModule_Create(&module_def);
}
