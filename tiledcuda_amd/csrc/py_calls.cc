// tiledcuda_amd._calls: what the Python entries do on an ordinary call - operands checked, outputs and workspace taken from torch's
// caching allocator, the C-ABI called on the current stream - without Python in between. A 128 x 64 x 256 product spends its
// time there: 7.1 us a call through ctypes, 4.2 here (3 of them the launch, 1 the allocation); a back-to-back product 8.4 -> 4.6.
// Every function returns None where a call is anything but ordinary (a subclass, another dtype or device, a shape that does not fit,
// an operand that is not contiguous, a status other than TCU_OK): the Python entry then runs as if this module were not there and
// reports what it always has. Nothing has been launched by then. (A launch that fails in the middle of an LSTM's steps is started
// again there.)
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>

#include <climits>
#include <cmath>
#include <cstring>

#include "tcu_c_api.h"

namespace {

/// The tensor behind `o` if it is a plain one, contiguous, of `dtype`, on the current device; else null.
const at::Tensor* plain(PyObject* o, at::ScalarType dtype, c10::DeviceIndex device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.scalar_type() != dtype || t.device().index() != device || !t.is_contiguous()) return nullptr;
    for (const int64_t n : t.sizes())
        if (n <= 0 || n > INT_MAX) return nullptr;
    return &t;
}

/// Whether there is a device to ask about at all: the first operand lives on one.
bool on_device(PyObject* o) { return THPVariable_CheckExact(o) && THPVariable_Unpack(o).is_cuda(); }
c10::DeviceIndex current_device() { return c10::hip::current_device(); }
void* current_stream(c10::DeviceIndex device) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream(); }
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
at::Tensor bytes(const at::Tensor& like, unsigned long long n) { return at::empty({static_cast<int64_t>(n)}, like.options().dtype(at::kByte)); }
/// The same for a workspace that a call can do without: undefined where the memory is not there.
at::Tensor bytes_if_free(const at::Tensor& like, unsigned long long n) {
    try {
        return bytes(like, n);
    } catch (const c10::OutOfMemoryError&) {
        return {};
    }
}

/// The call itself, without the interpreter's lock (it may wait for a place in the stream's queue).
template <typename F>
bool succeeds(F&& f) {
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = f();
    Py_END_ALLOW_THREADS
    return status == TCU_OK;
}

bool out_type(PyObject* o, at::ScalarType& type, int& code) {
    if (!THPDtype_Check(o)) return false;
    type = reinterpret_cast<THPDtype*>(o)->scalar_type;
    code = type == at::kFloat ? TCU_DTYPE_F32 : TCU_DTYPE_F16;
    return type == at::kFloat || type == at::kHalf;
}

// gemm(a, b_t, out_dtype)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3 || !on_device(args[0])) Py_RETURN_NONE;
    const auto device = current_device();
    const at::Tensor* a = plain(args[0], at::kHalf, device);
    const at::Tensor* b = a ? plain(args[1], at::kHalf, device) : nullptr;
    at::ScalarType type;
    int code;
    if (!b || a->dim() != 2 || b->dim() != 2 || a->size(1) != b->size(1) || !out_type(args[2], type, code)) Py_RETURN_NONE;
    const int M = int(a->size(0)), N = int(b->size(0)), K = int(a->size(1));
    at::Tensor c = at::empty({M, N}, a->options().dtype(type));
    void* const stream = current_stream(device);
    const void *ap = a->data_ptr(), *bp = b->data_ptr();
    void* const cp = c.data_ptr();
    bool ok;
    if (tcu_gemm_uses_workspace(M, N, K)) {
        const unsigned long long need = tcu_gemm_workspace_bytes(M, N, K);
        const at::Tensor ws = bytes(*a, need);
        void* const wp = ws.data_ptr();
        ok = succeeds([&] { return tcu_gemm_f16_ws(ap, bp, cp, M, N, K, code, wp, need, stream); });
    } else {
        ok = succeeds([&] { return tcu_gemm_f16(ap, bp, cp, M, N, K, code, TCU_GEMM_AUTO, stream); });
    }
    if (!ok) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

// b2b_gemm(a, b_t, c_t, out_dtype)
PyObject* b2b_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4 || !on_device(args[0])) Py_RETURN_NONE;
    const auto device = current_device();
    const at::Tensor* t[3];
    for (int i = 0; i < 3; ++i)
        if (!(t[i] = plain(args[i], at::kHalf, device)) || t[i]->dim() != t[0]->dim()) Py_RETURN_NONE;
    const int64_t d = t[0]->dim();
    at::ScalarType type;
    int code;
    if ((d != 2 && d != 3) || !out_type(args[3], type, code)) Py_RETURN_NONE;
    const int batch = d == 3 ? int(t[0]->size(0)) : 1;
    const int M = int(t[0]->size(-2)), K = int(t[0]->size(-1)), N = int(t[1]->size(-2)), P = int(t[2]->size(-2));
    if (t[1]->size(-1) != K || t[2]->size(-1) != N || (d == 3 && (t[1]->size(0) != batch || t[2]->size(0) != batch))) Py_RETURN_NONE;
    at::Tensor out = d == 3 ? at::empty({batch, M, P}, t[0]->options().dtype(type)) : at::empty({M, P}, t[0]->options().dtype(type));
    void* const stream = current_stream(device);
    const void *ap = t[0]->data_ptr(), *bp = t[1]->data_ptr(), *cp = t[2]->data_ptr();
    void* const op = out.data_ptr();
    if (!succeeds([&] { return tcu_b2b_gemm_f16(ap, bp, cp, op, M, N, K, P, batch, code, stream); })) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

bool attention(const void* q, const void* k, const void* v, void* o, int batch, int M, int N, int D, int P, float scale, int v_layout,
               const at::Tensor& like, c10::DeviceIndex device) {
    void* const stream = current_stream(device);
    // (in a captured stream nothing is allocated)
    const unsigned long long need = tcu_flash_attn_workspace_bytes(batch, M, N, D, P, v_layout);
    if (need > 0 && !capturing()) {
        const at::Tensor ws = bytes(like, need);
        void* const wp = ws.data_ptr();
        return succeeds([&] { return tcu_flash_attn_fwd_f16_ws(q, k, v, o, batch, M, N, D, P, scale, v_layout, wp, need, stream); });
    }
    return succeeds([&] { return tcu_flash_attn_fwd_f16(q, k, v, o, batch, M, N, D, P, scale, v_layout, stream); });
}

// flash_attention(q, k, v, scale)
PyObject* flash_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4 || !on_device(args[0]) || (args[3] != Py_None && !PyFloat_CheckExact(args[3]))) Py_RETURN_NONE;
    const auto device = current_device();
    const at::Tensor* t[3];
    for (int i = 0; i < 3; ++i)
        if (!(t[i] = plain(args[i], at::kHalf, device)) || t[i]->dim() != t[0]->dim()) Py_RETURN_NONE;
    const int64_t d = t[0]->dim();
    if (d < 2) Py_RETURN_NONE;
    int64_t batch = 1;
    for (int64_t i = 0; i + 2 < d; ++i) {
        if (t[1]->size(i) != t[0]->size(i) || t[2]->size(i) != t[0]->size(i)) Py_RETURN_NONE;
        batch *= t[0]->size(i);
        if (batch > INT_MAX) Py_RETURN_NONE;
    }
    const int M = int(t[0]->size(-2)), D = int(t[0]->size(-1)), N = int(t[1]->size(-2)), P = int(t[2]->size(-1));
    if (t[1]->size(-1) != D || t[2]->size(-2) != N) Py_RETURN_NONE;
    const float scale = float(args[3] == Py_None ? 1.0 / std::sqrt(double(D)) : PyFloat_AS_DOUBLE(args[3]));
    at::DimVector shape(t[0]->sizes());
    shape.back() = P;
    at::Tensor out = at::empty(shape, t[0]->options());
    if (!attention(t[0]->data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), out.data_ptr(), int(batch), M, N, D, P, scale, TCU_V_ROW_MAJOR,
                   *t[0], device))
        Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// flash_attention_fwd(Q, K, V, O, m, n, k, p, scale, batch) -> True
PyObject* flash_attention_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 10 || !on_device(args[0]) || !PyFloat_CheckExact(args[8])) Py_RETURN_NONE;
    const auto device = current_device();
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i)
        if (!(t[i] = plain(args[i], at::kHalf, device))) Py_RETURN_NONE;
    int64_t v[5];  // m, n, k, p, batch
    for (int i = 0; i < 5; ++i) {
        PyObject* const o = args[i < 4 ? 4 + i : 9];
        if (!PyLong_CheckExact(o)) Py_RETURN_NONE;
        int overflow = 0;
        v[i] = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow || v[i] <= 0 || v[i] > INT_MAX) Py_RETURN_NONE;
    }
    // (numel is below 2^62, and so is a product that equals one: compared as wide as needed)
    const auto holds = [&](const at::Tensor& x, int64_t rows, int64_t cols) { return __int128(v[4]) * rows * cols == x.numel(); };
    if (!holds(*t[0], v[0], v[2]) || !holds(*t[1], v[1], v[2]) || !holds(*t[2], v[3], v[1]) || !holds(*t[3], v[0], v[3])) Py_RETURN_NONE;
    if (!attention(t[0]->data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), t[3]->data_ptr(), int(v[4]), int(v[0]), int(v[1]), int(v[2]),
                   int(v[3]), float(PyFloat_AS_DOUBLE(args[8])), TCU_V_COL_MAJOR, *t[0], device))
        Py_RETURN_NONE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// lstm(x, W, bias, h0, c0) -> (h_all, c_T)
PyObject* lstm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5 || !on_device(args[0])) Py_RETURN_NONE;
    const auto device = current_device();
    const at::Tensor *x = plain(args[0], at::kHalf, device), *W = x ? plain(args[1], at::kHalf, device) : nullptr;
    const at::Tensor* bias = W ? plain(args[2], at::kHalf, device) : nullptr;
    if (!bias || x->dim() != 3 || W->dim() != 2 || bias->dim() != 1) Py_RETURN_NONE;
    const int T = int(x->size(0)), B = int(x->size(1)), I = int(x->size(2)), H = int(W->size(0) / 4);
    if (H == 0 || W->size(0) != 4 * int64_t(H) || W->size(1) != int64_t(I) + H || bias->size(0) != 4 * int64_t(H)) Py_RETURN_NONE;
    const void* state[2] = {nullptr, nullptr};
    for (int i = 0; i < 2; ++i) {
        if (args[3 + i] == Py_None) continue;
        const at::Tensor* s = plain(args[3 + i], i == 0 ? at::kHalf : at::kFloat, device);
        if (!s || s->dim() != 2 || s->size(0) != B || s->size(1) != H) Py_RETURN_NONE;
        state[i] = s->data_ptr();
    }
    at::Tensor h_all = at::empty({T, B, H}, x->options()), c_out = at::empty({B, H}, x->options().dtype(at::kFloat));
    void* const stream = current_stream(device);
    const void *xp = x->data_ptr(), *wp = W->data_ptr(), *bp = bias->data_ptr();
    void *hp = h_all.data_ptr(), *cp = c_out.data_ptr();
    bool ok;
    at::Tensor layer_ws;
    const unsigned long long layer_need = tcu_lstm_uses_layer(T, B, I, H) && !capturing() ? tcu_lstm_layer_workspace_bytes(T, B, I, H) : 0;
    if (layer_need > 0) layer_ws = bytes_if_free(*x, layer_need);
    if (layer_ws.defined()) {
        void* const sp = layer_ws.data_ptr();
        ok = succeeds([&] { return tcu_lstm_f16_layer(xp, wp, bp, state[0], state[1], hp, cp, T, B, I, H, sp, layer_need, stream); });
    } else if (tcu_lstm_uses_workspace(T, B, I, H)) {
        const unsigned long long need = tcu_lstm_workspace_bytes(T, B, I, H);
        const at::Tensor ws = bytes(*x, need);
        void* const sp = ws.data_ptr();
        ok = succeeds([&] { return tcu_lstm_f16_ws(xp, wp, bp, state[0], state[1], hp, cp, T, B, I, H, sp, need, stream); });
    } else {
        ok = succeeds([&] { return tcu_lstm_f16(xp, wp, bp, state[0], state[1], hp, cp, T, B, I, H, stream); });
    }
    if (!ok) Py_RETURN_NONE;
    THPObjectPtr pair(PyTuple_New(2));
    if (!pair) return nullptr;
    PyTuple_SET_ITEM(pair.get(), 0, THPVariable_Wrap(std::move(h_all)));
    PyTuple_SET_ITEM(pair.get(), 1, THPVariable_Wrap(std::move(c_out)));
    return pair.release();
    END_HANDLE_TH_ERRORS
}

// scatter_nd(data, indices, updates, mode) -> True
PyObject* scatter_nd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4 || !on_device(args[0]) || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    const auto device = current_device();
    const at::ScalarType type = THPVariable_Unpack(args[0]).scalar_type();
    if (type != at::kFloat && type != at::kHalf) Py_RETURN_NONE;
    const at::Tensor *data = plain(args[0], type, device), *indices = data ? plain(args[1], at::kLong, device) : nullptr;
    const at::Tensor* updates = indices ? plain(args[2], type, device) : nullptr;
    if (!updates || indices->dim() < 1) Py_RETURN_NONE;
    const int64_t k = indices->size(-1), rank = data->dim(), count = indices->numel() / k;
    if (k > rank || rank > 8) Py_RETURN_NONE;
    long long dims[8];
    int64_t slice = 1;
    for (int64_t i = 0; i < rank; ++i) {
        dims[i] = data->size(i);
        if (i >= k) slice *= dims[i];
    }
    if (__int128(count) * slice != updates->numel()) Py_RETURN_NONE;
    void* const stream = current_stream(device);
    void* const dp = data->data_ptr();
    const void *up = updates->data_ptr(), *ip = indices->data_ptr();
    const int mode = int(PyLong_AsLong(args[3])), dtype = type == at::kFloat ? TCU_DTYPE_F32 : TCU_DTYPE_F16;
    if (!succeeds([&] { return tcu_scatter_nd(dp, up, ip, dims, int(rank), count, int(k), dtype, mode, nullptr, stream); })) Py_RETURN_NONE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"gemm", reinterpret_cast<PyCFunction>(&gemm), METH_FASTCALL, nullptr},
    {"b2b_gemm", reinterpret_cast<PyCFunction>(&b2b_gemm), METH_FASTCALL, nullptr},
    {"flash_attention", reinterpret_cast<PyCFunction>(&flash_attention), METH_FASTCALL, nullptr},
    {"flash_attention_fwd", reinterpret_cast<PyCFunction>(&flash_attention_fwd), METH_FASTCALL, nullptr},
    {"lstm", reinterpret_cast<PyCFunction>(&lstm), METH_FASTCALL, nullptr},
    {"scatter_nd", reinterpret_cast<PyCFunction>(&scatter_nd), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__calls() {
    // torch's C++ classes are those of the release that this was compiled against
    THPObjectPtr torch(PyImport_ImportModule("torch")), version(torch ? PyObject_GetAttrString(torch.get(), "__version__") : nullptr);
    THPObjectPtr text(version ? PyObject_Str(version.get()) : nullptr);
    const char* const running = text ? PyUnicode_AsUTF8(text.get()) : nullptr;
    if (!running) return nullptr;
    if (std::strcmp(running, TCU_TORCH_VERSION) != 0)
        return PyErr_Format(PyExc_ImportError, "compiled for torch %s, this is %s", TCU_TORCH_VERSION, running);
    return PyModule_Create(&kModule);
}
