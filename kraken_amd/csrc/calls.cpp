// The common forms of the package's calls, from the Python arguments to the launch in one native step.
//
// A call whose kernel takes a few microseconds is bound by its host path: reading a tensor's properties from Python costs
// 0.05 to 0.1 us each, a tensor or stream object 1 to 2, and a call needs some thirty of them where the launch itself
// takes 3.  Each function here takes the arguments of one wrapper, looks at them directly and launches; where anything
// is not of the plain form (another type, layout, device, alignment, a list of buffers, a subclass, sizes that do not
// fit, an error code of the library) it launches nothing and returns None, and the wrapper's general path, which
// has every check and message, runs instead.  So nothing is accepted here that the general path does not accept, and
// the library gets the same arguments from both.
// Host time of one call, us, general path / here: 16 rows of 8192, W = 8, reduce + RMSNorm 8.9 / 4.1; RMSNorm alone
// 7.5 / 4.9; 8 x 1024 x 1024 product + all-reduce 11.7 / 4.7, + reduce-scatter 12.9 / 5.5.  Calls one behind the other: fp32
// operands, one row of 3328 x 768 with seven peers 22.2 / 6.6, 47 x 2176 x 704 18.2 / 9.1; copy-engine reduce-scatter 32 x 1216 x 1024 18.6 /
// 10.6; gather + product, 4 shards of 2 x 1088, N = 5728 22.4 / 11.4, 8 of 16 x 1792, N = 1152 27.7 / 18.9 (fp8 29.8 / 23.2).
//
// The entry points of libkraken_amd.so and the helpers in Python are handed over by bind(); this file keeps nothing else.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/core/grad_mode.h>

#include "../../include/kraken_amd.h"

namespace {

// ---- bound once, when the module is loaded ------------------------------------------------------
decltype(&kr_reduce_bf16) reduce_bf16;
decltype(&kr_reduce_ptrs_bf16) reduce_ptrs_bf16;
decltype(&kr_reduce_striped_bf16) reduce_striped_bf16;
decltype(&kr_reduce_striped_ptrs_bf16) reduce_striped_ptrs_bf16;
decltype(&kr_striped_share_numel) striped_share_numel;
decltype(&kr_rmsnorm_workspace_bytes) rmsnorm_workspace_bytes;
decltype(&kr_reduce_rmsnorm_ws_bf16) reduce_rmsnorm_ws_bf16;
decltype(&kr_reduce_rmsnorm_ptrs_ws_bf16) reduce_rmsnorm_ptrs_ws_bf16;
decltype(&kr_rmsnorm_bf16) rmsnorm_bf16;
decltype(&kr_gemm_workspace_bytes) gemm_workspace_bytes;
decltype(&kr_gemm_reduce_bf16) gemm_reduce_bf16;
decltype(&kr_gemm_reduce_ws_bf16) gemm_reduce_ws_bf16;
decltype(&kr_gemm_f32_pairs) gemm_f32_pairs;
decltype(&kr_gemm_f32_workspace_bytes) gemm_f32_workspace_bytes;
decltype(&kr_gemm_reduce_f32_ws) gemm_reduce_f32_ws;
decltype(&kr_split_pairs_fp32) split_pairs_fp32;
decltype(&kr_gemm_pairs_workspace_bytes) gemm_pairs_workspace_bytes;
decltype(&kr_gemm_reduce_pairs_ws) gemm_reduce_pairs_ws;
decltype(&kr_reduce_rotated_ptrs_bf16) reduce_rotated_ptrs_bf16;
decltype(&kr_gather_chunks) gather_chunks;
decltype(&kr_gather_matmul_direct) gather_matmul_direct;
decltype(&kr_gather_matmul_bf16) gather_matmul_bf16;
decltype(&kr_gemm_fp8_workspace_bytes) gemm_fp8_workspace_bytes;
decltype(&kr_gemm_fp8_ws) gemm_fp8_ws;
decltype(&kr_gemm_fp8_wide_workspace_bytes) gemm_fp8_wide_workspace_bytes;
decltype(&kr_gemm_fp8_wide_ws) gemm_fp8_wide_ws;
PyObject* raw_stream;       // device index -> handle of its current stream
PyObject* row_exchange;     // (device index, bytes, stream) -> (workspace tensor, status tensor) of the split-row kernel
PyObject* row_watch;        // (status tensor): look at it once the work enqueued so far is done
PyObject* gemm_workspace;   // (device index, bytes, stream) -> workspace tensor or None
PyObject* waits_check;      // (): raises if a bounded wait of an earlier call ran out

struct Ref {                // a reference that is given back
    PyObject* p;
    explicit Ref(PyObject* o) : p(o) {}
    ~Ref() { Py_XDECREF(p); }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
};

struct NoGil {              // other Python threads run while the library is in a launch
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// A tensor of a plain form: strided memory on a HIP device, no subclass and nothing a transform has wrapped.
const at::Tensor* plain(PyObject* o, at::ScalarType type) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    using K = c10::DispatchKey;
    static const c10::DispatchKeySet wrapped({K::Functionalize, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Python});
    if (!t.defined() || t.scalar_type() != type || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
        t.key_set().has_any(wrapped))
        return nullptr;
    return &t;
}

const at::Tensor* contiguous(PyObject* o, at::ScalarType type = at::kBFloat16) {
    const at::Tensor* t = plain(o, type);
    return t != nullptr && t->is_contiguous() ? t : nullptr;
}

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

bool integer(PyObject* o, int64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

bool stream_of(const at::Tensor& t, void*& stream) {
    const Ref index(PyLong_FromLong(t.get_device()));
    if (index.p == nullptr) return false;
    const Ref handle(PyObject_CallOneArg(raw_stream, index.p));
    if (handle.p == nullptr) return false;
    stream = PyLong_AsVoidPtr(handle.p);
    return PyErr_Occurred() == nullptr;
}

// The W buffers of a reduce: contiguous slices of one tensor, entry `rank` replaced by an input of its own.
struct Sources {
    const char* base = nullptr;
    int W = 0;
    int64_t cap = 0, stride = 0;      // elements of a slice, from slice to slice
    const void* table[KR_MAX_WORLD];
    bool stacked = true;      // false: the addresses are in `table`

    bool of(const at::Tensor& stack) {
        if (stack.dim() < 2 || stack.size(0) < 1 || stack.size(0) > KR_MAX_WORLD || stack.numel() == 0) return false;
        W = (int)stack.size(0);
        cap = stack.numel() / W;
        stride = W > 1 ? stack.stride(0) : cap;
        if (!stack.is_contiguous() && !stack.select(0, 0).is_contiguous()) return false;
        base = (const char*)stack.const_data_ptr();
        return true;
    }
    bool replace(int64_t rank, const at::Tensor& x) {
        const void* p = x.const_data_ptr();
        if (p == base + rank * stride * 2) return true;
        if (!aligned(p)) return false;
        for (int r = 0; r < W; ++r) table[r] = base + r * stride * 2;
        table[rank] = p;
        stacked = false;
        return true;
    }
};

#define KR_NOT_HERE return Py_NewRef(Py_None)

// one_shot_all_reduce(stack) -> result
PyObject* all_reduce(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const at::Tensor* stack = n_args == 1 ? plain(args[0], at::kBFloat16) : nullptr;
    Sources s;
    if (stack == nullptr || !s.of(*stack) || s.cap % 8 != 0) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*stack, stream)) return nullptr;
    at::Tensor out;
    int rc;
    {
        const NoGil released;
        out = at::empty(stack->sizes().slice(1), stack->options());
        rc = reduce_bf16(s.base, s.W, s.stride, s.cap, nullptr, 0, 0, 1, out.mutable_data_ptr(), stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// one_shot_all_reduce_bias(stack, x, bias, output, rank) -> True
PyObject* all_reduce_bias(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 5) KR_NOT_HERE;
    const at::Tensor *stack = plain(args[0], at::kBFloat16), *out = contiguous(args[3]);
    const at::Tensor *x = args[1] == Py_None ? nullptr : contiguous(args[1]), *bias = args[2] == Py_None ? nullptr : contiguous(args[2]);
    Sources s;
    int64_t rank;
    if (stack == nullptr || out == nullptr || (x == nullptr && args[1] != Py_None) || (bias == nullptr && args[2] != Py_None) ||
        !s.of(*stack) || !integer(args[4], rank) || rank < 0 || rank >= s.W)
        KR_NOT_HERE;
    const at::Tensor& ref = x != nullptr ? *x : *out;
    const int64_t numel = ref.numel(), D = ref.dim() >= 1 ? ref.size(-1) : numel, index = stack->get_device();
    if (numel == 0 || numel % 8 != 0 || out->numel() != numel || numel > s.cap || out->get_device() != index) KR_NOT_HERE;
    if (bias != nullptr && ((bias->numel() != numel && bias->numel() != D) || bias->get_device() != index)) KR_NOT_HERE;
    if (x != nullptr && (x->get_device() != index || !s.replace(rank, *x))) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*stack, stream)) return nullptr;
    int rc;
    {
        const NoGil released;
        const void* bp = bias != nullptr ? bias->const_data_ptr() : nullptr;
        const int64_t bn = bias != nullptr ? bias->numel() : 0;
        void* op = out->mutable_data_ptr();
        rc = s.stacked ? reduce_bf16(s.base, s.W, s.stride, numel, bp, bn, D, 1, op, stream)
                       : reduce_ptrs_bf16(s.table, s.W, numel, bp, bn, D, 1, op, stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// one rank's share of a two-shot reduce of n elements; `out` may be any size the caller has checked
int two_shot(const Sources& s, int64_t n, bool striped, int64_t block, int64_t rank, const at::Tensor* bias, int64_t D, void* out,
             int64_t out_numel, void* stream) {
    const void* bp = bias != nullptr ? bias->const_data_ptr() : nullptr;
    int64_t bn = bias != nullptr ? bias->numel() : 0, off = 0;
    if (out_numel != n && striped)
        return s.stacked ? reduce_striped_bf16(s.base, s.W, s.stride, n, bp, block, (int)rank, out, stream)
                         : reduce_striped_ptrs_bf16(s.table, s.W, n, bp, block, (int)rank, out, stream);
    if (out_numel != n) {
        off = rank * out_numel;
        if (bn == n) {
            bp = (const uint16_t*)bp + off;
            bn = out_numel;
        }
    }
    if (s.stacked) return reduce_bf16(s.base + 2 * off, s.W, s.stride, out_numel, bp, bn, D, 0, out, stream);
    const void* table[KR_MAX_WORLD];
    for (int r = 0; r < s.W; ++r) table[r] = (const uint16_t*)s.table[r] + off;
    return reduce_ptrs_bf16(table, s.W, out_numel, bp, bn, D, 0, out, stream);
}

// two_shot_all_reduce(stack, rank, striped, block) -> this rank's share
PyObject* two_shot_share(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const at::Tensor* stack = n_args == 4 ? plain(args[0], at::kBFloat16) : nullptr;
    Sources s;
    int64_t rank, block;
    if (stack == nullptr || !s.of(*stack) || s.cap % 8 != 0 || !integer(args[1], rank) || rank < 0 || rank >= s.W ||
        !integer(args[3], block) || block < 1 || block % s.W != 0)
        KR_NOT_HERE;
    const bool striped = args[2] == Py_True;
    const int64_t share = striped ? striped_share_numel(s.cap, s.W, block, (int)rank) : s.cap / s.W;
    if (share <= 0 || (!striped && (s.cap % s.W != 0 || share % 8 != 0))) KR_NOT_HERE;
    std::vector<int64_t> shape{share};
    if (!striped && stack->size(1) % s.W == 0) {
        shape.assign(stack->sizes().begin() + 1, stack->sizes().end());
        shape[0] /= s.W;
    }
    void* stream;
    if (!stream_of(*stack, stream)) return nullptr;
    at::Tensor out;
    int rc;
    {
        const NoGil released;
        out = at::empty(shape, stack->options());
        // (one rank owns everything: the general path passes an offset of 0 as well)
        rc = striped ? reduce_striped_bf16(s.base, s.W, s.stride, s.cap, nullptr, block, (int)rank, out.mutable_data_ptr(), stream)
                     : two_shot(s, s.cap, false, block, rank, nullptr, 0, out.mutable_data_ptr(), share, stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// two_shot_all_reduce_bias(stack, x, bias, output, block, rank, striped, numel or None) -> True
PyObject* two_shot_bias(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 8) KR_NOT_HERE;
    const at::Tensor *stack = plain(args[0], at::kBFloat16), *out = contiguous(args[3]);
    const at::Tensor *x = args[1] == Py_None ? nullptr : contiguous(args[1]), *bias = args[2] == Py_None ? nullptr : contiguous(args[2]);
    Sources s;
    int64_t block, rank, n;
    if (stack == nullptr || out == nullptr || (x == nullptr && args[1] != Py_None) || (bias == nullptr && args[2] != Py_None) ||
        !s.of(*stack) || !integer(args[4], block) || block < 1 || block % s.W != 0 || !integer(args[5], rank) || rank < 0 || rank >= s.W)
        KR_NOT_HERE;
    const bool striped = args[6] == Py_True;
    const int64_t on = out->numel(), index = stack->get_device();
    if (x != nullptr) n = x->numel();
    else if (args[7] != Py_None) {
        if (!integer(args[7], n)) KR_NOT_HERE;
    } else n = on == s.cap || on * s.W == s.cap || striped ? s.cap : on * s.W;
    if (n <= 0 || n % 8 != 0 || n > s.cap || out->get_device() != index) KR_NOT_HERE;
    if (x != nullptr && x->dim() < 1) KR_NOT_HERE;
    const int64_t D = x != nullptr ? x->size(-1) : stack->size(-1);
    if (on != n) {
        const int64_t share = striped ? striped_share_numel(n, s.W, block, (int)rank) : n / s.W;
        if (share <= 0 || on != share || (!striped && (n % s.W != 0 || share % 8 != 0))) KR_NOT_HERE;
    }
    if (bias != nullptr) {
        const int64_t bn = bias->numel();
        if (bias->get_device() != index || !(bn == n || (bn == D && (on == n || (!striped && on % D == 0))))) KR_NOT_HERE;
    }
    if (x != nullptr && (x->get_device() != index || !s.replace(rank, *x))) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*stack, stream)) return nullptr;
    int rc;
    {
        const NoGil released;
        rc = two_shot(s, n, striped, block, rank, bias, D, out->mutable_data_ptr(), on, stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// *_all_reduce_bias_rms_norm(stack, x, bias, w, y, eps, rank) -> True
PyObject* reduce_rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 7) KR_NOT_HERE;
    const at::Tensor *stack = plain(args[0], at::kBFloat16), *w = contiguous(args[3]), *y = contiguous(args[4]);
    const at::Tensor *x = args[1] == Py_None ? nullptr : contiguous(args[1]), *bias = args[2] == Py_None ? nullptr : contiguous(args[2]);
    Sources s;
    int64_t rank;
    if (stack == nullptr || w == nullptr || y == nullptr || (x == nullptr && args[1] != Py_None) || (bias == nullptr && args[2] != Py_None) ||
        !s.of(*stack) || !PyFloat_CheckExact(args[5]) || !integer(args[6], rank) || rank < 0 || rank >= s.W)
        KR_NOT_HERE;
    const int64_t index = stack->get_device();
    if (y->dim() < 1 || y->numel() == 0 || y->get_device() != index || w->get_device() != index) KR_NOT_HERE;
    const int64_t D = y->size(-1), numel = y->numel(), rows = numel / D;
    if (D % 8 != 0 || w->dim() != 1 || w->size(0) != D || numel > s.cap) KR_NOT_HERE;
    if (bias != nullptr && ((bias->numel() != numel && bias->numel() != D) || bias->get_device() != index)) KR_NOT_HERE;
    if (x != nullptr && (x->get_device() != index || x->sizes() != y->sizes() || x->strides() != y->strides() || !s.replace(rank, *x))) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*stack, stream)) return nullptr;
    // a few long rows: their wavefronts meet in the stream's workspace and report through its status word
    const int64_t bytes = rmsnorm_workspace_bytes(s.W, rows, D);
    const Ref exchange(bytes > 0 ? PyObject_CallFunction(row_exchange, "LLK", (long long)index, (long long)bytes, (unsigned long long)(uintptr_t)stream) : nullptr);
    void* ws = nullptr;
    int64_t ws_bytes = 0;
    int32_t* status = nullptr;
    if (bytes > 0) {
        if (exchange.p == nullptr) return nullptr;
        const at::Tensor &ws_t = THPVariable_Unpack(PyTuple_GET_ITEM(exchange.p, 0)), &st_t = THPVariable_Unpack(PyTuple_GET_ITEM(exchange.p, 1));
        ws = ws_t.mutable_data_ptr();
        ws_bytes = ws_t.numel();
        status = (int32_t*)st_t.mutable_data_ptr();
    }
    int rc;
    {
        const NoGil released;
        const void* bp = bias != nullptr ? bias->const_data_ptr() : nullptr;
        const int vec = bias != nullptr && bias->numel() == D && rows != 1;
        const void* wp = w->const_data_ptr();
        void* yp = y->mutable_data_ptr();
        const float eps = (float)PyFloat_AS_DOUBLE(args[5]);
        rc = s.stacked ? reduce_rmsnorm_ws_bf16(s.base, s.W, s.stride, rows, D, bp, vec, wp, eps, yp, ws, ws_bytes, status, stream)
                       : reduce_rmsnorm_ptrs_ws_bf16(s.table, s.W, rows, D, bp, vec, wp, eps, yp, ws, ws_bytes, status, stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    if (bytes > 0) {
        const Ref done(PyObject_CallOneArg(row_watch, PyTuple_GET_ITEM(exchange.p, 1)));
        if (done.p == nullptr) return nullptr;
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// rms_norm(x, w, eps) -> y
PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 3) KR_NOT_HERE;
    const at::Tensor *x = contiguous(args[0]), *w = contiguous(args[1]);
    if (x == nullptr || w == nullptr || !PyFloat_CheckExact(args[2]) || x->dim() < 1 || x->numel() == 0 || x->get_device() != w->get_device()) KR_NOT_HERE;
    const int64_t D = x->size(-1);
    if (D % 8 != 0 || w->dim() != 1 || w->size(0) != D) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*x, stream)) return nullptr;
    at::Tensor y;
    int rc;
    {
        const NoGil released;
        y = at::empty_like(*x);
        rc = rmsnorm_bf16(x->const_data_ptr(), w->const_data_ptr(), (float)PyFloat_AS_DOUBLE(args[2]),
                          x->numel() / D, D, y.mutable_data_ptr(), stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// What a product does where its operands are of a form the kernels read: launched, left to the general path, or a Python error.
enum Done { kLaunched, kNotHere, kError };

// The stream's scratch, `bytes` of it; none where none is needed or to be had.
struct Scratch {
    Ref tensor;
    void* p = nullptr;
    int64_t bytes = 0;
    Scratch(int64_t index, int64_t need, void* stream)
        : tensor(need > 0 ? PyObject_CallFunction(gemm_workspace, "LLK", (long long)index, (long long)need, (unsigned long long)(uintptr_t)stream) : nullptr) {
        if (tensor.p == nullptr || tensor.p == Py_None) return;
        const at::Tensor& t = THPVariable_Unpack(tensor.p);
        p = t.mutable_data_ptr();
        bytes = t.numel();
    }
};

// out [rows, N] = (a @ b)[row0 .. row0 + rows - 1] + peers + bias, the other rows to c_full; a and b both bf16, or both fp32
Done product(const at::Tensor& a, const at::Tensor& b, const at::Tensor* peers, const at::Tensor* bias, const at::Tensor* c_full, int64_t row0,
             int64_t rows, bool out_fp32, int64_t pivot, void* stream, at::Tensor& out) {
    const bool f32 = a.scalar_type() == at::kFloat;
    if (a.dim() != 2 || b.dim() != 2 || a.size(1) != b.size(0) || b.scalar_type() != a.scalar_type()) return kNotHere;
    const int64_t M = a.size(0), N = b.size(1), K = a.size(1), index = a.get_device(), unit = f32 ? 4 : 8;
    if (M == 0 || N == 0 || K == 0 || N % 8 != 0 || K % 8 != 0 || rows < 1 || row0 < 0 || row0 + rows > M || b.get_device() != index) return kNotHere;
    if (a.stride(1) != 1 || a.stride(0) % unit != 0 || !aligned(a.const_data_ptr()) || !aligned(b.const_data_ptr())) return kNotHere;
    if (!(b.stride(1) == 1 && b.stride(0) % unit == 0) && !(b.stride(0) == 1 && b.stride(1) % unit == 0)) return kNotHere;
    if (peers != nullptr && (peers->dim() != 3 || peers->size(0) < 1 || peers->size(0) >= KR_MAX_WORLD || peers->size(1) != rows ||
                             peers->size(2) != N || peers->get_device() != index))
        return kNotHere;
    if (bias != nullptr && (bias->dim() != 1 || bias->size(0) != N || bias->get_device() != index)) return kNotHere;
    if (c_full != nullptr && (c_full->dim() != 2 || c_full->size(0) != M || c_full->size(1) != N || c_full->get_device() != index)) return kNotHere;
    // (fp32: strides the kernels refuse, and more tiles than the one that splits in registers is for, go the general way)
    bool pairs = f32 && gemm_f32_pairs(M, N, K) == 1;
    const bool few = ((M + 127) / 128) * ((N + 127) / 128) <= 512;
    if (f32 && (a.stride(0) < K || (b.stride(1) == 1 ? b.stride(0) < N : b.stride(1) < K))) return kNotHere;
    if (f32 && !pairs && !few) return kNotHere;
    at::Tensor parts;
    {
        const NoGil released;
        out = at::empty({rows, N}, a.options().dtype(out_fp32 ? at::kFloat : at::kBFloat16));
        if (pairs) {
            try {
                parts = at::empty({M + N, (K + 31) / 32 * 64}, a.options().dtype(at::kBFloat16));
            } catch (const c10::OutOfMemoryError&) {     // (in registers it needs no memory)
                if (!few) throw;
                pairs = false;
            }
        }
    }
    const Scratch ws(index, pairs ? gemm_pairs_workspace_bytes(M, N, K) : f32 ? gemm_f32_workspace_bytes(M, N, K) : gemm_workspace_bytes(M, N, K), stream);
    if (PyErr_Occurred()) return kError;
    const NoGil released;
    const void *ap = a.const_data_ptr(), *bp = b.const_data_ptr();
    const void* pp = peers != nullptr ? peers->const_data_ptr() : nullptr;
    const void* biasp = bias != nullptr ? bias->const_data_ptr() : nullptr;
    void* cp = c_full != nullptr ? c_full->mutable_data_ptr() : nullptr;
    void* op = out.mutable_data_ptr();
    const int P = peers != nullptr ? (int)peers->size(0) : 0;
    const int64_t pstride = peers != nullptr ? rows * N : 0;
    int rc;
    if (f32) {
        const void* table[KR_MAX_WORLD];
        for (int q = 0; q < P; ++q) table[q] = (const uint16_t*)pp + q * pstride;
        if (pairs) {
            uint16_t *apart = (uint16_t*)parts.mutable_data_ptr(), *bpart = apart + M * parts.size(1);
            rc = split_pairs_fp32(ap, a.stride(0), bp, b.stride(0), b.stride(1), M, N, K, apart, bpart, stream);
            if (rc == KR_OK)
                rc = gemm_reduce_pairs_ws(apart, bpart, M, N, K, table, P, biasp, row0, rows, cp, op, out_fp32, pivot, ws.p, ws.bytes, stream);
        } else {
            rc = gemm_reduce_f32_ws(ap, a.stride(0), 1, bp, b.stride(0), b.stride(1), M, N, K, table, P, biasp, row0, rows, cp, op, out_fp32, pivot, ws.p,
                                    ws.bytes, stream);
        }
    } else {
        rc = ws.bytes > 0 ? gemm_reduce_ws_bf16(ap, a.stride(0), 1, bp, b.stride(0), b.stride(1), M, N, K, pp, P, pstride, biasp, row0, rows, cp, op,
                                                out_fp32, pivot, ws.p, ws.bytes, stream)
                          : gemm_reduce_bf16(ap, a.stride(0), 1, bp, b.stride(0), b.stride(1), M, N, K, pp, P, pstride, biasp, row0, rows, cp, op,
                                             out_fp32, pivot, stream);
    }
    return rc == KR_OK ? kLaunched : kNotHere;
}

// gemm(a, b, peers, bias, c_full, band_row0, band_rows, out_fp32, pivot) -> out [band_rows, N]: bf16 or fp32 operands in a
// layout the kernels read, peers [P, band_rows, N] as one tensor or None
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 9) KR_NOT_HERE;
    const at::Tensor* a = plain(args[0], at::kBFloat16);
    if (a == nullptr) a = plain(args[0], at::kFloat);
    if (a == nullptr) KR_NOT_HERE;
    const at::Tensor* b = plain(args[1], a->scalar_type());
    const at::Tensor *peers = args[2] == Py_None ? nullptr : contiguous(args[2]), *bias = args[3] == Py_None ? nullptr : contiguous(args[3]);
    const at::Tensor* c_full = args[4] == Py_None ? nullptr : contiguous(args[4]);
    int64_t row0, rows, pivot;
    if (b == nullptr || (peers == nullptr && args[2] != Py_None) || (bias == nullptr && args[3] != Py_None) ||
        (c_full == nullptr && args[4] != Py_None) || !integer(args[5], row0) || !integer(args[6], rows) || !integer(args[8], pivot))
        KR_NOT_HERE;
    void* stream;
    if (!stream_of(*a, stream)) return nullptr;
    at::Tensor out;
    const Done done = product(*a, *b, peers, bias, c_full, row0, rows, args[7] == Py_True, pivot, stream, out);
    if (done == kError) return nullptr;
    if (done == kNotHere) KR_NOT_HERE;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

struct Bytes {              // of device memory, [lo, hi)
    const char *lo, *hi;
    explicit Bytes(const at::Tensor& t) : lo((const char*)t.const_data_ptr()), hi(lo) {
        int64_t last = t.numel() > 0 ? 1 : 0;
        for (int64_t d = 0; t.numel() > 0 && d < t.dim(); ++d) last += (t.size(d) - 1) * t.stride(d);
        hi = lo + last * t.element_size();
    }
    bool apart(const Bytes& o) const { return hi <= o.lo || o.hi <= lo; }
};

// reduce_scatter_sent(a, b, peers, sent, rank, round_each) -> out [M / W, N]: the copy-engine form whose product stores the other
// ranks' bands in `sent` itself, everything in memory of its own
PyObject* reduce_scatter_sent(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 6) KR_NOT_HERE;
    const at::Tensor *a = plain(args[0], at::kBFloat16), *b = plain(args[1], at::kBFloat16), *peers = contiguous(args[2]), *sent = contiguous(args[3]);
    int64_t rank;
    if (a == nullptr || b == nullptr || peers == nullptr || sent == nullptr || !integer(args[4], rank)) KR_NOT_HERE;
    if (a->dim() != 2 || b->dim() != 2 || peers->dim() != 3 || sent->dim() != 3 || a->size(0) == 0 || b->size(1) == 0) KR_NOT_HERE;
    const int64_t W = peers->size(0) + 1, M = a->size(0), N = b->size(1), index = a->get_device();
    if (W < 2 || W > KR_MAX_WORLD || M % W != 0 || rank < 0 || rank >= W) KR_NOT_HERE;
    const int64_t rows = M / W;
    if (peers->size(1) != rows || peers->size(2) != N || peers->get_device() != index) KR_NOT_HERE;
    if (sent->size(0) != W || sent->size(1) != rows || sent->size(2) != N || sent->get_device() != index) KR_NOT_HERE;
    if (sent->requires_grad() || sent->is_inference() || !aligned(sent->const_data_ptr()) || !aligned(peers->const_data_ptr()) || rows * N % 8 != 0) KR_NOT_HERE;
    const Bytes written(*sent);
    if (!written.apart(Bytes(*a)) || !written.apart(Bytes(*b)) || !written.apart(Bytes(*peers))) KR_NOT_HERE;
    const Ref checked(PyObject_CallNoArgs(waits_check));     // (raises for an earlier call's wait that ran out)
    if (checked.p == nullptr) return nullptr;
    void* stream;
    if (!stream_of(*a, stream)) return nullptr;
    at::Tensor own;
    {
        const at::Tensor c_full = sent->detach().view({M, N});     // (the same memory)
        const Done done = product(*a, *b, nullptr, nullptr, &c_full, rank * rows, rows, false, (rank + 1) % W * rows, stream, own);
        if (done == kError) return nullptr;
        if (done == kNotHere) KR_NOT_HERE;
    }
    at::Tensor out;
    int rc;
    {
        const NoGil released;
        sent->unsafeGetTensorImpl()->bump_version();
        out = at::empty({rows, N}, a->options());
        const void* table[KR_MAX_WORLD];
        for (int64_t r = 0, q = 0; r < W; ++r) table[r] = r == rank ? own.const_data_ptr() : (const uint16_t*)peers->const_data_ptr() + q++ * rows * N;
        rc = reduce_rotated_ptrs_bf16(table, (int)W, rows, N, (int)rank, args[5] == Py_True, out.mutable_data_ptr(), stream);
    }
    if (rc != KR_OK) KR_NOT_HERE;     // (the general path does all of it again)
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// out [M, N] = a @ b on fp8 operands, b transposed-contiguous
Done product_fp8(const at::Tensor& a, int64_t M, int64_t K, const at::Tensor& b, int64_t pivot, void* stream, at::Tensor& out) {
    const int64_t N = b.size(1);
    if (K % 16 != 0 || N % 16 != 0 || !aligned(a.const_data_ptr()) || !aligned(b.const_data_ptr())) return kNotHere;
    const bool whole = M % 256 == 0 && N % 256 == 0 && K % 128 == 0;     // (sums of 16 bits; the others keep 24)
    const Scratch ws(a.get_device(), whole ? gemm_fp8_workspace_bytes(M, N, K) : gemm_fp8_wide_workspace_bytes(M, N, K), stream);
    if (PyErr_Occurred()) return kError;
    const NoGil released;
    out = at::empty({M, N}, a.options());
    const int rc = whole ? gemm_fp8_ws(a.const_data_ptr(), K, b.const_data_ptr(), K, M, N, K, out.mutable_data_ptr(), 2, ws.p, ws.bytes, stream)
                         : gemm_fp8_wide_ws(a.const_data_ptr(), K, b.const_data_ptr(), K, M, N, K, out.mutable_data_ptr(), pivot, ws.p, ws.bytes, stream);
    return rc == KR_OK ? kLaunched : kNotHere;
}

// gather_matmul(shards, b, a_out, progress, rank, splits, gather) -> (gathered, c).  gather: a list of shards or a stack, and a
// matrix and flags of the caller's, all plain memory apart from each other that autograd does not follow; else a stack that is the
// gathered matrix, and neither.
PyObject* gather_matmul(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 7) KR_NOT_HERE;
    const bool gather = args[6] == Py_True, listed = PyList_CheckExact(args[0]);
    int64_t rank, splits;
    if (!integer(args[4], rank) || !integer(args[5], splits) || splits < 1) KR_NOT_HERE;
    PyObject* first = listed ? (PyList_GET_SIZE(args[0]) > 0 ? PyList_GET_ITEM(args[0], 0) : nullptr) : args[0];
    if (first == nullptr) KR_NOT_HERE;
    at::ScalarType type = at::kBFloat16;
    const at::Tensor* s0 = contiguous(first);
    if (s0 == nullptr) s0 = contiguous(first, type = at::kFloat8_e4m3fn);
    if (s0 == nullptr || s0->dim() != (listed ? 2 : 3) || s0->numel() == 0) KR_NOT_HERE;
    const int64_t W = listed ? PyList_GET_SIZE(args[0]) : s0->size(0), m = s0->size(listed ? 0 : 1), K = s0->size(listed ? 1 : 2), M = W * m;
    const at::Tensor* b = plain(args[1], type);
    if (W > KR_MAX_WORLD || rank < 0 || rank >= W || b == nullptr || b->dim() != 2 || b->size(0) != K || b->size(1) == 0 || b->stride(0) != 1 ||
        b->stride(1) != K || b->get_device() != s0->get_device())
        KR_NOT_HERE;
    const int64_t N = b->size(1), index = s0->get_device(), esize = s0->element_size();
    if (N % 8 != 0 || K % 8 != 0 || !aligned(b->const_data_ptr())) KR_NOT_HERE;
    const bool fp8 = type == at::kFloat8_e4m3fn;
    if (fp8 && (N % 16 != 0 || K % 16 != 0)) KR_NOT_HERE;
    void* stream;
    if (!stream_of(*s0, stream)) return nullptr;
    at::Tensor c, whole;
    if (!gather) {
        if (listed || args[2] != Py_None || args[3] != Py_None) KR_NOT_HERE;
        whole = s0->view({M, K});
        const Done done = fp8 ? product_fp8(whole, M, K, *b, rank * m, stream, c) : product(whole, *b, nullptr, nullptr, nullptr, 0, M, false, rank * m, stream, c);
        if (done == kError) return nullptr;
        if (done == kNotHere) KR_NOT_HERE;
    } else {
        const at::Tensor *a_out = contiguous(args[2], type), *progress = contiguous(args[3], at::kInt);
        if (a_out == nullptr || progress == nullptr || a_out->dim() != 2 || a_out->size(0) != M || a_out->size(1) != K || a_out->get_device() != index ||
            progress->get_device() != index || progress->numel() < W * splits || m % splits != 0)
            KR_NOT_HERE;
        const bool recording = at::GradMode::is_enabled();
        if (a_out->is_inference() || progress->is_inference() || progress->requires_grad() || (recording && a_out->requires_grad())) KR_NOT_HERE;
        const int64_t size = m * K * esize, chunk = size / splits;
        const char* to = (const char*)a_out->const_data_ptr();
        if (!aligned(to) || chunk % 16 != 0) KR_NOT_HERE;
        const void* from[KR_MAX_WORLD];
        for (int64_t r = 0; r < W; ++r) {
            const at::Tensor* t = listed && r > 0 ? contiguous(PyList_GET_ITEM(args[0], r), type) : s0;
            if (t == nullptr || t->sizes() != s0->sizes() || t->get_device() != index || (recording && t->requires_grad())) KR_NOT_HERE;
            const char* p = (const char*)t->const_data_ptr() + (listed ? 0 : r * size);
            if (!aligned(p) || !(p + size <= to || p >= to + W * size)) KR_NOT_HERE;
            from[r] = p;
        }
        const Bytes flags(*progress), result(*a_out);
        if (!flags.apart(result) || !result.apart(Bytes(*b))) KR_NOT_HERE;
        const bool direct = !fp8 && gather_matmul_direct((int)W, m, N, K) == 1;
        const Ref checked(PyObject_CallNoArgs(waits_check));     // (raises for an earlier call's wait that ran out)
        if (checked.p == nullptr) return nullptr;
        int rc;
        {
            const NoGil released;
            progress->fill_(0);
            if (direct) c = at::empty({M, N}, s0->options());
            rc = direct ? gather_matmul_bf16(from, (int)W, (int)rank, m, a_out->mutable_data_ptr(), b->const_data_ptr(), K, N, K, c.mutable_data_ptr(), stream)
                        : gather_chunks(from, (int)W, (int)splits, (int)rank, chunk, a_out->mutable_data_ptr(), (uint32_t*)progress->mutable_data_ptr(), stream);
            if (rc == KR_OK) {
                a_out->unsafeGetTensorImpl()->bump_version();
                if (direct) progress->view(-1).slice(0, 0, W * splits).fill_(1);
            }
        }
        if (rc != KR_OK) KR_NOT_HERE;
        if (!direct) {
            const Done done = fp8 ? product_fp8(*a_out, M, K, *b, rank * m, stream, c) : product(*a_out, *b, nullptr, nullptr, nullptr, 0, M, false, rank * m, stream, c);
            if (done == kError) return nullptr;
            if (done == kNotHere) KR_NOT_HERE;     // (the general path gathers again)
        }
        whole = *a_out;
    }
    const Ref gathered(gather ? Py_NewRef(args[2]) : THPVariable_Wrap(whole)), result(THPVariable_Wrap(c));
    if (gathered.p == nullptr || result.p == nullptr) return nullptr;
    return PyTuple_Pack(2, gathered.p, result.p);
    END_HANDLE_TH_ERRORS
}

// bind(addresses by name, raw_stream, row_exchange, row_watch, gemm_workspace, waits_check)
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *table, *rs, *re, *rw, *gw, *wc;
    if (!PyArg_ParseTuple(args, "O!OOOOO", &PyDict_Type, &table, &rs, &re, &rw, &gw, &wc)) return nullptr;
    const auto address = [&](const char* name, auto& fn) {
        PyObject* v = PyDict_GetItemString(table, name);
        if (v == nullptr) {
            PyErr_SetString(PyExc_KeyError, name);
            return false;
        }
        fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(PyLong_AsVoidPtr(v));
        return PyErr_Occurred() == nullptr;
    };
    if (!address("kr_reduce_bf16", reduce_bf16) || !address("kr_reduce_ptrs_bf16", reduce_ptrs_bf16) ||
        !address("kr_reduce_striped_bf16", reduce_striped_bf16) || !address("kr_reduce_striped_ptrs_bf16", reduce_striped_ptrs_bf16) ||
        !address("kr_striped_share_numel", striped_share_numel) || !address("kr_rmsnorm_workspace_bytes", rmsnorm_workspace_bytes) ||
        !address("kr_reduce_rmsnorm_ws_bf16", reduce_rmsnorm_ws_bf16) || !address("kr_reduce_rmsnorm_ptrs_ws_bf16", reduce_rmsnorm_ptrs_ws_bf16) ||
        !address("kr_rmsnorm_bf16", rmsnorm_bf16) || !address("kr_gemm_workspace_bytes", gemm_workspace_bytes) ||
        !address("kr_gemm_reduce_bf16", gemm_reduce_bf16) || !address("kr_gemm_reduce_ws_bf16", gemm_reduce_ws_bf16) ||
        !address("kr_gemm_f32_pairs", gemm_f32_pairs) || !address("kr_gemm_f32_workspace_bytes", gemm_f32_workspace_bytes) ||
        !address("kr_gemm_reduce_f32_ws", gemm_reduce_f32_ws) || !address("kr_split_pairs_fp32", split_pairs_fp32) ||
        !address("kr_gemm_pairs_workspace_bytes", gemm_pairs_workspace_bytes) || !address("kr_gemm_reduce_pairs_ws", gemm_reduce_pairs_ws) ||
        !address("kr_reduce_rotated_ptrs_bf16", reduce_rotated_ptrs_bf16) || !address("kr_gather_chunks", gather_chunks) ||
        !address("kr_gather_matmul_direct", gather_matmul_direct) || !address("kr_gather_matmul_bf16", gather_matmul_bf16) ||
        !address("kr_gemm_fp8_workspace_bytes", gemm_fp8_workspace_bytes) || !address("kr_gemm_fp8_ws", gemm_fp8_ws) ||
        !address("kr_gemm_fp8_wide_workspace_bytes", gemm_fp8_wide_workspace_bytes) || !address("kr_gemm_fp8_wide_ws", gemm_fp8_wide_ws))
        return nullptr;
    PyObject** slots[] = {&raw_stream, &row_exchange, &row_watch, &gemm_workspace, &waits_check};
    PyObject* values[] = {rs, re, rw, gw, wc};
    for (int i = 0; i < 5; ++i) {
        PyObject* old = *slots[i];
        *slots[i] = Py_NewRef(values[i]);
        Py_XDECREF(old);
    }
    Py_RETURN_NONE;
}

#define KR_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {KR_FAST(all_reduce), KR_FAST(all_reduce_bias), KR_FAST(two_shot_share), KR_FAST(two_shot_bias),
                         KR_FAST(reduce_rms_norm), KR_FAST(rms_norm), KR_FAST(gemm), KR_FAST(reduce_scatter_sent), KR_FAST(gather_matmul), {"bind", bind, METH_VARARGS, nullptr}, {}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
    PyObject* m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", KR_TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
