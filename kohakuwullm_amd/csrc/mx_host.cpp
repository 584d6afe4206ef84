// The host side of the eager path: what a module does around its launches -- looking at operands, allocating results,
// filling in arguments -- as a CPython extension over libmxfp8_hip.so.
//
// Every function here stands for the plain case of a Python function of the same name in kernels/, which describes the
// operation and serves every other case.  A function returns None, before it has launched any of the library's kernels, for a call
// that is not plain: a tensor that is not a strided one on the current GPU, a shape or layout that is refused or laid out anew there, a
// call that is traced, transformed, intercepted by a mode or dispatched by a subclass, a timer or another library installed in
// the binding.  The caller then takes the Python way, where such a call raises, copies or dispatches as it always did.
//
// Why: a linear layer over 8 tokens took 28.8 us of which the GPU worked 12.8; a training step of one over 4096 tokens 171 of
// which 50.  ctypes converts 12 to 20 arguments per launch in 2 us, torch.empty parses its keywords in 1 to 2.
#include <Python.h>
#include <dlfcn.h>

#include <vector>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/headeronly/version.h>

#include "mxfp8_hip.h"

using at::ScalarType;
using at::Tensor;

namespace {

// ---- the library -----------------------------------------------------------------------------------------------------------

#define MX_ENTRIES(F)                                                                                                       \
    F(mx_quantize_rows) F(mx_quantize_tokens) F(mx_quantize_tokens_side) F(mx_join_codes) F(mx_quantize_dual_batch)         \
    F(mx_swiglu_quantize_tokens) F(mx_swiglu_bwd_quantize_tokens) F(mx_gemm_nt) F(mx_gemm_nt_batch) F(mx_activation_gemm_nt) F(mx_rmsnorm_quantize) \
    F(mx_rmsnorm_backward) F(mx_rmsnorm_weight_grad) F(mx_router_topk) F(mx_router_backward_workspace)                      \
    F(mx_router_topk_backward_onto) F(mx_expert_sort_workspace) F(mx_expert_sort_positions) F(mx_experts_gemm1)                  \
    F(mx_grouped_gemm_nt) F(mx_experts_combine_onto) F(mx_experts_gemm2_dgrad_parts) F(mx_experts_gate_grad) F(mx_quantize_cols_grouped) F(mx_grouped_wgrad_nt)

struct Library {
#define F(name) decltype(&::name) name = nullptr;
    MX_ENTRIES(F)
#undef F
} lib;

PyObject *binding = nullptr;         // the dict of kohakuwullm_amd._lib
PyObject *bound_cdll = nullptr;      // what its `_lib` holds while these pointers are the right ones
PyObject *bound_invoke = nullptr;    // its own `invoke`
PyObject *s_timer, *s_cdll, *s_invoke, *s_check, *s_workspace, *s_workspaces;

// Thrown where a call turns out not to be plain; nothing has been launched then.
struct Declined {};
#define MX_NEED(cond) \
    if (!(cond)) throw Declined()

bool engaged() {
    return binding && PyDict_GetItem(binding, s_timer) == Py_None && PyDict_GetItem(binding, s_cdll) == bound_cdll &&
           PyDict_GetItem(binding, s_invoke) == bound_invoke && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A status other than MX_OK raises what the binding raises for it.
void check(int status, const char *what) {
    if (status == MX_OK) return;
    PyObject *done = PyObject_CallFunction(PyDict_GetItem(binding, s_check), "is", status, what);
    Py_XDECREF(done);
    if (done) PyErr_SetString(PyExc_RuntimeError, what);
    throw python_error();
}
// Other Python threads run while a launch waits for a place in its queue, or an allocation or copy for memory, as they do under
// ctypes and in PyTorch's own operators.  Nothing in the guarded scope touches a Python object.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() noexcept(false) { PyEval_RestoreThread(state); }  // ends a daemon thread by unwinding it at interpreter exit
};
#define MX_CALL(name, ...) ([&] { Unlocked open; return lib.name(__VA_ARGS__); }())
#define MX_RUN(name, ...) check(MX_CALL(name, __VA_ARGS__), #name)
#define MX_COPY(expression) ([&]() -> Tensor { Unlocked open; return (expression); }())  // a PyTorch operator that may allocate and launch

// ---- tensors ---------------------------------------------------------------------------------------------------------------

constexpr ScalarType FP8 = at::kFloat8_e4m3fn, U8 = at::kByte, I32 = at::kInt;
constexpr int64_t BLOCK = 32, PANEL = 128, TILE_ROWS = 65535 * PANEL, ROW_CHUNKS = 0x7FFFFF00;

int code_of(ScalarType t) {
    switch (t) {
    case at::kBFloat16: return MX_BF16;
    case at::kHalf: return MX_FP16;
    case at::kFloat: return MX_FP32;
    default: throw Declined();
    }
}
bool half_type(ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }

bool plain(const Tensor &t) {
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
           !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize})) &&
           t.device().index() == c10::hip::current_device();
}

const uint8_t *bytes(const Tensor &t) { return (const uint8_t *)t.const_data_ptr(); }
bool aligned(const Tensor &t, uintptr_t a) { return (uintptr_t)t.const_data_ptr() % a == 0; }
void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef size, ScalarType type, const Tensor &like) {
    Unlocked open;
    return Tensor(at::detail::empty_cuda(size, type, like.device(), std::nullopt));
}

// rows x cols at `offset` elements into `whole`, rows `pitch` apart.
Tensor piece(const Tensor &whole, int64_t offset, int64_t rows, int64_t cols, int64_t pitch) {
    Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(whole.storage()), whole.key_set(), whole.dtype());
    if (!whole.is_inference()) t.unsafeGetTensorImpl()->set_version_counter(whole.unsafeGetTensorImpl()->version_counter());
    t.unsafeGetTensorImpl()->set_sizes_and_strides(at::IntArrayRef({rows, cols}), at::IntArrayRef({pitch, 1}), offset);
    return t;
}
// A matrix with `spare` elements behind each row, the last one included.
Tensor pitched(int64_t rows, int64_t cols, int64_t spare, ScalarType type, const Tensor &like) {
    return piece(empty({rows, cols + spare}, type, like), 0, rows, cols, cols + spare);
}

// (codes, scale bytes) of a matrix.
struct Quantized {
    Tensor q, s;
};

int64_t token_extent(int64_t tokens) {
    const int64_t panels = (tokens + PANEL - 1) / PANEL * PANEL, groups = (tokens + 4 * PANEL - 1) / (4 * PANEL) * 4 * PANEL;
    return 16 * (groups - panels) <= panels && groups <= TILE_ROWS ? groups : panels;
}

Tensor contiguous(const Tensor &t) { return t.is_contiguous() ? t : MX_COPY(t.contiguous()); }
// All dimensions but the last one as rows.
Tensor as_matrix(const Tensor &x) {
    if (x.dim() == 2) return x;
    return x.is_contiguous() ? x.view({-1, x.size(-1)}) : MX_COPY(x.reshape({-1, x.size(-1)}));
}

// A matrix the quantizers read as it lies: unit column stride, rows that start on 16 bytes.
Tensor aligned_rows(const Tensor &x) {
    const int64_t pitch = x.stride(0);
    if (x.stride(1) != 1 || pitch < x.size(1) || pitch * x.element_size() % 16 || !aligned(x, 16)) return MX_COPY(x.clone(at::MemoryFormat::Contiguous));
    return x;
}

Tensor activation_matrix(const Tensor &x, ScalarType compute) {
    MX_NEED(plain(x) && x.dim() >= 1 && x.numel() > 0 && half_type(compute));
    Tensor m = as_matrix(x);
    if (m.scalar_type() != compute && m.scalar_type() != at::kFloat) m = MX_COPY(m.to(compute));
    code_of(m.scalar_type());
    return aligned_rows(m);
}

std::vector<int64_t> with_last(const Tensor &x, int64_t last) {
    std::vector<int64_t> size = x.sizes().vec();
    size.back() = last;
    return size;
}

// ---- quantizers ------------------------------------------------------------------------------------------------------------

Quantized quantize_rows(const Tensor &x) {
    MX_NEED(plain(x) && x.dim() == 2 && x.size(1) % BLOCK == 0 && x.numel() > 0);
    const int64_t m = x.size(0), k = x.size(1);
    const int code = code_of(x.scalar_type());
    Quantized r{empty({m, k}, FP8, x), empty({m, k / BLOCK}, U8, x)};
    MX_RUN(mx_quantize_rows, x.const_data_ptr(), code, m, k, x.stride(0), x.stride(1), (uint8_t *)r.q.data_ptr(), k,
           (uint8_t *)r.s.data_ptr(), k / BLOCK, stream_of(x));
    return r;
}

struct Tokens {
    Quantized row, token;  // `token` undefined where it was not asked for
};

Quantized token_buffers(int64_t rows, int64_t cols, const Tensor &like) {
    const int64_t mt = token_extent(rows);
    return {empty({mt / PANEL, cols, PANEL}, FP8, like), empty({cols, mt / BLOCK}, U8, like)};
}
uint8_t *codes_out(const Quantized &t) { return t.q.defined() ? (uint8_t *)t.q.data_ptr() : nullptr; }
uint8_t *scales_out(const Quantized &t) { return t.s.defined() ? (uint8_t *)t.s.data_ptr() : nullptr; }
int64_t pitch_out(const Quantized &t) { return t.s.defined() ? t.s.size(1) : 0; }

// `x` as activation_matrix returns it.
Tokens quantize_tokens(const Tensor &x, ScalarType compute, int64_t cols, bool token_axis) {
    MX_NEED(plain(x) && x.dim() == 2 && x.numel() > 0 && half_type(compute));
    const int64_t m = x.size(0), kv = x.size(1), k = cols ? cols : kv;
    const int code = code_of(x.scalar_type());
    MX_NEED(x.stride(1) == 1 && m <= TILE_ROWS && m * k / 8 < ROW_CHUNKS && kv % 8 == 0 && k % BLOCK == 0);
    Tokens r;
    r.row = {empty({m, k}, FP8, x), empty({m, k / BLOCK}, U8, x)};
    if (token_axis || k != kv) r.token = token_buffers(m, k, x);
    MX_RUN(mx_quantize_tokens, x.const_data_ptr(), code, code_of(compute), m, kv, x.stride(0), token_extent(m), k,
           (uint8_t *)r.row.q.data_ptr(), k, (uint8_t *)r.row.s.data_ptr(), k / BLOCK, codes_out(r.token), scales_out(r.token),
           pitch_out(r.token), stream_of(x));
    return r;
}

// What _MXFP8Linear.forward makes of its input.
Tokens quantize_input(const Tensor &x2d, ScalarType compute, bool token_axis) {
    if (token_axis || x2d.scalar_type() != compute) return quantize_tokens(x2d, compute, 0, token_axis);
    Tokens r;
    r.row = quantize_rows(x2d);
    return r;
}

Tokens quantize_side(const std::vector<Tensor> &xs) {
    MX_NEED(!xs.empty() && xs.size() <= 8);
    const int64_t m = xs[0].size(0);
    mx_side_source src[8];
    int64_t k = 0;
    for (size_t i = 0; i < xs.size(); i++) {
        const Tensor &x = xs[i];
        MX_NEED(plain(x) && x.dim() == 2 && x.size(0) == m && x.numel() > 0 && half_type(x.scalar_type()) && x.scalar_type() == xs[0].scalar_type() &&
                x.stride(1) == 1 && x.size(1) % PANEL == 0);
        src[i] = {x.const_data_ptr(), x.size(1), x.stride(0)};
        k += x.size(1);
    }
    MX_NEED(m <= TILE_ROWS);
    Tokens r;
    r.row = {empty({m, k}, FP8, xs[0]), empty({m, k / BLOCK}, U8, xs[0])};
    r.token = token_buffers(m, k, xs[0]);
    MX_RUN(mx_quantize_tokens_side, src, (int)xs.size(), code_of(xs[0].scalar_type()), m, token_extent(m), (uint8_t *)r.row.q.data_ptr(), k,
           (uint8_t *)r.row.s.data_ptr(), k / BLOCK, codes_out(r.token), scales_out(r.token), pitch_out(r.token), stream_of(xs[0]));
    return r;
}

Quantized join_codes(const std::vector<Quantized> &parts) {
    MX_NEED(parts.size() > 1 && parts.size() <= 8);
    const Tensor &like = parts[0].q;
    MX_NEED(plain(like) && like.dim() == 2);
    const int64_t rows = like.size(0);
    mx_code_source src[8];
    int64_t k = 0;
    for (size_t i = 0; i < parts.size(); i++) {
        const Tensor &q = parts[i].q, &s = parts[i].s;
        MX_NEED(plain(q) && plain(s) && q.dim() == 2 && s.dim() == 2 && q.size(0) == rows && s.size(0) == rows && q.is_contiguous() &&
                s.is_contiguous() && aligned(q, 16) && aligned(s, 4) && q.size(1) % PANEL == 0 && s.size(1) * BLOCK == q.size(1));
        src[i] = {bytes(q), bytes(s), q.size(1), q.stride(0), s.stride(0)};
        k += q.size(1);
    }
    Quantized r{empty({rows, k}, FP8, like), empty({rows, k / BLOCK}, U8, like)};
    MX_RUN(mx_join_codes, src, (int)parts.size(), rows, (uint8_t *)r.q.data_ptr(), k, (uint8_t *)r.s.data_ptr(), k / BLOCK, stream_of(like));
    return r;
}

Tokens swiglu_tokens(const Tensor &gu, bool rounded, bool token_axis) {
    MX_NEED(plain(gu) && gu.dim() == 2 && gu.numel() > 0 && half_type(gu.scalar_type()) && gu.stride(1) == 1 && gu.size(1) % (2 * PANEL) == 0);
    const int64_t m = gu.size(0), h = gu.size(1) / 2;
    MX_NEED(m <= TILE_ROWS && m * h / 8 < ROW_CHUNKS);
    Tokens r;
    r.row = {empty({m, h}, FP8, gu), empty({m, h / BLOCK}, U8, gu)};
    if (token_axis) r.token = token_buffers(m, h, gu);
    MX_RUN(mx_swiglu_quantize_tokens, gu.const_data_ptr(), code_of(gu.scalar_type()), rounded, m, h, gu.stride(0), token_extent(m),
           (uint8_t *)r.row.q.data_ptr(), h, (uint8_t *)r.row.s.data_ptr(), h / BLOCK, codes_out(r.token), scales_out(r.token),
           pitch_out(r.token), stream_of(gu));
    return r;
}

Tokens swiglu_bwd_tokens(const Tensor &dh, const Tensor &gu, bool rounded) {
    MX_NEED(plain(gu) && plain(dh) && gu.dim() == 2 && dh.dim() == 2 && gu.numel() > 0 && half_type(gu.scalar_type()) &&
            dh.scalar_type() == gu.scalar_type() && gu.size(1) % (2 * PANEL) == 0 && dh.size(0) == gu.size(0) && 2 * dh.size(1) == gu.size(1));
    MX_NEED(dh.stride(1) == 1 && gu.stride(1) == 1 && gu.stride(0) >= gu.size(1) && gu.stride(0) % 8 == 0 && aligned(gu, 16));
    const int64_t m = gu.size(0), h = gu.size(1) / 2, mt = token_extent(m);
    MX_NEED(m <= TILE_ROWS);
    Tokens r;
    r.row = {empty({2 * h / PANEL, m, PANEL}, FP8, gu), empty({m, 2 * h / BLOCK}, U8, gu)};
    r.token = token_buffers(m, 2 * h, gu);
    MX_RUN(mx_swiglu_bwd_quantize_tokens, dh.const_data_ptr(), dh.stride(0), gu.const_data_ptr(), gu.stride(0), code_of(gu.scalar_type()), rounded, m,
           h, mt, (uint8_t *)r.row.q.data_ptr(), PANEL, (uint8_t *)r.row.s.data_ptr(), 2 * h / BLOCK, codes_out(r.token),
           scales_out(r.token), pitch_out(r.token), stream_of(gu));
    return r;
}

// ---- products --------------------------------------------------------------------------------------------------------------

// The binding's scratch tensor of (device, stream).  The binding keeps it, and alone: whoever empties its cache has the memory back.
Tensor workspace(const Tensor &like) {
    PyObject *kept = PyDict_GetItem(binding, s_workspaces);
    PyObject *key = Py_BuildValue("(iK)", (int)like.device().index(), (unsigned long long)(uintptr_t)stream_of(like));
    if (!key) throw python_error();
    PyObject *ws = kept && PyDict_Check(kept) ? PyDict_GetItem(kept, key) : nullptr;
    Py_DECREF(key);
    if (ws && THPVariable_Check(ws)) return THPVariable_Unpack(ws);
    PyObject *arg = THPVariable_Wrap(like);
    ws = PyObject_CallFunctionObjArgs(PyDict_GetItem(binding, s_workspace), arg, nullptr);
    Py_DECREF(arg);
    if (!ws) throw python_error();
    const Tensor t = THPVariable_Unpack(ws);
    Py_DECREF(ws);
    return t;
}

// Rows and contraction length of a code matrix, (rows, K) or stage-major (K / 128, rows, 128).
void code_shape(const Tensor &q, int64_t &rows, int64_t &k) {
    if (q.dim() == 3) {
        MX_NEED(q.size(2) == PANEL && q.is_contiguous() && aligned(q, 16));
        rows = q.size(1), k = q.size(0) * PANEL;
    } else {
        MX_NEED(q.dim() == 2 && q.stride(1) == 1);
        rows = q.size(0), k = q.size(1);
    }
}

// A quantized weight or saved operand, looked at before the first launch of a call whose products `describe` looks at later.
void check_operand(const Quantized &t) {
    MX_NEED(plain(t.q) && plain(t.s) && t.s.dim() == 2 && t.s.stride(1) == 1 && t.q.element_size() == 1 && t.s.element_size() == 1);
    int64_t rows, k;
    code_shape(t.q, rows, k);
    MX_NEED(rows > 0 && k > 0 && k % BLOCK == 0 && t.s.size(0) == rows && t.s.size(1) == k / BLOCK);
}

struct Product {
    Tensor aq, as, bq, bs;
};

mx_gemm_problem describe(const Product &p) {
    MX_NEED(plain(p.aq) && plain(p.as) && plain(p.bq) && plain(p.bs));
    int64_t m, n, k, kb;
    code_shape(p.aq, m, k);
    code_shape(p.bq, n, kb);
    MX_NEED(k == kb && k % BLOCK == 0 && m > 0 && n > 0 && k > 0);
    MX_NEED(p.as.dim() == 2 && p.bs.dim() == 2 && p.as.size(0) == m && p.bs.size(0) == n && p.as.size(1) == k / BLOCK && p.bs.size(1) == k / BLOCK &&
            p.as.stride(1) == 1 && p.bs.stride(1) == 1);
    MX_NEED(p.aq.element_size() == 1 && p.as.element_size() == 1 && p.bq.element_size() == 1 && p.bs.element_size() == 1);
    if (p.aq.dim() == 3 || p.bq.dim() == 3)  // the kernels that read panels take aligned rows alone
        for (const Tensor *t : {&p.aq, &p.bq})
            MX_NEED(t->dim() == 3 || (t->stride(0) >= t->size(1) && t->stride(0) % 16 == 0 && aligned(*t, 16)));
    return {bytes(p.aq), bytes(p.as), bytes(p.bq), bytes(p.bs), nullptr, m, n, k, p.aq.dim() == 3 ? PANEL : p.aq.stride(0), p.as.stride(0),
            p.bq.dim() == 3 ? PANEL : p.bq.stride(0), p.bs.stride(0), n};
}

// A @ B^T into `size` (whose product is M x N), or with `pad` spare elements behind every row of an M x N matrix.
Tensor matmul(const Product &p, ScalarType type, at::IntArrayRef size, int64_t pad) {
    const mx_gemm_problem d = describe(p);
    const int code = code_of(type);
    const Tensor ws = workspace(p.aq);
    Tensor out = pad ? pitched(d.M, d.N, pad, type, p.aq)
                     : empty(size.empty() ? at::IntArrayRef({d.M, d.N}) : size, type, p.aq);
    if (p.aq.dim() == 3 || p.bq.dim() == 3) {
        mx_gemm_problem one = d;
        one.c = out.data_ptr(), one.ldc = d.N + pad;
        MX_RUN(mx_gemm_nt_batch, &one, 1, code, ws.data_ptr(), ws.numel(), stream_of(p.aq));
    } else {
        MX_RUN(mx_gemm_nt, d.aq, d.a_scale, d.bq, d.b_scale, out.data_ptr(), code, d.M, d.N, d.K, d.lda, d.ldas, d.ldb, d.ldbs, d.N + pad, 0,
               ws.data_ptr(), ws.numel(), stream_of(p.aq));
    }
    return out;
}

std::vector<Tensor> matmul_batch(const std::vector<Product> &ps, ScalarType type, at::IntArrayRef first_size = {}) {
    MX_NEED(!ps.empty() && ps.size() <= 16);
    const int code = code_of(type);
    mx_gemm_problem d[16];
    for (size_t i = 0; i < ps.size(); i++) d[i] = describe(ps[i]);
    const Tensor ws = workspace(ps[0].aq);
    std::vector<Tensor> outs;
    for (size_t i = 0; i < ps.size(); i++) {
        outs.push_back(empty(i == 0 && !first_size.empty() ? first_size : at::IntArrayRef({d[i].M, d[i].N}), type, ps[0].aq));
        d[i].c = outs.back().data_ptr();
    }
    MX_RUN(mx_gemm_nt_batch, d, (int)ps.size(), code, ws.data_ptr(), ws.numel(), stream_of(ps[0].aq));
    return outs;
}

// The products of a few rows with several weights, the rows quantized on the way; false, with nothing launched, for more rows
// or another layout than that kernel takes, and for more than 64 columns per CU: every workgroup of 16 columns quantizes the rows
// again, which then costs what the launch saves (us in two launches / in one, 16 rows: 1536 -> 16384 9.8 / 9.5, 1536 -> 32768
// 15.8 / 16.9, 512 -> 131072 23.6 / 25.0, 1536 -> 131072 45.9 / 54.7).  `outs` are allocated here, x's shape with the weights' widths.
constexpr int64_t FEW_ROW_COLUMNS = 64 * 256;
bool activation_products(const Tensor &x, const Tensor &x2d, ScalarType compute, const std::vector<Quantized> &ws, std::vector<Tensor> &outs) {
    if (x2d.size(0) > 32 || ws.size() > 4) return false;
    int64_t columns = 0;
    for (const Quantized &w : ws) columns += w.q.defined() && w.q.dim() ? w.q.size(0) : 0;
    if (columns > FEW_ROW_COLUMNS) return false;
    mx_gemm_problem d[4];
    for (size_t j = 0; j < ws.size(); j++) {
        const Tensor &q = ws[j].q, &s = ws[j].s;
        MX_NEED(plain(q) && plain(s) && q.dim() == 2 && s.dim() == 2 && q.stride(1) == 1 && s.stride(1) == 1 && q.size(1) == x2d.size(1) &&
                s.size(0) == q.size(0) && s.size(1) * BLOCK == q.size(1) && q.element_size() == 1 && s.element_size() == 1 && q.size(0) > 0);
        outs.push_back(empty(with_last(x, q.size(0)), compute, x2d));
        d[j] = {nullptr, nullptr, bytes(q), bytes(s), outs.back().data_ptr(), x2d.size(0), q.size(0), q.size(1), 0, 0, q.stride(0), s.stride(0), q.size(0)};
    }
    const int status = MX_CALL(mx_activation_gemm_nt, x2d.const_data_ptr(), code_of(x2d.scalar_type()), x2d.stride(0), d, (int)ws.size(), code_of(compute), stream_of(x2d));
    if (status == MX_EUNSUPPORTED) {
        outs.clear();
        return false;
    }
    check(status, "mx_activation_gemm_nt");
    return true;
}

// ---- arguments and results -------------------------------------------------------------------------------------------------

struct Args {
    PyObject *const *v;
    Py_ssize_t n;
    Py_ssize_t i = 0;
    PyObject *next() {
        if (i >= n) throw std::invalid_argument("too few arguments");
        return v[i++];
    }
    static Tensor as_tensor(PyObject *o) {
        if (o == Py_None) return Tensor();
        MX_NEED(THPVariable_CheckExact(o));  // a tensor or a parameter; a subclass dispatches its operators itself
        return THPVariable_Unpack(o);
    }
    Tensor tensor() { return as_tensor(next()); }
    ScalarType dtype() {
        PyObject *o = next();
        MX_NEED(THPDtype_Check(o));
        return ((THPDtype *)o)->scalar_type;
    }
    int64_t integer() {
        const int64_t r = PyLong_AsLongLong(next());
        if (r == -1 && PyErr_Occurred()) throw python_error();
        return r;
    }
    double number() {
        const double r = PyFloat_AsDouble(next());
        if (r == -1.0 && PyErr_Occurred()) throw python_error();
        return r;
    }
    bool flag() { return PyObject_IsTrue(next()) == 1; }
    std::vector<Tensor> tensors() { return as_tensors(next()); }
    static std::vector<Tensor> as_tensors(PyObject *o) {
        MX_NEED(PyList_Check(o) || PyTuple_Check(o));
        std::vector<Tensor> r;
        for (Py_ssize_t j = 0; j < PySequence_Fast_GET_SIZE(o); j++) r.push_back(as_tensor(PySequence_Fast_GET_ITEM(o, j)));
        return r;
    }
    Quantized quantized() {
        const std::vector<Tensor> pair = tensors();
        MX_NEED(pair.size() == 2);
        return {pair[0], pair[1]};
    }
};

PyObject *wrap(const Tensor &t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
PyObject *wrap_all(const std::vector<Tensor> &ts, bool list = false) {
    PyObject *r = list ? PyList_New((Py_ssize_t)ts.size()) : PyTuple_New((Py_ssize_t)ts.size());
    if (!r) throw python_error();
    for (size_t j = 0; j < ts.size(); j++) {
        PyObject *o = wrap(ts[j]);
        if (!o) {
            Py_DECREF(r);
            throw python_error();
        }
        if (list) PyList_SET_ITEM(r, (Py_ssize_t)j, o);
        else PyTuple_SET_ITEM(r, (Py_ssize_t)j, o);
    }
    return r;
}

// A METH_FASTCALL entry around `F`: declined calls give None.
template <PyObject *(*F)(Args &)>
PyObject *entry(PyObject *, PyObject *const *v, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!engaged()) Py_RETURN_NONE;
    Args a{v, n};
    try {
        return F(a);
    } catch (const Declined &) {
        Py_RETURN_NONE;
    }
    END_HANDLE_TH_ERRORS
}

// ---- entries: quantizers and products --------------------------------------------------------------------------------------

PyObject *py_quantize_rows(Args &a) {
    const Quantized r = quantize_rows(a.tensor());
    return wrap_all({r.q, r.s});
}

PyObject *wrap_tokens(const Tokens &r) { return wrap_all({r.row.q, r.row.s, r.token.q, r.token.s}); }

PyObject *py_quantize_tokens(Args &a) {
    const Tensor x = a.tensor();
    const ScalarType compute = a.dtype();
    const int64_t cols = a.integer();
    return wrap_tokens(quantize_tokens(x, compute, cols, a.flag()));
}
PyObject *py_quantize_side(Args &a) { return wrap_tokens(quantize_side(a.tensors())); }
PyObject *py_join_codes(Args &a) {
    PyObject *o = a.next();
    MX_NEED(PyList_Check(o) || PyTuple_Check(o));
    std::vector<Quantized> parts;
    for (Py_ssize_t j = 0; j < PySequence_Fast_GET_SIZE(o); j++) {
        const std::vector<Tensor> pair = Args::as_tensors(PySequence_Fast_GET_ITEM(o, j));
        MX_NEED(pair.size() == 2);
        parts.push_back({pair[0], pair[1]});
    }
    const Quantized r = join_codes(parts);
    return wrap_all({r.q, r.s});
}
PyObject *py_swiglu_tokens(Args &a) {
    const Tensor gu = a.tensor();
    const bool rounded = a.flag();
    return wrap_tokens(swiglu_tokens(gu, rounded, a.flag()));
}
PyObject *py_swiglu_bwd_tokens(Args &a) {
    const Tensor dh = a.tensor(), gu = a.tensor();
    return wrap_tokens(swiglu_bwd_tokens(dh, gu, a.flag()));
}
PyObject *py_matmul(Args &a) {
    Product p;
    p.aq = a.tensor(), p.as = a.tensor(), p.bq = a.tensor(), p.bs = a.tensor();
    const ScalarType type = a.dtype();
    const int64_t pad = a.integer();
    MX_NEED(pad >= 0 && p.aq.defined() && p.bq.defined() && p.aq.dim() == 2 && p.bq.dim() == 2);
    return wrap(matmul(p, type, {}, pad));
}
PyObject *py_matmul_batch(Args &a) {
    PyObject *o = a.next();
    MX_NEED(PyList_Check(o) || PyTuple_Check(o));
    std::vector<Product> ps;
    for (Py_ssize_t j = 0; j < PySequence_Fast_GET_SIZE(o); j++) {
        const std::vector<Tensor> t = Args::as_tensors(PySequence_Fast_GET_ITEM(o, j));
        MX_NEED(t.size() == 4);
        ps.push_back({t[0], t[1], t[2], t[3]});
    }
    return wrap_all(matmul_batch(ps, a.dtype()), true);
}

// Row and column quantization of many matrices behind one launch per 24; views of two allocations.
PyObject *py_quantize_dual_batch(Args &a) {
    const std::vector<Tensor> xs = a.tensors();
    MX_NEED(!xs.empty());
    int64_t total = 0;
    for (const Tensor &x : xs) {
        MX_NEED(plain(x) && x.dim() == 2 && x.numel() > 0 && x.size(0) % BLOCK == 0 && x.size(1) % BLOCK == 0 && x.stride(1) == 1 &&
                x.device() == xs[0].device() && x.scalar_type() == xs[0].scalar_type());
        total += x.numel();
    }
    const int code = code_of(xs[0].scalar_type());
    const Tensor codes = empty({2 * total}, FP8, xs[0]), scales = empty({2 * total / BLOCK}, U8, xs[0]);
    std::vector<mx_quant_problem> problems;
    PyObject *out = PyList_New((Py_ssize_t)xs.size());
    if (!out) throw python_error();
    int64_t at = 0;
    for (size_t j = 0; j < xs.size(); j++) {
        const Tensor &x = xs[j];
        const int64_t m = x.size(0), k = x.size(1), n = m * k;
        const Tensor q = piece(codes, 2 * at, m, k, k), qt = piece(codes, 2 * at + n, k, m, m);
        const Tensor s = piece(scales, 2 * at / BLOCK, m, k / BLOCK, k / BLOCK), st = piece(scales, (2 * at + n) / BLOCK, k, m / BLOCK, m / BLOCK);
        problems.push_back({x.const_data_ptr(), (uint8_t *)q.data_ptr(), (uint8_t *)s.data_ptr(), (uint8_t *)qt.data_ptr(), (uint8_t *)st.data_ptr(),
                            m, k, x.stride(0), k, k / BLOCK, m, m / BLOCK});
        PyList_SET_ITEM(out, (Py_ssize_t)j, wrap_all({q, s, qt, st}));
        at += n;
    }
    const int status = MX_CALL(mx_quantize_dual_batch, problems.data(), (int)problems.size(), code, stream_of(xs[0]));
    if (status != MX_OK) Py_DECREF(out);
    check(status, "mx_quantize_dual_batch");
    return out;
}

// ---- entries: linear layers ------------------------------------------------------------------------------------------------

// (out, xtq, xts) of _MXFP8Linear.forward.
PyObject *py_linear_forward(Args &a) {
    const Tensor x = a.tensor();
    const ScalarType compute = a.dtype();
    const Quantized w{a.tensor(), a.tensor()};
    const bool token_axis = a.flag();
    check_operand(w);
    MX_NEED(w.q.dim() == 2 && x.defined() && x.dim() >= 1 && x.size(-1) == w.q.size(1));
    const Tensor x2d = activation_matrix(x, compute);
    std::vector<Tensor> few;
    if (!token_axis && activation_products(x, x2d, compute, {w}, few)) return wrap_all({few[0], Tensor(), Tensor()});
    const Tokens in = quantize_input(x2d, compute, token_axis);
    const Tensor out = matmul({in.row.q, in.row.s, w.q, w.s}, compute, with_last(x, w.q.size(0)), 0);
    return wrap_all({out, in.token.q, in.token.s});
}

// Whether nothing but the result of a call on these tensors can matter to anybody: no gradient is recorded and no tangent
// carried.  An autograd function's forward may then run without the function.
bool unrecorded(const Tensor &t) { return !at::GradMode::is_enabled() && plain(t) && !t._fw_grad(0).defined(); }

PyObject *py_unrecorded(Args &a) {
    while (a.i < a.n) {
        const Tensor t = a.tensor();
        if (t.defined() && !unrecorded(t)) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

// MXFP8Linear.forward where no gradient is recorded.
PyObject *py_linear_eval(Args &a) {
    const Tensor x = a.tensor(), weight = a.tensor();
    const Quantized w{a.tensor(), a.tensor()};
    check_operand(w);
    MX_NEED(x.defined() && unrecorded(x) && unrecorded(weight) && w.q.dim() == 2 && x.dim() >= 1 && x.size(-1) == w.q.size(1));
    const ScalarType compute = at::autocast::is_autocast_enabled(at::kCUDA) ? at::autocast::get_autocast_dtype(at::kCUDA) : x.scalar_type();
    const Tensor x2d = activation_matrix(x, compute);
    std::vector<Tensor> out;
    if (activation_products(x, x2d, compute, {w}, out)) return wrap(out[0]);
    const Tokens in = quantize_input(x2d, compute, false);
    return wrap(matmul({in.row.q, in.row.s, w.q, w.s}, compute, with_last(x, w.q.size(0)), 0));
}

// (dx, dw) of _MXFP8Linear.backward for a width that needs no padding.
PyObject *py_linear_backward(Args &a) {
    const Tensor dout = a.tensor();
    const ScalarType compute = a.dtype();
    const Quantized xt{a.tensor(), a.tensor()}, w{a.tensor(), a.tensor()};
    const bool need_dx = a.flag(), need_dw = a.flag();
    const ScalarType x_type = a.dtype(), dw_type = a.dtype();
    MX_NEED(plain(w.q) && w.q.dim() == 2 && dout.defined() && dout.dim() >= 1 && dout.size(-1) == w.q.size(1) && (need_dx || need_dw));
    code_of(x_type), code_of(dw_type);
    if (need_dw) MX_NEED(plain(xt.q) && xt.q.dim() == 3 && xt.q.size(0) * PANEL == token_extent(dout.numel() / dout.size(-1)));
    for (const Quantized *t : {&w, &xt}) {
        if (t == &xt && !need_dw) continue;
        check_operand(*t);
        // beside an operand in panels the kernels take aligned rows alone
        MX_NEED(t->q.dim() == 3 || (t->q.stride(0) >= t->q.size(1) && t->q.stride(0) % 16 == 0 && aligned(t->q, 16)));
    }
    const Tensor d2d = activation_matrix(dout, compute);
    const std::vector<int64_t> dx_size = with_last(dout, w.q.size(0));
    Tensor dx, dw;
    if (!need_dw) {
        const Quantized d = quantize_rows(d2d.scalar_type() == compute ? d2d : MX_COPY(d2d.to(compute)));
        return wrap_all({matmul({d.q, d.s, w.q, w.s}, x_type, dx_size, 0), dw});
    }
    const Tokens d = quantize_tokens(d2d, compute, 0, true);
    const Product wgrad{d.token.q, d.token.s, xt.q, xt.s}, dgrad{d.row.q, d.row.s, w.q, w.s};
    if (need_dx && x_type == dw_type) {
        const std::vector<Tensor> r = matmul_batch({dgrad, wgrad}, x_type, dx_size);
        return wrap_all(r);
    }
    dw = matmul(wgrad, dw_type, {}, 0);
    if (need_dx) dx = matmul(dgrad, x_type, dx_size, 0);
    return wrap_all({dx, dw});
}

// ([out, ...], xtq, xts) of _MXFP8LinearGroup.forward.
PyObject *py_group_forward(Args &a) {
    const Tensor x = a.tensor();
    const ScalarType compute = a.dtype();
    PyObject *caches = a.next();
    const bool token_axis = a.flag();
    MX_NEED(PyList_Check(caches) || PyTuple_Check(caches));
    std::vector<Quantized> ws;
    for (Py_ssize_t j = 0; j < PySequence_Fast_GET_SIZE(caches); j++) {
        const std::vector<Tensor> c = Args::as_tensors(PySequence_Fast_GET_ITEM(caches, j));
        MX_NEED(c.size() == 4);
        check_operand({c[0], c[1]});
        MX_NEED(c[0].dim() == 2 && c[0].is_contiguous() && c[1].is_contiguous() && x.defined() && x.dim() >= 1 && c[0].size(1) == x.size(-1));
        ws.push_back({c[0], c[1]});
    }
    MX_NEED(!ws.empty() && ws.size() <= 8);
    const Tensor x2d = activation_matrix(x, compute);
    std::vector<Tensor> outs;
    if (!token_axis && activation_products(x, x2d, compute, ws, outs)) {
        outs.resize(outs.size() + 2);  // no operand along the tokens
        return wrap_all(outs);
    }
    const Tokens in = quantize_tokens(x2d, compute, 0, token_axis);
    mx_gemm_problem d[8];
    for (size_t j = 0; j < ws.size(); j++) {
        d[j] = describe({in.row.q, in.row.s, ws[j].q, ws[j].s});
        outs.push_back(empty(with_last(x, d[j].N), compute, x2d));
        d[j].c = outs.back().data_ptr();
    }
    const Tensor scratch = workspace(x2d);
    MX_RUN(mx_gemm_nt_batch, d, (int)ws.size(), code_of(compute), scratch.data_ptr(), scratch.numel(), stream_of(x2d));
    outs.push_back(in.token.q);
    outs.push_back(in.token.s);
    return wrap_all(outs);
}

// (y, xtq, xts, gu, htq, hts) of _MXFP8SwiGLUMLP.forward with operands in whole panels.
PyObject *py_swiglu_mlp_forward(Args &a) {
    const Tensor x = a.tensor();
    const ScalarType compute = a.dtype();
    const Quantized in = a.quantized(), out = a.quantized();
    const bool rounded = a.flag(), wgrad_in = a.flag(), wgrad_out = a.flag();
    const int64_t pad = a.integer();
    for (const Quantized *w : {&in, &out}) {
        check_operand(*w);
        MX_NEED(w->q.dim() == 2 && w->q.is_contiguous() && w->s.is_contiguous());
    }
    MX_NEED(x.defined() && x.dim() >= 1 && x.size(-1) == in.q.size(1) && in.q.size(0) == 2 * out.q.size(1) && out.q.size(1) % PANEL == 0);
    const Tensor x2d = activation_matrix(x, compute);
    MX_NEED(x2d.size(0) * out.q.size(1) / 8 < ROW_CHUNKS);
    Tokens xs;
    Tensor gu;
    std::vector<Tensor> few;
    if (!wgrad_in && activation_products(x2d, x2d, compute, {in}, few)) {
        gu = few[0];
    } else {
        xs = quantize_tokens(x2d, compute, 0, wgrad_in);
        gu = matmul({xs.row.q, xs.row.s, in.q, in.s}, compute, {}, pad);
    }
    const Tokens hs = swiglu_tokens(gu, rounded, wgrad_out);
    const Tensor y = matmul({hs.row.q, hs.row.s, out.q, out.s}, compute, with_last(x, out.q.size(0)), 0);
    return wrap_all({y, xs.token.q, xs.token.s, gu, hs.token.q, hs.token.s});
}

// ---- entries: RMSNorm ------------------------------------------------------------------------------------------------------

bool norm_weight_ok(const Tensor &w, const Tensor &x) {
    return plain(w) && w.dim() == 1 && w.is_contiguous() && w.size(0) == x.size(-1) && (w.scalar_type() == x.scalar_type() || w.scalar_type() == at::kFloat);
}

// (out, x2d, rstd) of _RMSNorm.forward without an MXFP8 operand.
PyObject *py_rmsnorm_forward(Args &a) {
    const Tensor x = a.tensor(), w = a.tensor();
    const double eps = a.number();
    MX_NEED(plain(x) && x.dim() >= 1 && x.numel() > 0 && half_type(x.scalar_type()) && (!w.defined() || norm_weight_ok(w, x)));
    const Tensor x2d = contiguous(as_matrix(x));
    const int64_t m = x2d.size(0), k = x2d.size(1);
    const Tensor rstd = empty({m}, at::kFloat, x), out = empty(x.sizes(), x.scalar_type(), x);
    MX_RUN(mx_rmsnorm_quantize, x2d.const_data_ptr(), code_of(x.scalar_type()), m, k, k, w.defined() ? w.const_data_ptr() : nullptr,
           w.defined() ? code_of(w.scalar_type()) : 0, (float)eps, out.data_ptr(), k, (float *)rstd.data_ptr(), nullptr, 0, nullptr, 0, stream_of(x));
    return wrap_all({out, x2d, rstd});
}

// (dx, dw) of _RMSNorm.backward; `most` partial rows of the weight's gradient at most.
PyObject *py_rmsnorm_backward(Args &a) {
    const Tensor dout = a.tensor(), x2d = a.tensor(), w = a.tensor(), rstd = a.tensor();
    const bool need_dw = a.flag();
    const int64_t most = a.integer();
    MX_NEED(plain(dout) && plain(x2d) && plain(rstd) && x2d.dim() == 2 && x2d.numel() > 0 && x2d.is_contiguous() && rstd.is_contiguous() &&
            rstd.scalar_type() == at::kFloat && rstd.numel() == x2d.size(0) && dout.dim() >= 1 && dout.numel() == x2d.numel() &&
            dout.size(-1) == x2d.size(1) && dout.scalar_type() == x2d.scalar_type() && half_type(x2d.scalar_type()) && (!w.defined() || norm_weight_ok(w, x2d)));
    const Tensor d2d = contiguous(as_matrix(dout));
    const int64_t m = x2d.size(0), k = x2d.size(1), parts = std::max<int64_t>(1, std::min((m + 3) / 4, most));
    const bool has_w = w.defined() && need_dw;
    const Tensor dx = empty(dout.sizes(), x2d.scalar_type(), x2d);
    Tensor part, dw;
    if (has_w) part = empty({parts, k}, at::kFloat, x2d), dw = empty({k}, w.scalar_type(), x2d);
    MX_RUN(mx_rmsnorm_backward, x2d.const_data_ptr(), code_of(x2d.scalar_type()), m, k, k, w.defined() ? w.const_data_ptr() : nullptr,
           w.defined() ? code_of(w.scalar_type()) : 0, d2d.const_data_ptr(), k, (const float *)rstd.const_data_ptr(), dx.data_ptr(), k,
           has_w ? (float *)part.data_ptr() : nullptr, parts, stream_of(x2d));
    if (has_w) MX_RUN(mx_rmsnorm_weight_grad, (const float *)part.const_data_ptr(), parts, k, dw.data_ptr(), code_of(w.scalar_type()), stream_of(x2d));
    return wrap_all({dx, dw});
}

// ---- entries: mixture of experts -------------------------------------------------------------------------------------------

// (idx, gate, scores, counts) of _RouteTopK.forward; operands as operands_fit accepts them, x as aligned_rows returns it.
PyObject *py_route_forward(Args &a) {
    const Tensor x = a.tensor(), w = a.tensor(), bias = a.tensor();
    const int64_t top_k = a.integer();
    const bool norm = a.flag();
    const double factor = a.number();
    const bool keep = a.flag();
    MX_NEED(plain(x) && plain(w) && x.dim() == 2 && w.dim() == 2 && w.is_contiguous() && x.stride(1) == 1 && x.size(1) == w.size(1) &&
            (!bias.defined() || (plain(bias) && bias.is_contiguous() && bias.dim() == 1 && bias.size(0) == w.size(0))));
    const int64_t t = x.size(0), e = w.size(0);
    const int xc = code_of(x.scalar_type()), wc = code_of(w.scalar_type()), bc = bias.defined() ? code_of(bias.scalar_type()) : 0;
    const Tensor idx = empty({t, top_k}, at::kLong, x), gate = empty({t, top_k}, x.scalar_type(), x), counts = empty({e}, I32, x);
    Tensor scores;
    if (keep) scores = empty({t, top_k}, at::kFloat, x);
    MX_RUN(mx_router_topk, x.const_data_ptr(), xc, x.stride(0), w.const_data_ptr(), wc, bias.defined() ? bias.const_data_ptr() : nullptr, bc, t,
           x.size(1), e, top_k, norm, (float)factor, (int64_t *)idx.data_ptr(), gate.data_ptr(), keep ? (float *)scores.data_ptr() : nullptr,
           (int32_t *)counts.data_ptr(), stream_of(x));
    return wrap_all({idx, gate, scores, counts});
}

// (dx, dw) of _RouteTopK.backward.
PyObject *py_route_backward(Args &a) {
    const Tensor grad = a.tensor(), x = a.tensor(), w = a.tensor(), idx = a.tensor(), scores = a.tensor();
    const bool norm = a.flag();
    const double factor = a.number();
    const bool need_dx = a.flag(), need_dw = a.flag();
    const Tensor onto = a.tensor();  // what dx is added to, or nothing
    if (onto.defined())
        MX_NEED(need_dx && plain(x) && plain(onto) && onto.dim() == 2 && onto.sizes() == x.sizes() && onto.scalar_type() == x.scalar_type() && onto.stride(1) == 1 &&
                onto.stride(0) >= onto.size(1) && onto.stride(0) * onto.element_size() % 16 == 0 && aligned(onto, 16));
    MX_NEED(plain(grad) && plain(x) && plain(w) && plain(idx) && plain(scores) && x.dim() == 2 && w.dim() == 2 && idx.dim() == 2 && x.numel() > 0 &&
            w.is_contiguous() && aligned(w, 16) && idx.is_contiguous() && scores.is_contiguous() && idx.scalar_type() == at::kLong &&
            scores.scalar_type() == at::kFloat && x.stride(1) == 1 && x.stride(0) >= x.size(1) && x.stride(0) * x.element_size() % 16 == 0 &&
            aligned(x, 16) && grad.numel() == idx.numel() && scores.numel() == idx.numel());
    const Tensor g = contiguous(grad);
    const int64_t t = x.size(0), d = x.size(1), e = w.size(0);
    const int gc = code_of(g.scalar_type()), xc = code_of(x.scalar_type()), wc = code_of(w.scalar_type());
    Tensor dx, dw, scratch;
    if (need_dx) dx = empty({t, d}, x.scalar_type(), x);
    int64_t words = 0;
    if (need_dw) {
        dw = empty(w.sizes(), w.scalar_type(), x);
        words = lib.mx_router_backward_workspace(t, d, e);
        MX_NEED(words >= 0);
        scratch = empty({words}, at::kFloat, x);
    }
    MX_RUN(mx_router_topk_backward_onto, onto.defined() ? onto.const_data_ptr() : nullptr, onto.defined() ? onto.stride(0) : 0, g.const_data_ptr(), gc, (const int64_t *)idx.const_data_ptr(), (const float *)scores.const_data_ptr(),
           x.const_data_ptr(), xc, x.stride(0), w.const_data_ptr(), wc, t, d, e, idx.size(1), norm, (float)factor,
           need_dx ? dx.data_ptr() : nullptr, d, need_dw ? dw.data_ptr() : nullptr, words ? (float *)scratch.data_ptr() : nullptr, words, stream_of(x));
    return wrap_all({dx, dw});
}

// (offsets, order, token_of, max_rows, positions) of expert_sort_positions.
PyObject *py_expert_sort(Args &a) {
    const Tensor flat = a.tensor(), counts = a.tensor();
    const int64_t top_k = a.integer(), experts = a.integer();
    const bool positions = a.flag();
    MX_NEED(plain(flat) && plain(counts) && flat.dim() == 1 && flat.is_contiguous() && (flat.scalar_type() == at::kLong || flat.scalar_type() == I32) &&
            counts.scalar_type() == I32 && counts.dim() == 1 && counts.size(0) == experts && counts.is_contiguous() && top_k > 0);
    const int64_t n = flat.numel(), need = lib.mx_expert_sort_workspace(n, experts);
    MX_NEED(need >= 0);
    const Tensor offsets = empty({experts + 1}, I32, flat), order = empty({n}, I32, flat), token_of = empty({n}, I32, flat), most = empty({1}, I32, flat);
    const Tensor scratch = empty({need}, I32, flat);
    Tensor inverse;
    if (positions) inverse = empty({n}, I32, flat);
    MX_RUN(mx_expert_sort_positions, flat.const_data_ptr(), (int)flat.element_size(), n, (const int32_t *)counts.const_data_ptr(), top_k, experts,
           (int32_t *)offsets.data_ptr(), (int32_t *)order.data_ptr(), (int32_t *)token_of.data_ptr(), (int32_t *)most.data_ptr(),
           positions ? (int32_t *)inverse.data_ptr() : nullptr, (int32_t *)scratch.data_ptr(), need, stream_of(flat));
    return wrap_all({offsets, order, token_of, most, inverse});
}

// The four quantized copies of an expert stack's two matrices: (E, N, K) codes and (E, N, K / 32) scales, any expert and row stride.
struct Stack {
    Quantized w;
    int64_t e, n, k;
};
Stack stack(const Quantized &w) {
    MX_NEED(plain(w.q) && plain(w.s) && w.q.dim() == 3 && w.s.dim() == 3 && w.q.stride(2) == 1 && w.s.stride(2) == 1 && w.q.element_size() == 1 &&
            w.s.size(0) == w.q.size(0) && w.s.size(1) == w.q.size(1) && w.s.size(2) * BLOCK == w.q.size(2));
    return {w, w.q.size(0), w.q.size(1), w.q.size(2)};
}
#define MX_STACK(of) bytes((of).w.q), bytes((of).w.s), (of).w.q.stride(0), (of).w.q.stride(1), (of).w.s.stride(0), (of).w.s.stride(1)

constexpr int64_t SCALE_ROW_SLACK = 16;
int64_t padded_rows(int64_t rows, int64_t experts) { return ((rows + PANEL - 1) / PANEL + experts) * PANEL; }
Quantized expert_token_buffers(int64_t cols, int64_t mpad, const Tensor &like) {
    return {empty({mpad / PANEL, cols, PANEL}, FP8, like), pitched(cols, mpad / BLOCK, SCALE_ROW_SLACK, U8, like)};
}

// How the rows are routed; all of them int32.
struct Routing {
    Tensor gate, token_of, order, offsets, positions;
    int64_t m, top_k;
    const int32_t *p(const Tensor &t) const { return (const int32_t *)t.const_data_ptr(); }
};

// y = a . w^T row by row, then out[t] = base[t], where given, + sum over t's pairs of gate * y.
Tensor routed_product(const Quantized &a, const Stack &w, const Routing &r, const Tensor &gate, int64_t tokens, ScalarType type, bool made, Tensor &positions,
                      const Tensor &base = Tensor()) {
    const Tensor y = empty({r.m, w.n}, type, a.q), out = empty({tokens, w.n}, type, a.q);
    const int code = code_of(type);
    MX_RUN(mx_grouped_gemm_nt, bytes(a.q), bytes(a.s), r.m, a.q.stride(0), a.s.stride(0), nullptr, MX_STACK(w), r.p(r.offsets), w.e, y.data_ptr(), code,
           w.n, r.m, w.n, w.k, stream_of(a.q));
    if (!made) positions = empty({tokens * r.top_k}, I32, a.q);
    MX_RUN(mx_experts_combine_onto, base.defined() ? base.const_data_ptr() : nullptr, base.defined() ? base.stride(0) : 0, y.const_data_ptr(), w.n, made ? nullptr : r.p(r.order), r.p(r.offsets), w.e,
           gate.defined() ? gate.const_data_ptr() : nullptr, gate.defined() ? code_of(gate.scalar_type()) : 0, (int32_t *)positions.data_ptr(), tokens,
           r.top_k, out.data_ptr(), code, w.n, r.m, w.n, stream_of(a.q));
    return out;
}

Routing routing(const Tensor &x, const Tensor &gate, const Tensor &token_of, const Tensor &order, const Tensor &offsets, const Tensor &positions, int64_t experts) {
    const int64_t tokens = x.size(0);
    MX_NEED(tokens > 0 && plain(gate) && gate.dim() == 1 && gate.is_contiguous() && gate.numel() % tokens == 0 && gate.numel() >= tokens);
    code_of(gate.scalar_type());
    for (const Tensor *t : {&token_of, &order, &offsets}) MX_NEED(plain(*t) && t->scalar_type() == I32 && t->dim() == 1 && t->is_contiguous());
    MX_NEED(offsets.numel() == experts + 1 && order.numel() == token_of.numel() && token_of.numel() > 0);
    const int64_t top_k = gate.numel() / tokens;
    if (positions.defined()) MX_NEED(plain(positions) && positions.scalar_type() == I32 && positions.is_contiguous() && positions.numel() == tokens * top_k);
    return {gate, token_of, order, offsets, positions, token_of.numel(), top_k};
}

// (out, hq, hs, pre, htq, hts, positions) of _MXFP8Experts.forward where `order` is the pair index.
PyObject *py_experts_forward(Args &a) {
    const Tensor x = a.tensor();
    const Tensor gate = a.tensor(), token_of = a.tensor(), order = a.tensor(), offsets = a.tensor(), positions = a.tensor();
    const Stack w_in = stack(a.quantized()), w_out = stack(a.quantized());
    const int64_t hidden = a.integer();
    const bool needs_grad = a.flag(), token_axis = a.flag();
    const Tensor base = a.tensor();
    MX_NEED(plain(x) && x.dim() == 2 && x.stride(1) == 1 && half_type(x.scalar_type()) && hidden % BLOCK == 0 && w_out.n % 8 == 0);
    if (base.defined())
        MX_NEED(plain(base) && base.sizes() == x.sizes() && base.scalar_type() == x.scalar_type() && base.stride(1) == 1 && base.stride(0) >= base.size(1) &&
                base.stride(0) % 8 == 0 && aligned(base, 16));
    const int64_t dim = x.size(1);
    MX_NEED(w_in.k == dim && w_in.n == 2 * hidden && w_out.n == dim && w_out.k == hidden && w_out.e == w_in.e && dim % BLOCK == 0);
    Routing r = routing(x, gate, token_of, order, offsets, positions, w_in.e);
    const ScalarType type = x.scalar_type();
    const Quantized xs = quantize_rows(x), h{empty({r.m, hidden}, FP8, x), empty({r.m, hidden / BLOCK}, U8, x)};
    Tensor pre;
    if (needs_grad) pre = empty({r.m, 2 * hidden}, type, x);
    Quantized ht;
    if (token_axis) ht = expert_token_buffers(hidden, padded_rows(r.m, w_in.e), x);
    MX_RUN(mx_experts_gemm1, bytes(xs.q), bytes(xs.s), x.size(0), dim, dim / BLOCK, r.p(token_of), MX_STACK(w_in), r.p(offsets), w_in.e,
           (uint8_t *)h.q.data_ptr(), hidden, (uint8_t *)h.s.data_ptr(), hidden / BLOCK, needs_grad ? pre.data_ptr() : nullptr, needs_grad ? 2 * hidden : 0,
           codes_out(ht), token_axis ? PANEL : 0, scales_out(ht), token_axis ? ht.s.stride(0) : 0, code_of(type), r.m, hidden, dim, stream_of(x));
    Tensor inverse = positions;
    const Tensor out = routed_product(h, w_out, r, gate, x.size(0), type, positions.defined(), inverse, base);
    return wrap_all({out, h.q, h.s, pre, ht.q, ht.s, inverse});
}

// (dx, dw_in, dw_out, dgate) of _MXFP8Experts.backward.
PyObject *py_experts_backward(Args &a) {
    const Tensor dout_any = a.tensor(), x = a.tensor(), hq = a.tensor(), hs = a.tensor(), pre = a.tensor();
    const Tensor gate = a.tensor(), token_of = a.tensor(), order = a.tensor(), offsets = a.tensor(), positions = a.tensor();
    const Tensor htq = a.tensor(), hts = a.tensor();
    const Stack w_in = stack(a.quantized()), w_out = stack(a.quantized());  // both as DGRAD contracts them
    const int64_t hidden = a.integer();
    const bool need_win = a.flag(), need_wout = a.flag();
    MX_NEED(plain(dout_any) && plain(x) && plain(hq) && plain(hs) && plain(pre) && x.dim() == 2 && x.stride(1) == 1 && half_type(x.scalar_type()) &&
            dout_any.scalar_type() == x.scalar_type() && dout_any.sizes() == x.sizes() && positions.defined());
    const int64_t dim = x.size(1);
    MX_NEED(w_in.n == dim && w_in.k == 2 * hidden && w_out.n == hidden && w_out.k == dim && w_out.e == w_in.e && dim % 8 == 0 && need_win);
    const Routing r = routing(x, gate, token_of, order, offsets, positions, w_in.e);
    const int64_t mpad = padded_rows(r.m, w_in.e);
    MX_NEED(hq.is_contiguous() && hs.is_contiguous() && pre.is_contiguous() && hq.numel() == r.m * hidden && hs.numel() == r.m * hidden / BLOCK &&
            pre.numel() == 2 * r.m * hidden && pre.scalar_type() == x.scalar_type() && aligned(hq, 16) && aligned(hs, 4) && aligned(pre, 16));
    auto token_operand = [&](const Tensor &q, const Tensor &s, int64_t cols) {
        MX_NEED(plain(q) && plain(s) && q.dim() == 3 && q.is_contiguous() && aligned(q, 16) && q.size(0) == mpad / PANEL && q.size(1) == cols &&
                q.size(2) == PANEL && s.dim() == 2 && s.stride(1) == 1 && s.size(0) == cols && s.size(1) == mpad / BLOCK &&
                s.stride(0) == s.size(1) + SCALE_ROW_SLACK && aligned(s, 4));
    };
    if (need_wout) token_operand(htq, hts, hidden);
    const Tensor dout = contiguous(dout_any);
    const ScalarType type = x.scalar_type();
    const int code = code_of(type);
    void *const st = stream_of(x);
    const Quantized d = quantize_rows(dout);
    const Quantized dp{empty({r.m, 2 * hidden}, FP8, x), empty({r.m, 2 * hidden / BLOCK}, U8, x)};
    const Tensor dgate = empty({gate.numel()}, gate.scalar_type(), x), parts = empty({(hidden + PANEL - 1) / PANEL, gate.numel()}, at::kFloat, x);
    const Quantized pt = expert_token_buffers(2 * hidden, mpad, x);
    MX_RUN(mx_experts_gemm2_dgrad_parts, bytes(d.q), bytes(d.s), x.size(0), dim, dim / BLOCK, r.p(token_of), r.p(order), gate.const_data_ptr(),
           code_of(gate.scalar_type()), MX_STACK(w_out), r.p(offsets), w_out.e, bytes(hq), hidden, bytes(hs), hidden / BLOCK, pre.const_data_ptr(), nullptr,
           2 * hidden, (uint8_t *)dp.q.data_ptr(), 2 * hidden, (uint8_t *)dp.s.data_ptr(), 2 * hidden / BLOCK, codes_out(pt), PANEL, scales_out(pt),
           pt.s.stride(0), (float *)parts.data_ptr(), gate.numel(), code, r.m, hidden, dim, st);
    MX_RUN(mx_experts_gate_grad, (const float *)parts.const_data_ptr(), gate.numel(), hidden, (const int32_t *)positions.const_data_ptr(), dgate.data_ptr(),
           code_of(gate.scalar_type()), gate.numel(), st);
    Tensor inverse = positions;
    const Tensor dx = routed_product(dp, w_in, r, Tensor(), x.size(0), type, true, inverse);
    const Tensor ws = workspace(x);
    auto columns = [&](const Tensor &rows, bool scaled) {
        const Quantized t = expert_token_buffers(dim, mpad, x);
        MX_RUN(mx_quantize_cols_grouped, rows.const_data_ptr(), code, rows.stride(0), dim, 0, r.p(token_of), scaled ? gate.const_data_ptr() : nullptr,
               scaled ? code_of(gate.scalar_type()) : 0, scaled ? r.p(order) : nullptr, r.p(offsets), w_in.e, r.m, codes_out(t), PANEL, scales_out(t),
               t.s.stride(0), st);
        return t;
    };
    auto wgrad = [&](const Tensor &aq, const Tensor &as, const Tensor &bq, const Tensor &bs) {
        const int64_t n = aq.size(1), k = bq.size(1);
        const Tensor dw = empty({w_in.e, n, k}, type, x);
        MX_RUN(mx_grouped_wgrad_nt, bytes(aq), bytes(as), PANEL, as.stride(0), bytes(bq), bytes(bs), PANEL, bs.stride(0), r.p(offsets), w_in.e, r.m,
               dw.data_ptr(), code, dw.stride(0), dw.stride(1), n, k, ws.data_ptr(), ws.numel(), st);
        return dw;
    };
    Tensor dw_in, dw_out;
    if (need_wout) {
        const Quantized dt = columns(dout, true);
        dw_out = wgrad(dt.q, dt.s, htq, hts);
    }
    const Quantized xt = columns(x, false);
    dw_in = wgrad(pt.q, pt.s, xt.q, xt.s);
    return wrap_all({dx, dw_in, dw_out, dgate});
}

// bind(path, cdll, invoke, module): take the entry points from the library at `path`, which `cdll` is; `module` is the ctypes binding,
// `invoke` its own call function.
PyObject *bind(PyObject *, PyObject *args) {
    const char *path;
    PyObject *cdll, *invoke, *module;
    if (!PyArg_ParseTuple(args, "sOOO", &path, &cdll, &invoke, &module)) return nullptr;
    void *so = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!so) return PyErr_Format(PyExc_RuntimeError, "%s: %s", path, dlerror());
    Library found;
#define F(name)                                                              \
    found.name = (decltype(found.name))dlsym(so, #name);                      \
    if (!found.name) return PyErr_Format(PyExc_RuntimeError, "%s: no %s", path, #name);
    MX_ENTRIES(F)
#undef F
    lib = found;
    PyObject *dict = PyModule_GetDict(module);
    Py_INCREF(dict), Py_INCREF(cdll), Py_INCREF(invoke);
    bound_cdll = cdll, bound_invoke = invoke, binding = dict;
    Py_RETURN_NONE;
}

// (token_extent(tokens), padded_rows(rows, experts)): sizes that the Python functions compute as well.
PyObject *py_extents(PyObject *, PyObject *args) {
    long long tokens, rows, experts;
    if (!PyArg_ParseTuple(args, "LLL", &tokens, &rows, &experts)) return nullptr;
    return Py_BuildValue("(LL)", (long long)token_extent(tokens), (long long)padded_rows(rows, experts));
}

// Whether plain calls are made here at present.
PyObject *py_engaged(PyObject *, PyObject *) { return PyBool_FromLong(engaged()); }

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))entry<py_##name>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr}, {"engaged", py_engaged, METH_NOARGS, nullptr}, {"extents", py_extents, METH_VARARGS, nullptr},
    ENTRY(quantize_rows), ENTRY(quantize_tokens), ENTRY(quantize_side), ENTRY(join_codes), ENTRY(quantize_dual_batch),
    ENTRY(swiglu_tokens), ENTRY(swiglu_bwd_tokens), ENTRY(matmul), ENTRY(matmul_batch),
    ENTRY(linear_forward), ENTRY(linear_backward), ENTRY(group_forward), ENTRY(swiglu_mlp_forward),
    ENTRY(rmsnorm_forward), ENTRY(rmsnorm_backward),
    ENTRY(route_forward), ENTRY(route_backward), ENTRY(expert_sort), ENTRY(experts_forward), ENTRY(experts_backward),
    ENTRY(unrecorded), ENTRY(linear_eval),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "The plain cases of the eager path, see mx_host.cpp.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    s_timer = PyUnicode_InternFromString("TIMER");
    s_cdll = PyUnicode_InternFromString("_lib");
    s_invoke = PyUnicode_InternFromString("invoke");
    s_check = PyUnicode_InternFromString("check");
    s_workspace = PyUnicode_InternFromString("gemm_workspace");
    s_workspaces = PyUnicode_InternFromString("_WORKSPACES");
    PyObject *module = PyModule_Create(&module_def);
    if (!module || PyModule_AddStringConstant(module, "torch_version", TORCH_VERSION) ||
        PyModule_AddObject(module, "constants", Py_BuildValue("{s:L,s:L,s:L,s:L,s:L}", "BLOCK_SCALE", (long long)BLOCK, "PANEL", (long long)PANEL, "TILE_ROWS",
                                                              (long long)TILE_ROWS, "ROW_CHUNKS", (long long)ROW_CHUNKS, "SCALE_ROW_SLACK", (long long)SCALE_ROW_SLACK)))
        return nullptr;
    return module;
}
