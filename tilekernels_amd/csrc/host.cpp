// The call path of the public ops in native code: argument checks, output tensors and launch without the interpreter.
//
// What bounds a call on a few hundred tokens is the host: asserts, two to eight torch.empty and a ctypes call of some 15
// arguments in Python take 10 - 13 us, the kernel 2.5 - 5 us.  The functions here take the arguments of the op of the same
// name, all positional, and return its result, or None for everything out of the ordinary: arguments an assert would
// refuse, tensor subclasses, tensors off the current device, active torch modes and transforms, options few callers use.  The
// Python function then does the whole call itself, so that there is one place where calls are refused and its messages come from.
// The interpreter lock is released around allocation and launch, as torch.empty and ctypes do.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/GPUTrace.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <utility>

#include "../../include/tk_quant.h"

namespace {

struct General {};      // thrown: the Python function takes the call

void need(bool ordinary) {
    if (!ordinary) throw General{};
}

struct LaunchFailed {
    int status;
    const char *what;
};

// Status of a launch: refused arguments go to the Python function (which reports them), a HIP error is reported as it is.
void launched(int status, const char *what) {
    need(status >= 0);
    if (status > 0) throw LaunchFailed{status, what};
}

struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// Nothing that watches, records or transforms torch calls is active in this thread: such a thing must see the Python path's calls.
void need_plain_thread() {
    using c10::DispatchKey;
    static const c10::DispatchKeySet transforms{DispatchKey::Tracer, DispatchKey::FuncTorchDynamicLayerFrontMode,
                                                DispatchKey::FuncTorchDynamicLayerBackMode, DispatchKey::VmapMode, DispatchKey::Functionalize,
                                                DispatchKey::Python, DispatchKey::PythonDispatcher, DispatchKey::PreDispatch};
    need(!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_local_dispatch_key_set().included_.has_any(transforms));
}

const at::Tensor &tensor(PyObject *o) {
    using c10::DispatchKey;
    static const c10::DispatchKeySet wrapped{DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                             DispatchKey::Functionalize, DispatchKey::Batched, DispatchKey::Conjugate, DispatchKey::Negative,
                                             DispatchKey::ZeroTensor};
    need(THPVariable_CheckExact(o));
    const at::Tensor &t = THPVariable_Unpack(o);
    need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && t.unsafeGetTensorImpl()->has_storage());
    return t;
}

const at::Tensor *optional_tensor(PyObject *o) { return o == Py_None ? nullptr : &tensor(o); }

int64_t integer(PyObject *o) {
    need(PyLong_CheckExact(o));
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    need(overflow == 0);
    return v;
}

int small(PyObject *o) {
    const int64_t v = integer(o);
    need(v >= 0 && v <= INT32_MAX);
    return (int)v;
}

bool boolean(PyObject *o) {
    need(o == Py_True || o == Py_False);
    return o == Py_True;
}

struct Optional {
    bool given;
    float value;
};
Optional optional_float(PyObject *o) {
    if (o == Py_None) return {false, 0.0f};
    need(PyFloat_CheckExact(o));
    return {true, (float)PyFloat_AS_DOUBLE(o)};
}

bool text(PyObject *o, const char *s) { return PyUnicode_CheckExact(o) && PyUnicode_CompareWithASCIIString(o, s) == 0; }

std::pair<PyObject *, PyObject *> two(PyObject *o) {
    need(PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == 2);
    return {PyTuple_GET_ITEM(o, 0), PyTuple_GET_ITEM(o, 1)};
}

void need_device(const at::Tensor &first) { need(first.get_device() == c10::hip::current_device()); }
void need_same_device(const at::Tensor &first, const at::Tensor *other) { need(!other || other->get_device() == first.get_device()); }

bool is_matrix(const at::Tensor &t) { return t.dim() == 2 && t.size(0) > 0 && t.size(1) > 0; }
bool is_list(const at::Tensor &t, int64_t n) { return t.dim() == 1 && t.size(0) == n && t.scalar_type() == at::kInt && t.is_contiguous(); }

int plain_dtype(const at::Tensor &t) {
    need(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
    return t.scalar_type() == at::kBFloat16 ? TK_BF16 : TK_F32;
}

int code_format(PyObject *fmt) {
    if (text(fmt, "e4m3")) return TK_E4M3;
    if (text(fmt, "e2m1")) return TK_E2M1;
    need(text(fmt, "e5m6"));
    return TK_E5M6;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t align(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

void *stream() { return static_cast<void *>(c10::hip::getCurrentHIPStream().stream()); }

// torch.empty on the device of `like`, without the dispatcher (0.70 -> 0.35 us, and up to eight of them in a call), which need_plain_thread()
// and tensor() have found nothing to do for.  Where torch is told to fill what it leaves uninitialised, it does so.
at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor &like) {
    const at::Context &context = at::globalContext();
    if (context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory())
        return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
    return at::detail::empty_cuda(sizes, type, like.device(), c10::nullopt);
}

// The first rows x cols elements of a matrix of `ld` x cols that is stored column after column.
at::Tensor empty_columns(int64_t rows, int64_t cols, int64_t ld, at::ScalarType type, const at::Tensor &like) {
    at::Tensor t = empty({cols, ld}, type, like);
    const int64_t sizes[] = {rows, cols}, strides[] = {1, ld};
    t.unsafeGetTensorImpl()->set_sizes_and_strides(c10::IntArrayRef(sizes), c10::IntArrayRef(strides));
    return t;
}

at::Tensor empty_codes(int64_t rows, int64_t cols, int fmt, const at::Tensor &like) {
    if (fmt == TK_E5M6) return empty({rows, cols / 8 * 12}, at::kByte, like);
    return fmt == TK_E4M3 ? empty({rows, cols}, at::kFloat8_e4m3fn, like) : empty({rows, cols / 2}, at::kChar, like);
}

// Scale tensor of the layout the options name: `out` is what the caller gets, `ld` what the kernels are told.
struct Scales {
    int layout;
    int64_t ld;
    at::Tensor out;

    static int layout_of(bool col_major, bool round_sf, bool packed) {
        need(!packed || (col_major && round_sf));
        return packed ? TK_SF_COL_UE8M0 : (col_major ? TK_SF_COL_F32 : TK_SF_ROW_F32);
    }
    Scales(int layout_, int64_t nm, int64_t nk, const at::Tensor &like) : layout(layout_), ld(nk) {
        if (layout == TK_SF_ROW_F32) {
            out = empty({nm, nk}, at::kFloat, like);
            return;
        }
        // columns are stored one after the other, padded to 16 bytes: four fp32 scales, or four words of four exponent bytes
        const bool packed = layout == TK_SF_COL_UE8M0;
        const int64_t cols = packed ? ceil_div(nk, 4) : nk, rows = align(nm, 4);
        out = empty_columns(nm, cols, rows, packed ? at::kInt : at::kFloat, like);
        ld = packed ? rows * 4 : rows;
    }
};

// Layout and leading dimension of the scales of a quantised input, told apart as _input_sf_storage does.
struct InputScales {
    const void *data;
    int layout;
    int64_t ld;
    explicit InputScales(const at::Tensor &sf) : data(sf.const_data_ptr()) {
        need(is_matrix(sf));
        const bool col_major = sf.stride(0) == 1;
        const int64_t unit = sf.scalar_type() == at::kInt ? 4 : 1;
        need(sf.scalar_type() == at::kFloat || (sf.scalar_type() == at::kInt && col_major));
        need(col_major || sf.stride(1) == 1);
        layout = !col_major ? TK_SF_ROW_F32 : (unit == 4 ? TK_SF_COL_UE8M0 : TK_SF_COL_F32);
        const int rows = col_major ? 1 : 0;                 // dimension along which the storage rows follow each other
        ld = sf.stride(rows) * unit;
        if (sf.size(rows) == 1) ld = std::max(ld, sf.size(1 - rows) * unit);     // a single row's stride is arbitrary
    }
};

PyObject *wrap(const at::Tensor &t) { return THPVariable_Wrap(t); }

// Steals the references.
template <typename... T> PyObject *tuple(T... items) {
    PyObject *all[] = {items...}, *t = nullptr;
    bool ok = true;
    for (PyObject *o : all) ok = ok && o;
    if (ok) t = PyTuple_New(sizeof...(items));
    for (size_t i = 0; i < sizeof...(items); ++i) {
        if (t) PyTuple_SET_ITEM(t, (Py_ssize_t)i, all[i]);
        else Py_XDECREF(all[i]);
    }
    return t;
}

// (x or (data, sf), fmt, num_per_channels, x_block_size, col_major, round_sf, packed)
PyObject *per_token_cast(PyObject *const *a) {
    const int fmt = code_format(a[1]), group = small(a[2]);
    const bool round_sf = boolean(a[5]);
    const int layout = Scales::layout_of(boolean(a[4]), round_sf, boolean(a[6]));
    const bool tiled = group == 16 || group == 32 || group == 64 || group == 128;
    if (a[3] != Py_None) {
        const auto [data_o, sf_o] = two(a[0]);
        const auto [bm, bk] = two(a[3]);
        const int block_m = small(bm), block_k = small(bk);
        const at::Tensor &data = tensor(data_o), &in_sf = tensor(sf_o);
        need(tiled && fmt != TK_E5M6 && is_matrix(data) && data.stride(1) == 1);
        need_device(data);
        need_same_device(data, &in_sf);
        const bool fp4 = data.scalar_type() != at::kFloat8_e4m3fn;
        need(!fp4 || data.scalar_type() == at::kChar || data.scalar_type() == at::kByte);
        const int64_t M = data.size(0), K = data.size(1) * (fp4 ? 2 : 1), ld = M > 1 ? data.stride(0) * (fp4 ? 2 : 1) : K;
        const InputScales in(in_sf);
        at::Tensor out;
        Scales sf = [&] {
            WithoutGil no_gil;
            out = empty_codes(M, K, fmt, data);
            Scales s(layout, M, ceil_div(K, group), data);
            launched(tk_per_token_cast_quantized(data.const_data_ptr(), fp4 ? TK_E2M1 : TK_E4M3, M, K, ld, in.data, in.ld, in.layout, block_m,
                                                 block_k, out.mutable_data_ptr(), s.out.mutable_data_ptr(), s.ld, fmt, group, layout, round_sf,
                                                 stream()),
                     "tk_per_token_cast_quantized");
            return s;
        }();
        return tuple(wrap(out), wrap(sf.out));
    }
    const at::Tensor &x = tensor(a[0]);
    const int dtype = plain_dtype(x);
    need(is_matrix(x) && x.stride(1) == 1);
    need_device(x);
    const int64_t M = x.size(0), K = x.size(1), ld = M > 1 ? x.stride(0) : K;
    need(fmt == TK_E5M6 ? group == K && K % 8 == 0 : tiled || (group == K && K % 64 == 0));
    at::Tensor out;
    Scales sf = [&] {
        WithoutGil no_gil;
        out = empty_codes(M, K, fmt, x);
        Scales s(layout, M, ceil_div(K, group), x);
        launched(tk_per_token_cast(x.const_data_ptr(), dtype, M, K, ld, out.mutable_data_ptr(), s.out.mutable_data_ptr(), s.ld, fmt, group, layout,
                                   round_sf, TK_CAST_AND_SF, stream()),
                 "tk_per_token_cast");
        return s;
    }();
    return tuple(wrap(out), wrap(sf.out));
}

// (x, fmt, block_size, col_major, round_sf, packed)
PyObject *per_block_cast(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]);
    const int dtype = plain_dtype(x), fmt = code_format(a[1]);
    const auto [bm_o, bk_o] = two(a[2]);
    const int bm = small(bm_o), bk = small(bk_o);
    const bool round_sf = boolean(a[4]);
    const int layout = Scales::layout_of(boolean(a[3]), round_sf, boolean(a[5]));
    need(is_matrix(x) && x.is_contiguous() && x.size(1) % 64 == 0 && fmt != TK_E5M6);
    need((bm == 32 || bm == 128) && (bk == 32 || bk == 128));
    need_device(x);
    const int64_t M = x.size(0), K = x.size(1);
    at::Tensor out;
    Scales sf = [&] {
        WithoutGil no_gil;
        out = empty_codes(M, K, fmt, x);
        Scales s(layout, ceil_div(M, bm), ceil_div(K, bk), x);
        launched(tk_per_block_cast(x.const_data_ptr(), dtype, M, K, out.mutable_data_ptr(), s.out.mutable_data_ptr(), s.ld, fmt, bm, bk, layout,
                                   round_sf, TK_CAST_AND_SF, stream()),
                 "tk_per_block_cast");
        return s;
    }();
    return tuple(wrap(out), wrap(sf.out));
}

// ((data, sf), fmt, rows, columns, special_fmt)
PyObject *cast_back(PyObject *const *a) {
    const auto [data_o, sf_o] = two(a[0]);
    const at::Tensor &data = tensor(data_o), &in_sf = tensor(sf_o);
    const bool f32 = text(a[1], "fp32"), e5m6 = a[4] != Py_None;
    need(f32 || text(a[1], "bf16"));
    need(!e5m6 || text(a[4], "e5m6"));
    const int bm = small(a[2]), bk = small(a[3]);
    need(is_matrix(data) && data.is_contiguous());
    need_device(data);
    need_same_device(data, &in_sf);
    const at::ScalarType type = data.scalar_type();
    const bool fp4 = !e5m6 && type != at::kFloat8_e4m3fn;
    need(e5m6 ? type == at::kByte : !fp4 || type == at::kChar || type == at::kByte);
    const int64_t M = data.size(0), K = e5m6 ? data.size(1) * 2 / 3 : data.size(1) * (fp4 ? 2 : 1);
    need(K > 0 && K % (e5m6 ? 8 : 64) == 0);
    const InputScales in(in_sf);
    at::Tensor out;
    {
        WithoutGil no_gil;
        out = empty({M, K}, f32 ? at::kFloat : at::kBFloat16, data);
        launched(tk_cast_back(data.const_data_ptr(), e5m6 ? TK_E5M6 : (fp4 ? TK_E2M1 : TK_E4M3), M, K, in.data, in.ld, in.layout, bm, bk,
                              out.mutable_data_ptr(), f32 ? TK_F32 : TK_BF16, stream()),
                 "tk_cast_back");
    }
    return wrap(out);
}

// (x, fmt, num_per_channels, pos_to_token_topk, topk_weights, pos_to_expert, col_major, round_sf, packed, clamp, sf_clamp_min)
PyObject *swiglu_forward(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]);
    const at::Tensor *ptt = optional_tensor(a[3]), *weights = optional_tensor(a[4]), *experts = optional_tensor(a[5]);
    const int dtype = plain_dtype(x), group = small(a[2]);
    const bool round_sf = boolean(a[7]);
    const int layout = Scales::layout_of(boolean(a[6]), round_sf, boolean(a[8]));
    const Optional clamp = optional_float(a[9]), floor_ = optional_float(a[10]);
    need(text(a[1], "e4m3") && is_matrix(x) && x.is_contiguous() && x.size(1) % 256 == 0);
    const int64_t R = x.size(0), H = x.size(1) / 2;
    need(group == 128 || (group == H && layout == TK_SF_ROW_F32));
    if (ptt) need(is_list(*ptt, R) && weights && weights->dim() == 2 && weights->scalar_type() == at::kFloat && weights->is_contiguous());
    else need(!weights);
    if (experts) need(is_list(*experts, R));
    need_device(x);
    need_same_device(x, ptt);
    need_same_device(x, weights);
    need_same_device(x, experts);
    at::Tensor out;
    Scales sf = [&] {
        WithoutGil no_gil;
        out = empty_codes(R, H, TK_E4M3, x);
        Scales s(layout, R, ceil_div(H, group), x);
        launched(tk_swiglu_per_token_cast(x.const_data_ptr(), dtype, R, H, out.mutable_data_ptr(), s.out.mutable_data_ptr(), s.ld, group, layout,
                                          round_sf, floor_.given ? floor_.value : -1.0f, ptt ? ptt->const_data_ptr<int32_t>() : nullptr,
                                          weights ? weights->const_data_ptr<float>() : nullptr, weights ? weights->numel() : 0,
                                          experts ? experts->const_data_ptr<int32_t>() : nullptr, clamp.given, clamp.value, nullptr, 0, stream()),
                 "tk_swiglu_per_token_cast");
        return s;
    }();
    return tuple(wrap(out), wrap(sf.out));
}

// ((x, x_sf), grad_out, weight, pos_to_token_topk, token_topk_to_pos, num_per_channels, round_sf, clamp)
PyObject *swiglu_backward(PyObject *const *a) {
    const auto [x_o, sf_o] = two(a[0]);
    const at::Tensor &x = tensor(x_o), &x_sf = tensor(sf_o), &grad = tensor(a[1]), &weight = tensor(a[2]), &ptt = tensor(a[3]), &t2p = tensor(a[4]);
    const int group = small(a[5]);
    const bool round_sf = boolean(a[6]);
    const Optional clamp = optional_float(a[7]);
    need(group == 32 || group == 128);
    need(is_matrix(x) && x.scalar_type() == at::kFloat8_e4m3fn && x.is_contiguous() && x.size(1) % (2 * group) == 0);
    const int64_t R = x.size(0), H = x.size(1) / 2;
    need(x_sf.dim() == 2 && x_sf.size(0) == R && x_sf.size(1) == 2 * H / group && x_sf.scalar_type() == at::kFloat && x_sf.is_contiguous());
    need(grad.dim() == 2 && grad.size(0) == R && grad.size(1) == H && grad.scalar_type() == at::kBFloat16 && grad.is_contiguous());
    need(is_matrix(t2p) && t2p.scalar_type() == at::kInt && t2p.is_contiguous() && is_list(ptt, R));
    need(weight.dim() == 2 && weight.sizes() == t2p.sizes() && weight.scalar_type() == at::kFloat && weight.is_contiguous());
    need_device(x);
    for (const at::Tensor *t : {&x_sf, &grad, &weight, &ptt, &t2p}) need_same_device(x, t);
    at::Tensor out, codes, codes_sf, x_grad, weight_grad;
    {
        WithoutGil no_gil;
        out = empty({R, H}, at::kBFloat16, x);
        codes = empty({R, 2 * H}, at::kFloat8_e4m3fn, x);
        codes_sf = empty({R, 2 * H / group}, at::kFloat, x);
        x_grad = empty({R, 2 * H}, at::kBFloat16, x);
        weight_grad = empty(weight.sizes(), at::kFloat, x);
        launched(tk_swiglu_backward_per_token_cast(x.const_data_ptr(), x_sf.const_data_ptr<float>(), R, H, group, grad.const_data_ptr(),
                                                   weight.const_data_ptr<float>(), ptt.const_data_ptr<int32_t>(), t2p.const_data_ptr<int32_t>(),
                                                   weight.numel(), out.mutable_data_ptr(), codes.mutable_data_ptr(),
                                                   codes_sf.mutable_data_ptr<float>(), x_grad.mutable_data_ptr(), weight_grad.mutable_data_ptr<float>(),
                                                   round_sf, clamp.given, clamp.value, stream()),
                 "tk_swiglu_backward_per_token_cast");
    }
    return tuple(wrap(out), tuple(wrap(codes), wrap(codes_sf)), wrap(x_grad), wrap(weight_grad));
}

// The launch behind the per-channel casts, whose wrappers have checked the arguments:
// (x, x_sf, num_tokens, hidden, pos_to_token, num_tokens_out, num_per_tokens, round_sf, transpose, swiglu, clamp)
PyObject *per_channel_cast(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), *x_sf = optional_tensor(a[1]), *gather = optional_tensor(a[4]);
    const int64_t tokens = integer(a[2]), hidden = integer(a[3]), rows = integer(a[5]);
    const int group = small(a[6]);
    const bool round_sf = boolean(a[7]), transpose = boolean(a[8]), swiglu = boolean(a[9]);
    const Optional clamp = optional_float(a[10]);
    need(rows > 0 && hidden > 0 && group > 0);
    need_device(x);
    need_same_device(x, x_sf);
    need_same_device(x, gather);
    at::Tensor out, out_sf;
    {
        WithoutGil no_gil;
        out = transpose ? empty({hidden, rows}, at::kFloat8_e4m3fn, x) : empty({rows, hidden}, at::kFloat8_e4m3fn, x);
        out_sf = empty({ceil_div(rows, group), hidden}, at::kFloat, x);
        launched(tk_per_channel_cast(x.const_data_ptr(), x.scalar_type() == at::kFloat ? TK_F32 : TK_BF16,
                                     x_sf ? x_sf->const_data_ptr<float>() : nullptr, tokens, hidden,
                                     gather ? gather->const_data_ptr<int32_t>() : nullptr, rows, out.mutable_data_ptr(),
                                     out_sf.mutable_data_ptr<float>(), group, round_sf, transpose, swiglu, clamp.given, clamp.value, stream()),
                 "tk_per_channel_cast");
    }
    return tuple(wrap(out), wrap(out_sf));
}

// (topk_idx, num_experts, num_expanded_tokens, alignment, force_no_sync)
PyObject *get_fused_mapping(PyObject *const *a) {
    const at::Tensor &idx = tensor(a[0]);
    const int experts = small(a[1]), alignment = small(a[3]);
    int64_t expanded = integer(a[2]);
    const bool sync = expanded == 0 && !boolean(a[4]);
    // (the wait is the library's own: where torch is told to warn of waits, refuse or report them, Python's is the one it knows of)
    if (sync) need(c10::hip::warning_state().get_sync_debug_mode() == c10::hip::SyncDebugMode::L_DISABLED && !c10::impl::GPUTrace::get_trace());
    need(is_matrix(idx) && idx.is_contiguous() && idx.scalar_type() == at::kLong && experts > 0 && alignment > 0 && expanded >= 0);
    need(idx.size(0) <= INT32_MAX && idx.size(1) <= INT32_MAX);
    const int64_t tokens = idx.size(0), topk = idx.size(1);
    if (sync) expanded = (tokens * topk + (int64_t)(alignment - 1) * experts) / alignment * alignment;
    need_device(idx);
    at::Tensor pos_to_expert, pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end, counts, counts_host;
    {
        WithoutGil no_gil;
        pos_to_expert = empty({expanded}, at::kInt, idx);
        pos_to_token = empty({expanded}, at::kInt, idx);
        pos_to_token_topk = empty({expanded}, at::kInt, idx);
        token_topk_to_pos = empty({tokens, topk}, at::kInt, idx);
        expert_start = empty({experts}, at::kInt, idx);
        expert_end = empty({experts}, at::kInt, idx);
        counts = empty({experts}, at::kInt, idx);
        const int64_t words = std::max<int64_t>(tk_fused_mapping_workspace_bytes(tokens, (int)topk, experts), 4) / 4;
        const at::Tensor workspace = empty({words}, at::kInt, idx);
        const auto launch = [&](auto f, auto... more) {
            return f(idx.const_data_ptr<int64_t>(), tokens, (int)topk, experts, alignment, expanded, pos_to_expert.mutable_data_ptr<int32_t>(),
                     pos_to_token.mutable_data_ptr<int32_t>(), pos_to_token_topk.mutable_data_ptr<int32_t>(),
                     token_topk_to_pos.mutable_data_ptr<int32_t>(), expert_start.mutable_data_ptr<int32_t>(),
                     expert_end.mutable_data_ptr<int32_t>(), counts.mutable_data_ptr<int32_t>(), workspace.mutable_data_ptr(), words * 4, more...,
                     stream());
        };
        if (!sync) {
            launched(launch(tk_get_fused_mapping), "tk_get_fused_mapping");
        } else {
            counts_host = at::empty({experts}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
            launched(launch(tk_get_fused_mapping_with_counts, counts_host.mutable_data_ptr<int32_t>()), "tk_get_fused_mapping_with_counts");
            int64_t rows = 0;
            for (int e = 0; e < experts; ++e) rows += counts_host.const_data_ptr<int32_t>()[e];
            for (at::Tensor *t : {&pos_to_expert, &pos_to_token, &pos_to_token_topk}) t->unsafeGetTensorImpl()->set_sizes_contiguous({rows});
        }
    }
    PyObject *list = PyList_New(sync ? experts : 0);
    if (!list) return nullptr;
    if (sync)
        for (int e = 0; e < experts; ++e) PyList_SET_ITEM(list, e, PyLong_FromLong(counts_host.const_data_ptr<int32_t>()[e]));
    return tuple(wrap(pos_to_expert), wrap(pos_to_token), wrap(pos_to_token_topk), wrap(token_topk_to_pos), wrap(expert_start), wrap(expert_end),
                 wrap(counts), list);
}

// (x, x_sf or None, num_per_channels, token_topk_to_pos, pos_to_expert, col_major)
PyObject *expand_to_fused(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), *x_sf = optional_tensor(a[1]), &t2p = tensor(a[3]), &experts = tensor(a[4]);
    const bool col_major = boolean(a[5]);
    need(is_matrix(x) && x.is_contiguous() && is_matrix(t2p) && t2p.scalar_type() == at::kInt && t2p.is_contiguous() && t2p.size(0) == x.size(0));
    need(t2p.size(1) <= INT32_MAX && experts.dim() == 1 && is_list(experts, experts.size(0)) && experts.size(0) > 0);
    need_device(x);
    for (const at::Tensor *t : {x_sf, &t2p, &experts}) need_same_device(x, t);
    const int64_t tokens = x.size(0), hidden = x.size(1), rows = experts.size(0);
    int64_t sf_cols = 0;
    if (x_sf) {
        const int group = small(a[2]);
        const bool words = x_sf->scalar_type() == at::kInt;
        need((group == 32 || group == 128) && (words || x_sf->scalar_type() == at::kFloat) && (!words || col_major));
        sf_cols = ceil_div(hidden, group * (words ? 4 : 1));
        need(x_sf->dim() == 2 && x_sf->size(0) == tokens && x_sf->size(1) == sf_cols && x_sf->is_contiguous() && sf_cols <= INT32_MAX);
    }
    at::Tensor out, out_sf;
    {
        WithoutGil no_gil;
        out = empty({rows, hidden}, x.scalar_type(), x);
        int64_t ld = 0;
        if (x_sf) {
            ld = col_major ? align(rows, 4) : sf_cols;
            out_sf = col_major ? empty_columns(rows, sf_cols, ld, x_sf->scalar_type(), x)
                               : empty({rows, sf_cols}, x_sf->scalar_type(), x);
        }
        launched(tk_expand_to_fused(x.const_data_ptr(), tokens, hidden * x.element_size(), t2p.const_data_ptr<int32_t>(), (int)t2p.size(1),
                                    experts.const_data_ptr<int32_t>(), rows, out.mutable_data_ptr(), x_sf ? x_sf->const_data_ptr() : nullptr,
                                    (int)sf_cols, x_sf ? out_sf.mutable_data_ptr() : nullptr, ld, col_major, stream()),
                 "tk_expand_to_fused");
    }
    return x_sf ? tuple(wrap(out), wrap(out_sf)) : wrap(out);
}

// (x or (data, x_sf), topk_weights, token_topk_to_pos, fp8_format, sf)
PyObject *reduce_fused(PyObject *const *a) {
    PyObject *x_o = a[0], *x_sf_o = Py_None;
    if (PyTuple_CheckExact(x_o)) std::tie(x_o, x_sf_o) = two(x_o);
    const at::Tensor &x = tensor(x_o), *x_sf = optional_tensor(x_sf_o), *weights = optional_tensor(a[1]), &t2p = tensor(a[2]), *sf = optional_tensor(a[4]);
    const int dtype = plain_dtype(x);
    const bool fp8 = !text(a[3], "");
    need(!fp8 || text(a[3], "e4m3"));
    need(is_matrix(x) && x.size(1) % 256 == 0 && x.is_contiguous());
    need(is_matrix(t2p) && t2p.scalar_type() == at::kInt && t2p.is_contiguous() && t2p.size(1) <= INT32_MAX);
    if (x_sf) need(x_sf->dim() >= 1 && x_sf->size(0) == x.size(0) && x_sf->scalar_type() == at::kFloat && x_sf->is_contiguous());
    if (weights) need(weights->sizes() == t2p.sizes() && weights->scalar_type() == at::kFloat && weights->is_contiguous());
    if (sf) need(fp8 && sf->numel() >= 1 && sf->scalar_type() == at::kFloat);
    need_device(x);
    for (const at::Tensor *t : {x_sf, weights, &t2p, sf}) need_same_device(x, t);
    at::Tensor out;
    {
        WithoutGil no_gil;
        out = empty({t2p.size(0), x.size(1)}, fp8 ? at::kFloat8_e4m3fn : x.scalar_type(), x);
        launched(tk_reduce_fused(x.const_data_ptr(), dtype, x.size(0), x.size(1), x_sf ? x_sf->const_data_ptr<float>() : nullptr,
                                 weights ? weights->const_data_ptr<float>() : nullptr, t2p.const_data_ptr<int32_t>(), t2p.size(0), (int)t2p.size(1),
                                 out.mutable_data_ptr(), fp8 ? TK_OUT_E4M3 : dtype, sf ? sf->const_data_ptr<float>() : nullptr, stream()),
                 "tk_reduce_fused");
    }
    return wrap(out);
}

template <PyObject *(*OP)(PyObject *const *), int ARGS>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != ARGS) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    try {
        need_plain_thread();
        return OP(args);
    } catch (const General &) {
        Py_RETURN_NONE;
    } catch (const LaunchFailed &e) {
        PyObject *ffi = PyImport_ImportModule("tilekernels_amd._ffi");      // its check() raises
        PyObject *r = ffi ? PyObject_CallMethod(ffi, "check", "is", e.status, e.what) : nullptr;
        Py_XDECREF(ffi);
        return r;
    }
    END_HANDLE_TH_ERRORS
}

#define TK_HOST_OP(name, args) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, args>)), METH_FASTCALL, nullptr}
PyMethodDef kOps[] = {TK_HOST_OP(per_token_cast, 7),  TK_HOST_OP(per_block_cast, 6),    TK_HOST_OP(cast_back, 5),
                      TK_HOST_OP(swiglu_forward, 11), TK_HOST_OP(swiglu_backward, 8),   TK_HOST_OP(per_channel_cast, 11),
                      TK_HOST_OP(get_fused_mapping, 5), TK_HOST_OP(expand_to_fused, 6), TK_HOST_OP(reduce_fused, 5),
                      {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kOps, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&kModule); }
