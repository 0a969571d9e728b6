// torch-library shim: registers the torch_butterfly operators and forwards them to the
// C ABI of libbutterfly_hip.so.  No kernels live here.
//
// Operator names, argument order and checks follow the reference shim
// (csrc/butterfly.cpp:20-131): twiddle first, then input, the stride flag and the
// optional output size.  The base-4 operators are new; their argument order follows
// butterfly_multiply_base4_torch (torch_butterfly/multiply_base4.py:7-8).
//
// Device tensors go to the HIP library and nowhere else.  Host tensors are accepted by the three
// operators the reference has (butterfly_multiply, _fw, _bw), in float, double, complex64 and
// complex128 as there (csrc/butterfly.cpp:44-52, 84-92), and run on the single-threaded host
// path of host_path.hpp; the operators that are new here take device tensors only.

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/core/grad_mode.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/library.h>

#include <tuple>

#include "../../include/butterfly_hip.h"
#include "host_path.hpp"

namespace {

using at::Tensor;

#define CHECK_DEVICE(x) \
    TORCH_CHECK(x.device().type() == at::kCPU || x.device().type() == at::kCUDA, #x " must be on CPU or CUDA")
#define CHECK_SAME_DEVICE(x, y) TORCH_CHECK(x.device() == y.device(), #x " and " #y " must be on the same device")
#define CHECK_DIM(x, y) TORCH_CHECK(x.dim() == y, #x " must have dimension " #y)
#define CHECK_SHAPE(x, ...) \
    TORCH_CHECK(x.sizes() == at::IntArrayRef({__VA_ARGS__}), #x " must have shape (" #__VA_ARGS__ ")")

int dtype_code(const Tensor &t, const char *who)
{
    if (t.scalar_type() == at::kFloat) return BF_F32;
    if (t.scalar_type() == at::kComplexFloat) return BF_C64;
    TORCH_CHECK(false, who, ": device kernels support float32 and complex64, got ", t.scalar_type());
    return -1;
}

void require_device(const Tensor &t, const char *who)
{
    TORCH_CHECK(t.is_cuda(), who, ": tensors must live on a HIP device; this operator has no CPU path");
}

// ---- host tensors ---------------------------------------------------------------------------

bf_host::Shape host_shape(int64_t batch, int64_t nstacks, int64_t log_n, int64_t nblocks, int64_t input_size,
                          int64_t output_size, bool increasing_stride)
{
    bf_host::Shape sh;
    sh.batch = batch;
    sh.nstacks = nstacks;
    sh.log_n = log_n;
    sh.nblocks = nblocks;
    sh.input_size = input_size;
    sh.output_size = output_size;
    sh.increasing_stride = increasing_stride;
    return sh;
}

void host_strides(int64_t dst[3], const Tensor &t)
{
    for (int i = 0; i < 3; ++i) dst[i] = t.stride(i);
}

// Calls f(T()) with T the host path's scalar type for the tensor's dtype.
template <typename F>
void host_dispatch(const Tensor &t, const char *who, F &&f)
{
    switch (t.scalar_type()) {
        case at::kFloat: f(float()); break;
        case at::kDouble: f(double()); break;
        case at::kComplexFloat: f(bf_host::Cplx<float>()); break;
        case at::kComplexDouble: f(bf_host::Cplx<double>()); break;
        default: TORCH_CHECK(false, who, " not implemented for '", t.scalar_type(), "'");
    }
}

Tensor host_multiply_fw(const Tensor &twiddle, const Tensor &input, bool increasing_stride, int64_t log_n,
                        int64_t output_size, const char *who)
{
    const Tensor tw = twiddle.resolve_conj().contiguous();
    const Tensor x = input.resolve_conj();
    const int64_t n = (int64_t)1 << log_n;
    Tensor output = at::empty({x.size(0), x.size(1), n}, x.options());
    if (output_size < n) output = output.slice(2, 0, output_size);
    const bf_host::Shape sh = host_shape(x.size(0), x.size(1), log_n, tw.size(1), x.size(2), output_size, increasing_stride);
    int64_t xs[3], os[3];
    host_strides(xs, x);
    host_strides(os, output);
    host_dispatch(x, who, [&](auto tag) {
        using T = decltype(tag);
        bf_host::multiply_fw<T>(sh, static_cast<const T *>(tw.data_ptr()), static_cast<const T *>(x.data_ptr()), xs,
                                static_cast<T *>(output.data_ptr()), os);
    });
    return output;
}

std::tuple<Tensor, Tensor> host_multiply_bw(const Tensor &twiddle, const Tensor &input, const Tensor &grad,
                                            bool increasing_stride, int64_t log_n, const char *who)
{
    const Tensor tw = twiddle.resolve_conj().contiguous();
    const Tensor x = input.resolve_conj();
    const Tensor g = grad.resolve_conj();
    const int64_t n = (int64_t)1 << log_n;
    const int64_t input_size = x.size(2);
    Tensor d_twiddle = at::empty(tw.sizes(), tw.options());
    Tensor d_input = at::empty({x.size(0), x.size(1), std::max(input_size, n)}, x.options());
    if (input_size < n) d_input = d_input.slice(2, 0, input_size);
    const bf_host::Shape sh = host_shape(x.size(0), x.size(1), log_n, tw.size(1), input_size, g.size(2), increasing_stride);
    int64_t xs[3], gs[3], ds[3];
    host_strides(xs, x);
    host_strides(gs, g);
    host_strides(ds, d_input);
    host_dispatch(x, who, [&](auto tag) {
        using T = decltype(tag);
        bf_host::multiply_bw<T>(sh, static_cast<const T *>(tw.data_ptr()), static_cast<const T *>(x.data_ptr()), xs,
                                static_cast<const T *>(g.data_ptr()), gs, static_cast<T *>(d_twiddle.data_ptr()),
                                static_cast<T *>(d_input.data_ptr()), ds);
    });
    return std::make_tuple(d_twiddle, d_input);
}

void set_strides(int64_t dst[3], const Tensor &t)
{
    for (int i = 0; i < 3; ++i) dst[i] = t.size(i) > 1 ? t.stride(i) : 0;
    for (int i = 0; i < 3; ++i) TORCH_CHECK(dst[i] >= 0, "negative strides are not supported");
}

// PyTorch on ROCm presents HIP devices under the "cuda" device type; these are the stream
// and guard types that go with that.
void *current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

void check_rc(int rc, const char *who) { TORCH_CHECK(rc == BF_OK, who, ": ", bf_last_error()); }

// Answer of one of the library's size queries: BF_SIZE_INVALID means the problem was refused.
size_t valid_size(size_t bytes)
{
    TORCH_CHECK(bytes != BF_SIZE_INVALID, "torch_butterfly: ", bf_last_error());
    return bytes;
}

// Dense copy of a (small) twiddle tensor; also materialises lazy conjugation.
// dense and 16-byte aligned (the kernels read factor blocks with 16-byte loads): a contiguous view
// at an odd offset into its storage is copied
Tensor dense(const Tensor &t)
{
    Tensor d = t.resolve_conj().contiguous();
    if (d.numel() > 0 && (reinterpret_cast<uintptr_t>(d.data_ptr()) & 15) != 0) d = d.clone();
    return d;
}

// A column table of the *_perm operators: int32, n entries, dense, on the device of `like`.
// Its entries are the caller's responsibility (each table a permutation of 0..n-1).
const int32_t *table_ptr(const Tensor &t, Tensor &keep, const Tensor &like, int64_t n, const char *name,
                         const char *who)
{
    if (!t.defined()) return nullptr;
    TORCH_CHECK(t.device() == like.device(), who, ": ", name, " must be on the device of input");
    TORCH_CHECK(t.scalar_type() == at::kInt, who, ": ", name, " must be int32");
    TORCH_CHECK(t.dim() == 1 && t.size(0) == n, who, ": ", name, " must have n entries");
    keep = t.contiguous();
    return keep.data_ptr<int32_t>();
}

// What one call works on, besides the rows.
struct Operands {
    Tensor twiddle, twiddle2;      // base 2: twiddle; base 4: twiddle4 and twiddle2
    Tensor bias;                   // undefined: none
    Tensor in_perm, out_index;     // undefined: none
    Tensor in_scale, out_scale;    // layers, base 2: diagonals folded into the factors; undefined: none
    bool base4 = false;
    bool increasing_stride = true;
    bool real_input = false;       // layers, complex64: the input is real / only the output's real part is wanted
    bool real_output = false;
};

void scale_factors(const Tensor &twiddle, const Operands &o, Tensor &scaled, const char *who);
void scale_factors_bw(const Tensor &twiddle, const Operands &o, const Tensor &grad, Tensor &d_twiddle, Tensor &d_in,
                      Tensor &d_out, const char *who);

// Shapes and strides of a call.  rows: a 3-d view (batch, nstacks, width) of the caller's input.
// layer: the stacks share one input (nstacks is then the factors') and out_size counts the columns
// over all stacks; otherwise it counts those of one stack.
struct Call {
    bf_layer desc = {};
    int64_t n = 0;
    Tensor twiddle, twiddle2, bias, tables[2];   // dense forms the descriptor points into

    bf_problem &p() { return desc.problem; }
};

void check_factors(const Operands &o, const Tensor &input, const char *who)
{
    const Tensor &twiddle = o.twiddle;
    CHECK_DEVICE(twiddle); CHECK_DEVICE(input); CHECK_SAME_DEVICE(twiddle, input);
    CHECK_DIM(twiddle, 6);
    if (!o.base4) return;
    const Tensor &twiddle2 = o.twiddle2;
    CHECK_DEVICE(twiddle2); CHECK_SAME_DEVICE(twiddle2, input);
    CHECK_DIM(twiddle2, 6);
    TORCH_CHECK(twiddle2.size(2) <= 1, "twiddle2 must have shape (nstacks, nblocks, log_n % 2, n / 2, 2, 2)");
}

int64_t log_size(const Operands &o, const char *who)
{
    const int64_t log_n = o.base4 ? o.twiddle.size(2) * 2 + o.twiddle2.size(2) : o.twiddle.size(2);
    TORCH_CHECK(log_n <= 30, who, ": n must be a power of 2");
    return log_n;
}

// Checks the factors against the rows and fills everything but the strides of output and d_input.
void describe(Call &c, const Operands &o, int64_t batch, int64_t nstacks, int64_t input_size, const int64_t (&stride)[3],
              const Tensor &input, int64_t out_cols, int64_t total, bool shared, const char *who)
{
    const int64_t log_n = log_size(o, who), n = (int64_t)1 << log_n, nblocks = o.twiddle.size(1);
    c.n = n;
    if (o.base4) {
        const Tensor &twiddle4 = o.twiddle, &twiddle2 = o.twiddle2;
        if (log_n / 2 > 0) CHECK_SHAPE(twiddle4, nstacks, nblocks, log_n / 2, n / 4, 4, 4);
        if (log_n % 2 == 1) CHECK_SHAPE(twiddle2, nstacks, nblocks, 1, n / 2, 2, 2);
        TORCH_CHECK(twiddle4.scalar_type() == input.scalar_type() && twiddle2.scalar_type() == input.scalar_type(), who,
                    ": twiddle4, twiddle2 and input must have the same dtype");
    } else {
        const Tensor &twiddle = o.twiddle;
        CHECK_SHAPE(twiddle, nstacks, nblocks, log_n, n / 2, 2, 2);
        if (o.real_input) {
            TORCH_CHECK(twiddle.scalar_type() == at::kComplexFloat && input.scalar_type() == at::kFloat, who,
                        ": a real input needs complex64 twiddle and float32 input");
        } else {
            TORCH_CHECK(twiddle.scalar_type() == input.scalar_type(), who, ": twiddle and input must have the same dtype");
        }
        TORCH_CHECK(!o.real_output || twiddle.is_complex(), who, ": a real output needs complex64 twiddle");
    }
    bf_problem &p = c.p();
    p.dtype = dtype_code(o.twiddle, who);
    p.increasing_stride = o.increasing_stride;
    p.batch = batch;
    p.nstacks = nstacks;
    p.log_n = log_n;
    p.nblocks = nblocks;
    p.input_size = input_size;
    p.output_size = out_cols;
    for (int i = 0; i < 3; ++i) {
        TORCH_CHECK(stride[i] >= 0, "negative strides are not supported");
        p.input_stride[i] = stride[i];
    }
    c.desc.base4 = o.base4;
    c.desc.shared_input = shared;
    c.desc.real_input = o.real_input;
    c.desc.real_output = o.real_output;
    c.desc.total_output = total;
    c.twiddle = dense(o.twiddle);
    c.desc.twiddle = c.twiddle.data_ptr();
    if (o.base4) {
        c.twiddle2 = dense(o.twiddle2);
        c.desc.twiddle2 = c.twiddle2.data_ptr();
    }
    if (o.bias.defined()) {
        const Tensor &bias = o.bias;
        CHECK_DEVICE(bias); CHECK_SAME_DEVICE(bias, input);
        TORCH_CHECK(bias.scalar_type() == o.twiddle.scalar_type(), who, ": bias and input must have the same dtype");
        c.bias = dense(bias);
        c.desc.bias = c.bias.data_ptr();
    }
    c.desc.in_perm = table_ptr(o.in_perm, c.tables[0], input, n, "in_perm", who);
    c.desc.out_index = table_ptr(o.out_index, c.tables[1], input, n, "out_index", who);
    if (c.desc.in_perm || c.desc.out_index) TORCH_CHECK(input_size <= n, who, ": column tables need input_size <= n");
}

// d_input as backward_call() will lay it out: the forward plans what to keep with the same strides.
// A multiply's is a slice of an n-wide tensor (what the reference returns), a layer's is dense.
void set_d_input_strides(Call &c, bool layer)
{
    bf_problem &p = c.p();
    const int64_t width = layer ? p.input_size : std::max(p.input_size, c.n);
    const int64_t stacks = layer && p.nstacks == 1 ? 1 : p.nstacks;
    p.d_input_stride[0] = stacks * width;
    p.d_input_stride[1] = width;
    p.d_input_stride[2] = 1;
}

Tensor bytes_like(const Tensor &t, size_t bytes)
{
    return at::empty({(int64_t)bytes}, t.options().dtype(at::kByte));
}

// keep (may be NULL): where the call may leave the intermediate activations that a backward in
// several passes would otherwise recompute; defined on return when it did.
void forward_call(Call &c, const Tensor &x, Tensor &output, Tensor *keep, const char *who)
{
    if (keep) {
        const size_t kept = valid_size(bf_layer_kept_bytes(&c.desc));
        if (kept > 0) {
            *keep = bytes_like(x, kept);
            check_rc(bf_layer_fw(&c.desc, x.data_ptr(), output.data_ptr(), keep->data_ptr(), kept, nullptr, 0,
                                 current_stream()),
                     who);
            return;
        }
    }
    const size_t ws_bytes = valid_size(bf_layer_fw_workspace_bytes(&c.desc));
    Tensor ws;
    if (ws_bytes > 0) ws = bytes_like(x, ws_bytes);
    check_rc(bf_layer_fw(&c.desc, x.data_ptr(), output.data_ptr(), nullptr, 0, ws_bytes > 0 ? ws.data_ptr() : nullptr,
                         ws_bytes, current_stream()),
             who);
}

struct Gradients {
    Tensor twiddle, twiddle2, input, bias, in_scale, out_scale;
};

void backward_call(Call &c, const Tensor &x, const Tensor &g, const Tensor &kept, bool with_bias, Gradients &d,
                   const char *who)
{
    const size_t kept_bytes = kept.defined() ? (size_t)kept.numel() : 0;
    d.twiddle = at::empty_like(c.twiddle);
    if (c.desc.base4) d.twiddle2 = at::empty_like(c.twiddle2);
    if (with_bias) d.bias = at::empty({c.desc.total_output}, c.twiddle.options());
    const size_t ws_bytes = valid_size(bf_layer_bw_workspace_bytes(&c.desc, with_bias ? 1 : 0, kept_bytes));
    Tensor ws;
    if (ws_bytes > 0) ws = bytes_like(x, ws_bytes);
    check_rc(bf_layer_bw(&c.desc, x.data_ptr(), g.data_ptr(), kept_bytes > 0 ? kept.data_ptr() : nullptr, kept_bytes,
                         d.twiddle.data_ptr(), c.desc.base4 ? d.twiddle2.data_ptr() : nullptr,
                         d.input.defined() ? d.input.data_ptr() : nullptr,
                         with_bias ? d.bias.data_ptr() : nullptr, ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes,
                         current_stream()),
             who);
}

// ---- the multiply operators: input (batch, nstacks, width) ---------------------------------------

// Strides of a 3-d operand, zero where there is nothing to step over.
void strides_of(int64_t (&dst)[3], const Tensor &t)
{
    for (int i = 0; i < 3; ++i) dst[i] = t.size(i) > 1 ? t.stride(i) : 0;
}

Tensor multiply_fw(const Operands &o, const Tensor &input, c10::optional<int64_t> output_size, Tensor *keep, const char *who)
{
    check_factors(o, input, who);
    CHECK_DIM(input, 3);
    const int64_t log_n = log_size(o, who), n = (int64_t)1 << log_n;
    const int64_t batch = input.size(0), nstacks = input.size(1);
    const int64_t cols = output_size.has_value() ? output_size.value() : n;
    TORCH_CHECK(cols <= n, who, ": output_size must be <= n");
    TORCH_CHECK(cols >= 0, who, ": output_size must be >= 0");
    if (!o.base4 && input.is_cpu() && !o.bias.defined() && !o.in_perm.defined() && !o.out_index.defined()) {
        const Tensor &twiddle = o.twiddle;
        CHECK_SHAPE(twiddle, nstacks, o.twiddle.size(1), log_n, n / 2, 2, 2);
        TORCH_CHECK(twiddle.scalar_type() == input.scalar_type(), who, ": twiddle and input must have the same dtype");
        return host_multiply_fw(twiddle, input, o.increasing_stride, log_n, cols, who);
    }
    require_device(input, who);
    if (o.bias.defined()) {
        const Tensor &bias = o.bias;
        CHECK_DIM(bias, 2);
        CHECK_SHAPE(bias, nstacks, cols);
    }
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    const Tensor x = input.resolve_conj();
    int64_t stride[3];
    strides_of(stride, x);
    Call c;
    describe(c, o, batch, nstacks, input.size(2), stride, x, cols, nstacks * cols, false, who);
    // (a slice of an n-wide tensor when there are fewer columns)
    Tensor output = cols == n ? at::empty({batch, nstacks, n}, x.options())
                              : at::empty({batch, nstacks, n}, x.options()).slice(2, 0, cols);
    strides_of(c.p().output_stride, output);
    set_d_input_strides(c, false);
    forward_call(c, x, output, keep, who);
    return output;
}

// kept: what the forward left in its `keep` (undefined: the backward recomputes what it needs)
Gradients multiply_bw(const Operands &o, const Tensor &input, const Tensor &grad, const Tensor &kept, bool with_bias,
                      const char *who)
{
    check_factors(o, input, who);
    CHECK_DEVICE(grad); CHECK_SAME_DEVICE(input, grad);
    CHECK_DIM(input, 3); CHECK_DIM(grad, 3);
    const int64_t log_n = log_size(o, who), n = (int64_t)1 << log_n;
    const int64_t batch = input.size(0), nstacks = input.size(1), input_size = input.size(2), cols = grad.size(2);
    CHECK_SHAPE(grad, batch, nstacks, cols);
    TORCH_CHECK(cols <= n, who, ": grad must have at most n columns");
    TORCH_CHECK(grad.scalar_type() == input.scalar_type(), who, ": grad and input must have the same dtype");
    Gradients d;
    if (!o.base4 && input.is_cpu() && !with_bias && !o.in_perm.defined() && !o.out_index.defined()) {
        const Tensor &twiddle = o.twiddle;
        CHECK_SHAPE(twiddle, nstacks, o.twiddle.size(1), log_n, n / 2, 2, 2);
        TORCH_CHECK(twiddle.scalar_type() == input.scalar_type(), who, ": twiddle and input must have the same dtype");
        std::tie(d.twiddle, d.input) = host_multiply_bw(twiddle, input, grad, o.increasing_stride, log_n, who);
        return d;
    }
    require_device(input, who);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    const Tensor x = input.resolve_conj(), g = grad.resolve_conj();
    int64_t stride[3];
    strides_of(stride, x);
    Call c;
    describe(c, o, batch, nstacks, input_size, stride, x, cols, nstacks * cols, false, who);
    strides_of(c.p().output_stride, g);
    set_d_input_strides(c, false);
    d.input = at::empty({batch, nstacks, std::max(input_size, n)}, x.options());
    if (input_size < n) d.input = d.input.slice(2, 0, input_size);
    backward_call(c, x, g, kept, with_bias, d, who);
    if (with_bias) d.bias = d.bias.view({nstacks, cols});
    return d;
}

// ---- whole layers: input (*, width), output (*, out_size) -----------------------------------------

// The rows of a layer's input as a 2-d view or copy.
Tensor rows_of(const Tensor &input)
{
    const Tensor x = input.resolve_conj();
    return x.dim() == 2 ? x : x.reshape({-1, x.size(-1)});
}

void describe_layer(Call &c, const Operands &o, const Tensor &x, int64_t out_size, const char *who)
{
    const int64_t nstacks = o.twiddle.size(0), n = (int64_t)1 << log_size(o, who);
    TORCH_CHECK(out_size > (nstacks - 1) * n && out_size <= nstacks * n, who, ": out_size must end in the last stack");
    if (o.bias.defined()) TORCH_CHECK(o.bias.dim() == 1 && o.bias.size(0) == out_size, who, ": bias must have out_size entries");
    const int64_t stride[3] = {x.size(0) > 1 ? x.stride(0) : 0, 0, x.size(1) > 1 ? x.stride(1) : 0};
    describe(c, o, x.size(0), nstacks, x.size(1), stride, x, nstacks == 1 ? out_size : n, out_size, true, who);
    set_d_input_strides(c, true);
}

// The rows of real numbers in a form the kernels take: as they are, or (schedules that only the
// fallback kernels run, a bias in front of a real output) as complex ones.
bool takes_real(Call &c, const Operands &o)
{
    return (!o.real_input && !o.real_output) || bf_layer_takes_real(&c.desc) != 0;
}
Tensor as_complex(const Tensor &t) { return t.to(at::kComplexFloat); }

Tensor layer_fw(const Operands &o_, const Tensor &input, int64_t out_size, Tensor *keep, Tensor *scaled, const char *who)
{
    Operands o = o_;
    check_factors(o, input, who);
    TORCH_CHECK(input.dim() >= 1, who, ": input must have at least one dimension");
    require_device(input, who);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    if (o.in_scale.defined() || o.out_scale.defined()) {
        Tensor with;
        scale_factors(o.twiddle, o, with, who);
        o.twiddle = with;
        if (scaled) *scaled = with;
    }
    Tensor x = rows_of(input);
    c10::SmallVector<int64_t, 6> shape(input.sizes().begin(), input.sizes().end());
    shape.back() = out_size;
    // Rows of several stacks start at multiples of 128 bytes: the stacks are written by different
    // workgroups, and in rows that start anywhere each of their ends would share its cache line with
    // another one's (7282 rows of 45 stacks of 64 complex64, 2821 columns: 77 us against 64).
    // Only where the last stack is cut short: whole stacks fill a contiguous tensor.
    const int64_t line = 128 / (o.real_output ? 4 : (int64_t)o.twiddle.element_size());
    const int64_t nstacks = o.twiddle.size(0);
    const bool cut = nstacks > 1 && out_size < (nstacks << log_size(o, who));
    const int64_t pitch = cut ? (out_size + line - 1) / line * line : out_size;
    auto run = [&](Tensor &output) {
        Call c;
        describe_layer(c, o, x, out_size, who);
        bf_problem &p = c.p();
        p.output_stride[0] = pitch;
        p.output_stride[1] = p.output_size;
        p.output_stride[2] = 1;
        if (!takes_real(c, o)) return false;
        const auto options = o.real_output ? x.options().dtype(at::kFloat) : o.twiddle.options();
        if (pitch == out_size) {
            output = at::empty(shape, options);
        } else {
            c10::SmallVector<int64_t, 6> stride(shape.size(), 1);
            for (int64_t d = (int64_t)shape.size() - 2, step = pitch; d >= 0; --d) {
                stride[d] = step;
                step *= std::max<int64_t>(shape[d], 1);
            }
            output = at::empty_strided(shape, stride, options);
        }
        forward_call(c, x, output, keep, who);
        return true;
    };
    Tensor output;
    if (run(output)) return output;
    const bool real_output = o.real_output;
    if (o.real_input) x = as_complex(x);
    o.real_input = o.real_output = false;
    run(output);
    return real_output ? at::real(output).contiguous() : output;
}

// with_input: whether the input's gradient is wanted.  Where it is not, the sum over the stacks is left
// out; the kernels of a single stack write it all the same.
Gradients layer_bw(const Operands &o_, const Tensor &input, const Tensor &grad, const Tensor &kept, const Tensor &scaled,
                   bool with_bias, bool with_input, const char *who)
{
    Operands o = o_;
    TORCH_CHECK(o.real_output ? grad.scalar_type() == at::kFloat : grad.scalar_type() == o.twiddle.scalar_type(), who,
                ": grad and output must have the same dtype");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    if (scaled.defined()) o.twiddle = scaled;
    Tensor x = rows_of(input), g = rows_of(grad);
    Gradients d;
    auto run = [&] {
        Call c;
        describe_layer(c, o, x, g.size(1), who);
        bf_problem &p = c.p();
        p.output_stride[0] = g.size(0) > 1 ? g.stride(0) : 0;
        p.output_stride[2] = g.size(1) > 1 ? g.stride(1) : 0;
        p.output_stride[1] = p.output_size * p.output_stride[2];
        if (!takes_real(c, o) || (with_bias && o.real_output)) return false;
        if (with_input || p.nstacks == 1) d.input = at::empty(input.sizes(), x.options());
        backward_call(c, x, g, kept, with_bias, d, who);
        return true;
    };
    if (!run()) {
        const bool real_input = o.real_input;
        if (o.real_input) x = as_complex(x);
        if (o.real_output) g = as_complex(g);
        o.real_input = o.real_output = false;
        run();
        if (real_input && d.input.defined()) d.input = at::real(d.input).contiguous();
    }
    if (scaled.defined()) {
        const Tensor d_scaled = d.twiddle;
        scale_factors_bw(o_.twiddle, o_, d_scaled, d.twiddle, d.in_scale, d.out_scale, who);
    }
    return d;
}

// ---- autograd ---------------------------------------------------------------------------------------
//
// One node for all differentiable operators.  Written against Node itself: the Function wrapper
// keeps its state in a dictionary of boxed values and prepares for several outputs and in-place
// ones, which costs more host time than a small multiply takes on the GPU.  Forward-mode
// derivatives and second derivatives do not exist, as in the reference's Function
// (csrc/butterfly.cpp:99-118).

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

struct MultiplyNode : public torch::autograd::Node {
    SavedVariable twiddle, twiddle2, input, kept, in_scale, out_scale, scaled, in_perm, out_index;
    bool base4 = false, increasing_stride = true, with_bias = false, layer = false, has_kept = false;
    bool real_input = false, real_output = false, has_scaled = false, has_in_perm = false, has_out_index = false;
    const char *who = nullptr;

    // edges: twiddle, twiddle2, input, bias, in_scale, out_scale (those that the call does not have lead nowhere)
    variable_list apply(variable_list &&grads) override
    {
        variable_list out(num_outputs());
        if (!grads[0].defined()) return out;
        // (against another thread's release_variables or pass over the same graph)
        std::lock_guard<std::mutex> lock(mutex_);
        const auto self = getptr();
        Operands o;
        o.twiddle = twiddle.unpack(self);
        if (base4) o.twiddle2 = twiddle2.unpack(self);
        if (has_in_perm) o.in_perm = in_perm.unpack(self);
        if (has_out_index) o.out_index = out_index.unpack(self);
        o.base4 = base4;
        o.increasing_stride = increasing_stride;
        o.real_input = real_input;
        o.real_output = real_output;
        const Tensor x = input.unpack(self), planes = has_kept ? kept.unpack(self) : Tensor();
        Tensor with;
        if (has_scaled) {
            o.in_scale = in_scale.unpack(self);
            o.out_scale = out_scale.unpack(self);
            with = scaled.unpack(self);
        }
        // (an input without gradient: every first layer; a frozen bias)
        const bool want_input = task_should_compute_output(2), want_bias = with_bias && task_should_compute_output(3);
        at::AutoDispatchBelowADInplaceOrView below;
        Gradients d = layer ? layer_bw(o, x, grads[0], planes, with, want_bias, want_input, who)
                            : multiply_bw(o, x, grads[0], planes, want_bias, who);
        out[0] = std::move(d.twiddle);
        out[1] = std::move(d.twiddle2);
        out[2] = std::move(d.input);
        out[3] = std::move(d.bias);
        out[4] = std::move(d.in_scale);
        out[5] = std::move(d.out_scale);
        return out;
    }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        twiddle.reset_data();
        twiddle2.reset_data();
        input.reset_data();
        kept.reset_data();
        in_scale.reset_data();
        out_scale.reset_data();
        scaled.reset_data();
        in_perm.reset_data();
        out_index.reset_data();
    }

    std::string name() const override { return base4 ? "ButterflyMultiplyBase4Backward" : "ButterflyMultiplyBackward"; }
};

// Runs the forward and, when a gradient will be asked for, hangs the node behind its output.  The
// forward then runs along the backward's pass plan and keeps the activations between the passes
// (device tensors whose backward takes several passes: rows beyond 1024, more than two blocks),
// which the reference's Function leaves to its backward to recompute.
template <typename F>
Tensor differentiable(const Operands &o, const Tensor &input, bool layer, const char *who, F &&forward)
{
    // (a tangent would be dropped silently, with gradients asked for or not)
    for (const Tensor *t : {&o.twiddle, &o.twiddle2, &o.bias, &o.in_scale, &o.out_scale, &input})
        TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(), who, ": no forward-mode derivative");
    bool wanted = false;
    if (at::GradMode::is_enabled()) {
        for (const Tensor *t : {&o.twiddle, &o.twiddle2, &o.bias, &o.in_scale, &o.out_scale, &input})
            wanted = wanted || (t->defined() && t->requires_grad());
    }
    if (!wanted) {
        at::AutoDispatchBelowADInplaceOrView below;
        return forward(nullptr, nullptr);
    }
    std::shared_ptr<MultiplyNode> node(new MultiplyNode(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(o.twiddle, o.twiddle2, input, o.bias, o.in_scale, o.out_scale));
    Tensor kept, scaled, out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        out = forward(input.is_cuda() ? &kept : nullptr, &scaled);
    }
    node->twiddle = SavedVariable(o.twiddle, false);
    if (o.base4) node->twiddle2 = SavedVariable(o.twiddle2, false);
    node->input = SavedVariable(input, false);
    if (kept.defined()) {
        node->kept = SavedVariable(kept, false);
        node->has_kept = true;
    }
    if (scaled.defined()) {
        node->in_scale = SavedVariable(o.in_scale, false);
        node->out_scale = SavedVariable(o.out_scale, false);
        node->scaled = SavedVariable(scaled, false);
        node->has_scaled = true;
    }
    node->real_input = o.real_input;
    node->real_output = o.real_output;
    // (saved like the other operands: changed in place before the backward they raise)
    if (o.in_perm.defined()) {
        node->in_perm = SavedVariable(o.in_perm, false);
        node->has_in_perm = true;
    }
    if (o.out_index.defined()) {
        node->out_index = SavedVariable(o.out_index, false);
        node->has_out_index = true;
    }
    node->base4 = o.base4;
    node->increasing_stride = o.increasing_stride;
    node->with_bias = o.bias.defined();
    node->layer = layer;
    node->who = who;
    torch::autograd::set_history(out, node);
    return out;
}

// ---- registered operators ------------------------------------------------------------------------------

Tensor opt(const c10::optional<Tensor> &t) { return t.has_value() ? t.value() : Tensor(); }

Operands base2(const Tensor &twiddle, bool increasing_stride, const Tensor &bias = Tensor(),
               const Tensor &in_perm = Tensor(), const Tensor &out_index = Tensor())
{
    Operands o;
    o.twiddle = twiddle;
    o.bias = bias;
    o.in_perm = in_perm;
    o.out_index = out_index;
    o.increasing_stride = increasing_stride;
    return o;
}

Operands base4(const Tensor &twiddle4, const Tensor &twiddle2, bool increasing_stride, const Tensor &bias = Tensor())
{
    Operands o = base2(twiddle4, increasing_stride, bias);
    o.twiddle2 = twiddle2;
    o.base4 = true;
    return o;
}

Tensor butterfly_multiply_fw(const Tensor twiddle, const Tensor input, bool increasing_stride,
                             c10::optional<int64_t> output_size)
{
    return multiply_fw(base2(twiddle, increasing_stride), input, output_size, nullptr, "butterfly_multiply_fw");
}

std::tuple<Tensor, Tensor> butterfly_multiply_bw(const Tensor twiddle, const Tensor input,
                                                 const Tensor grad, bool increasing_stride)
{
    Gradients d = multiply_bw(base2(twiddle, increasing_stride), input, grad, Tensor(), false, "butterfly_multiply_bw");
    return {d.twiddle, d.input};
}

Tensor butterfly_multiply(Tensor twiddle, Tensor input, bool increasing_stride, c10::optional<int64_t> output_size)
{
    const char *who = "butterfly_multiply";
    const Operands o = base2(twiddle, increasing_stride);
    return differentiable(o, input, false, who, [&](Tensor *keep, Tensor *) { return multiply_fw(o, input, output_size, keep, who); });
}

// New operators (no counterpart in the reference's op set): the layer bias folded into the
// multiply, where Butterfly.post_process runs a separate elementwise pass
// (torch_butterfly/butterfly.py:152-169).  bias: (nstacks, output_size).
Tensor butterfly_multiply_bias_fw(const Tensor twiddle, const Tensor input, const Tensor bias,
                                  bool increasing_stride, c10::optional<int64_t> output_size)
{
    TORCH_CHECK(bias.defined(), "butterfly_multiply_bias_fw: bias is undefined");
    return multiply_fw(base2(twiddle, increasing_stride, bias), input, output_size, nullptr, "butterfly_multiply_bias_fw");
}

// (d_twiddle, d_input, d_bias): the backward of butterfly_multiply_bias_fw
std::tuple<Tensor, Tensor, Tensor> butterfly_multiply_bias_bw(const Tensor twiddle, const Tensor input,
                                                              const Tensor grad, bool increasing_stride)
{
    Gradients d = multiply_bw(base2(twiddle, increasing_stride), input, grad, Tensor(), true, "butterfly_multiply_bias_bw");
    return {d.twiddle, d.input, d.bias};
}

Tensor butterfly_multiply_bias(Tensor twiddle, Tensor input, Tensor bias, bool increasing_stride,
                               c10::optional<int64_t> output_size)
{
    const char *who = "butterfly_multiply_bias";
    TORCH_CHECK(bias.defined(), "butterfly_multiply_bias: bias is undefined");
    const Operands o = base2(twiddle, increasing_stride, bias);
    return differentiable(o, input, false, who, [&](Tensor *keep, Tensor *) { return multiply_fw(o, input, output_size, keep, who); });
}

// New operators: the multiply between two fixed column permutations, folded into the first
// read and the last write (in front: u[c] = input[in_perm[c]]; behind: output[out_index[c]] =
// y[c]; bias (nstacks, output_size) indexed by c).  Where the reference chains FixedPermutation
// and Butterfly modules (torch_butterfly/special.py:17-66), each permutation costs a pass of
// its own over the activations.  Tables: int32 (n,), undefined = identity.
Tensor butterfly_multiply_perm_fw(const Tensor twiddle, const Tensor input, c10::optional<Tensor> in_perm,
                                  c10::optional<Tensor> out_index, c10::optional<Tensor> bias,
                                  bool increasing_stride, c10::optional<int64_t> output_size)
{
    return multiply_fw(base2(twiddle, increasing_stride, opt(bias), opt(in_perm), opt(out_index)), input, output_size,
                       nullptr, "butterfly_multiply_perm_fw");
}

// (d_twiddle, d_input, d_bias); d_bias is empty unless with_bias
std::tuple<Tensor, Tensor, Tensor> butterfly_multiply_perm_bw(const Tensor twiddle, const Tensor input,
                                                              const Tensor grad, c10::optional<Tensor> in_perm,
                                                              c10::optional<Tensor> out_index, bool with_bias,
                                                              bool increasing_stride)
{
    Gradients d = multiply_bw(base2(twiddle, increasing_stride, Tensor(), opt(in_perm), opt(out_index)), input, grad,
                              Tensor(), with_bias, "butterfly_multiply_perm_bw");
    if (!with_bias) d.bias = at::empty({0}, grad.options());  // the schema has no optional results
    return {d.twiddle, d.input, d.bias};
}

Tensor butterfly_multiply_perm(Tensor twiddle, Tensor input, c10::optional<Tensor> in_perm,
                               c10::optional<Tensor> out_index, c10::optional<Tensor> bias, bool increasing_stride,
                               c10::optional<int64_t> output_size)
{
    const char *who = "butterfly_multiply_perm";
    const Operands o = base2(twiddle, increasing_stride, opt(bias), opt(in_perm), opt(out_index));
    return differentiable(o, input, false, who, [&](Tensor *keep, Tensor *) { return multiply_fw(o, input, output_size, keep, who); });
}

// A whole layer: input (*, width), zero padded or trimmed to n for each of the stacks (the leading
// dimension of the factors), to the first out_size columns of the stacks' outputs side by side,
// plus bias (out_size).  in_perm / out_index as above.  What Butterfly.forward does around its
// multiply (torch_butterfly/butterfly.py:113-169), without the chain of views, slices and pads
// that autograd would record and replay for it.
// in_scale (up to n entries) / out_scale (up to nstacks * n): diagonals directly in front of /
// behind the factors, multiplied into the first / last of them.  real_input / real_output, complex
// factors: the input is real, only the real part of the output is returned.
Tensor butterfly_layer(Tensor twiddle, Tensor input, c10::optional<Tensor> bias, c10::optional<Tensor> in_perm,
                       c10::optional<Tensor> out_index, c10::optional<Tensor> in_scale, c10::optional<Tensor> out_scale,
                       bool increasing_stride, int64_t out_size, bool real_input, bool real_output)
{
    const char *who = "butterfly_layer";
    Operands o = base2(twiddle, increasing_stride, opt(bias), opt(in_perm), opt(out_index));
    o.in_scale = opt(in_scale);
    o.out_scale = opt(out_scale);
    o.real_input = real_input;
    o.real_output = real_output;
    return differentiable(o, input, true, who, [&](Tensor *keep, Tensor *scaled) {
        return layer_fw(o, input, out_size, keep, scaled, who);
    });
}

Tensor butterfly_layer_base4(Tensor twiddle4, Tensor twiddle2, Tensor input, c10::optional<Tensor> bias,
                             bool increasing_stride, int64_t out_size)
{
    const char *who = "butterfly_layer_base4";
    const Operands o = base4(twiddle4, twiddle2, increasing_stride, opt(bias));
    return differentiable(o, input, true, who, [&](Tensor *keep, Tensor *) {
        return layer_fw(o, input, out_size, keep, nullptr, who);
    });
}

Tensor butterfly_multiply_base4_fw(const Tensor twiddle4, const Tensor twiddle2, const Tensor input,
                                   bool increasing_stride, c10::optional<int64_t> output_size)
{
    return multiply_fw(base4(twiddle4, twiddle2, increasing_stride), input, output_size, nullptr,
                       "butterfly_multiply_base4_fw");
}

std::tuple<Tensor, Tensor, Tensor> butterfly_multiply_base4_bw(const Tensor twiddle4, const Tensor twiddle2,
                                                               const Tensor input, const Tensor grad,
                                                               bool increasing_stride)
{
    Gradients d = multiply_bw(base4(twiddle4, twiddle2, increasing_stride), input, grad, Tensor(), false,
                              "butterfly_multiply_base4_bw");
    return {d.twiddle, d.twiddle2, d.input};
}

Tensor butterfly_multiply_base4(Tensor twiddle4, Tensor twiddle2, Tensor input, bool increasing_stride,
                                c10::optional<int64_t> output_size)
{
    const char *who = "butterfly_multiply_base4";
    const Operands o = base4(twiddle4, twiddle2, increasing_stride);
    return differentiable(o, input, false, who, [&](Tensor *keep, Tensor *) { return multiply_fw(o, input, output_size, keep, who); });
}

// d_bias (nstacks, output_size) = sum of grad (batch, nstacks, output_size) over the batch.
Tensor butterfly_bias_grad(const Tensor grad)
{
    CHECK_DEVICE(grad);
    CHECK_DIM(grad, 3);
    require_device(grad, "butterfly_bias_grad");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
    const Tensor g = grad.resolve_conj();
    bf_problem p = {};
    p.dtype = dtype_code(g, "butterfly_bias_grad");
    p.batch = g.size(0);
    p.nstacks = g.size(1);
    p.output_size = g.size(2);
    p.input_size = g.size(2);
    p.nblocks = 1;
    p.log_n = 1;
    while (((int64_t)1 << p.log_n) < p.output_size) ++p.log_n;
    set_strides(p.output_stride, g);
    Tensor d_bias = at::empty({p.nstacks, p.output_size}, g.options());
    const size_t ws_bytes = valid_size(bf_butterfly_bias_grad_workspace_bytes(&p));
    Tensor ws = at::empty({(int64_t)ws_bytes}, g.options().dtype(at::kByte));
    check_rc(bf_butterfly_bias_grad(&p, g.data_ptr(), d_bias.data_ptr(), ws.data_ptr(), ws_bytes, current_stream()),
             "butterfly_bias_grad");
    return d_bias;
}

// ---- diagonals folded into the factors ------------------------------------------------------
//
// twiddle (S, nb, log_n, n/2, 2, 2) -> the factors of diag(out_scale) B diag(in_scale): what a
// Diagonal module in front of / behind a Butterfly (torch_butterfly/diagonal.py:31-38) does to
// the activations, done to the first / last factor instead.  in_scale up to n entries,
// out_scale up to S * n, same dtype as twiddle; undefined = no diagonal on that side.
struct ScaleShapes {
    int64_t nstacks, nblocks, log_n;
};

ScaleShapes scale_shapes(const Tensor &twiddle, const Tensor &in_scale, const Tensor &out_scale, const char *who)
{
    CHECK_DEVICE(twiddle);
    CHECK_DIM(twiddle, 6);
    ScaleShapes s{twiddle.size(0), twiddle.size(1), twiddle.size(2)};
    TORCH_CHECK(s.log_n >= 1 && s.log_n <= 30 && s.nblocks >= 1, who, ": twiddle must have at least one factor");
    const int64_t n = (int64_t)1 << s.log_n;
    CHECK_SHAPE(twiddle, s.nstacks, s.nblocks, s.log_n, n / 2, 2, 2);
    dtype_code(twiddle, who);
    for (const Tensor *v : {&in_scale, &out_scale}) {
        if (!v->defined()) continue;
        TORCH_CHECK(v->device() == twiddle.device(), who, ": diagonals must be on the device of twiddle");
        TORCH_CHECK(v->dim() == 1, who, ": diagonals must be vectors");
        TORCH_CHECK(v->scalar_type() == twiddle.scalar_type(), who, ": diagonals must have the dtype of twiddle");
    }
    TORCH_CHECK(!in_scale.defined() || in_scale.size(0) <= n, who, ": in_scale has more than n entries");
    TORCH_CHECK(!out_scale.defined() || out_scale.size(0) <= s.nstacks * n, who,
                ": out_scale has more than nstacks * n entries");
    return s;
}

Tensor butterfly_scale_twiddle_fw(const Tensor twiddle, c10::optional<Tensor> in_scale,
                                  c10::optional<Tensor> out_scale, bool increasing_stride)
{
    const char *who = "butterfly_scale_twiddle_fw";
    const Tensor din = opt(in_scale), dout = opt(out_scale);
    const ScaleShapes s = scale_shapes(twiddle, din, dout, who);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(twiddle.device());
    const Tensor tw = dense(twiddle);
    const Tensor a = din.defined() ? dense(din) : din, b = dout.defined() ? dense(dout) : dout;
    Tensor out = at::empty_like(tw);
    check_rc(bf_butterfly_scale_twiddle(dtype_code(tw, who), s.nstacks, s.nblocks, s.log_n, increasing_stride,
                                        tw.data_ptr(), a.defined() ? a.data_ptr() : nullptr,
                                        a.defined() ? a.size(0) : 0, b.defined() ? b.data_ptr() : nullptr,
                                        b.defined() ? b.size(0) : 0, out.data_ptr(), current_stream()),
             who);
    return out;
}

// (d_twiddle, d_in_scale, d_out_scale); an empty tensor stands for the gradient of an absent diagonal
std::tuple<Tensor, Tensor, Tensor> butterfly_scale_twiddle_bw(const Tensor twiddle, c10::optional<Tensor> in_scale,
                                                              c10::optional<Tensor> out_scale, const Tensor grad,
                                                              bool increasing_stride)
{
    const char *who = "butterfly_scale_twiddle_bw";
    const Tensor din = opt(in_scale), dout = opt(out_scale);
    const ScaleShapes s = scale_shapes(twiddle, din, dout, who);
    CHECK_DEVICE(grad);
    TORCH_CHECK(grad.sizes() == twiddle.sizes() && grad.scalar_type() == twiddle.scalar_type() &&
                    grad.device() == twiddle.device(),
                who, ": grad must match twiddle in shape, dtype and device");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(twiddle.device());
    const Tensor tw = dense(twiddle), g = dense(grad);
    const Tensor a = din.defined() ? dense(din) : din, b = dout.defined() ? dense(dout) : dout;
    Tensor d_tw = at::empty_like(tw);
    Tensor d_a = at::empty({a.defined() ? a.size(0) : 0}, tw.options());
    Tensor d_b = at::empty({b.defined() ? b.size(0) : 0}, tw.options());
    check_rc(bf_butterfly_scale_twiddle_bw(dtype_code(tw, who), s.nstacks, s.nblocks, s.log_n, increasing_stride,
                                           tw.data_ptr(), a.defined() ? a.data_ptr() : nullptr,
                                           a.defined() ? a.size(0) : 0, b.defined() ? b.data_ptr() : nullptr,
                                           b.defined() ? b.size(0) : 0, g.data_ptr(), d_tw.data_ptr(),
                                           d_a.data_ptr(), d_b.data_ptr(), current_stream()),
             who);
    return {d_tw, d_a, d_b};
}

using torch::autograd::AutogradContext;

void scale_factors(const Tensor &twiddle, const Operands &o, Tensor &scaled, const char *)
{
    scaled = butterfly_scale_twiddle_fw(twiddle, o.in_scale.defined() ? c10::optional<Tensor>(o.in_scale) : c10::nullopt,
                                        o.out_scale.defined() ? c10::optional<Tensor>(o.out_scale) : c10::nullopt,
                                        o.increasing_stride);
}

void scale_factors_bw(const Tensor &twiddle, const Operands &o, const Tensor &grad, Tensor &d_twiddle, Tensor &d_in,
                      Tensor &d_out, const char *)
{
    auto r = butterfly_scale_twiddle_bw(twiddle, o.in_scale.defined() ? c10::optional<Tensor>(o.in_scale) : c10::nullopt,
                                        o.out_scale.defined() ? c10::optional<Tensor>(o.out_scale) : c10::nullopt, grad,
                                        o.increasing_stride);
    d_twiddle = std::get<0>(r);
    if (o.in_scale.defined()) d_in = std::get<1>(r);
    if (o.out_scale.defined()) d_out = std::get<2>(r);
}

class ButterflyScaleTwiddle : public torch::autograd::Function<ButterflyScaleTwiddle> {
public:
    static Tensor forward(AutogradContext *ctx, Tensor twiddle, c10::optional<Tensor> in_scale,
                          c10::optional<Tensor> out_scale, bool increasing_stride)
    {
        ctx->saved_data["increasing_stride"] = increasing_stride;
        ctx->saved_data["has_in"] = in_scale.has_value();
        ctx->saved_data["has_out"] = out_scale.has_value();
        variable_list saved = {twiddle};
        if (in_scale.has_value()) saved.push_back(in_scale.value());
        if (out_scale.has_value()) saved.push_back(out_scale.value());
        ctx->save_for_backward(saved);
        return butterfly_scale_twiddle_fw(twiddle, in_scale, out_scale, increasing_stride);
    }

    static variable_list backward(AutogradContext *ctx, variable_list grad_output)
    {
        const auto saved = ctx->get_saved_variables();
        const bool has_in = ctx->saved_data["has_in"].toBool(), has_out = ctx->saved_data["has_out"].toBool();
        c10::optional<Tensor> in_scale, out_scale;
        size_t next = 1;
        if (has_in) in_scale = saved[next++];
        if (has_out) out_scale = saved[next++];
        auto r = butterfly_scale_twiddle_bw(saved[0], in_scale, out_scale, grad_output[0],
                                            ctx->saved_data["increasing_stride"].toBool());
        return {std::get<0>(r), has_in ? std::get<1>(r) : Tensor(), has_out ? std::get<2>(r) : Tensor(), Tensor()};
    }
};

Tensor butterfly_scale_twiddle(Tensor twiddle, c10::optional<Tensor> in_scale, c10::optional<Tensor> out_scale,
                               bool increasing_stride)
{
    return ButterflyScaleTwiddle::apply(twiddle, in_scale, out_scale, increasing_stride);
}

int64_t hip_version() { return bf_hip_version(); }

}  // namespace

TORCH_LIBRARY(torch_butterfly, m)
{
    m.def("butterfly_multiply_fw", butterfly_multiply_fw);
    m.def("butterfly_multiply_bw", butterfly_multiply_bw);
    m.def("butterfly_multiply", butterfly_multiply);
    m.def("butterfly_multiply_bias_fw", butterfly_multiply_bias_fw);
    m.def("butterfly_bias_grad", butterfly_bias_grad);
    m.def("butterfly_multiply_bias_bw", butterfly_multiply_bias_bw);
    m.def("butterfly_multiply_bias", butterfly_multiply_bias);
    m.def("butterfly_multiply_perm_fw", butterfly_multiply_perm_fw);
    m.def("butterfly_multiply_perm_bw", butterfly_multiply_perm_bw);
    m.def("butterfly_multiply_perm", butterfly_multiply_perm);
    m.def("butterfly_layer", butterfly_layer);
    m.def("butterfly_layer_base4", butterfly_layer_base4);
    m.def("butterfly_scale_twiddle_fw", butterfly_scale_twiddle_fw);
    m.def("butterfly_scale_twiddle_bw", butterfly_scale_twiddle_bw);
    m.def("butterfly_scale_twiddle", butterfly_scale_twiddle);
    m.def("butterfly_multiply_base4_fw", butterfly_multiply_base4_fw);
    m.def("butterfly_multiply_base4_bw", butterfly_multiply_base4_bw);
    m.def("butterfly_multiply_base4", butterfly_multiply_base4);
    m.def("hip_version", hip_version);
}
