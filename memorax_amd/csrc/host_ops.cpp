// The host side of the library for torch: what runs between a Python call and the kernel launches behind it, as
// native code (the extension module memorax_amd._native).
//
// A call on a small rollout is bound by the host: checking the arguments, allocating the outputs, filling in a
// C call and -- by far the most -- recording and running the autograd node.  As Python (ctypes calls inside
// torch.autograd.Function) a forward and backward pair took 125-165 us whatever the arrays' size, most of it in
// the backward, where the engine's thread had to fetch the interpreter's lock from the thread that waits for it.
// Here the nodes are C++ (no interpreter in the backward at all) and one layer of functions does checks,
// allocation and launch for them and for memorax_amd/kernels.py alike.
//
// The entry points of the C ABI are bound at run time (bind()) from whatever build of the library Python has
// loaded; nothing here links against it.
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContextLight.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/generated/Functions.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <numeric>

#include "memorax_amd.h"

namespace py = pybind11;

namespace {

using at::Tensor;
using c10::IntArrayRef;
using c10::ScalarType;
using OptTensor = std::optional<Tensor>;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------------------ entry points
#define MRX_BOUND(X)                                                                                                 \
    X(mrx_status_string) X(mrx_chunk_size) X(mrx_delta_chunk_size) X(mrx_scan_workspace) X(mrx_column_sum) X(mrx_linear_scan_fwd_segmented) X(mrx_linear_scan_bwd_segmented)     \
    X(mrx_linear_scan_last) X(mrx_mingru_scan_fwd) X(mrx_mingru_scan_fwd_segmented) X(mrx_mingru_scan_bwd_segmented) X(mrx_mlstm_gates_fwd)                     \
    X(mrx_place_inputs) X(mrx_mlstm_gate_rows_fwd) X(mrx_mlstm_gate_rows_bwd)                                                           \
    X(mrx_mlstm_keys_fwd) X(mrx_mlstm_keys_bwd) X(mrx_mlstm_read_fwd) X(mrx_mlstm_read_bwd)                         \
    X(mrx_mlstm_gates_bwd) X(mrx_rms_norm_fwd) X(mrx_rms_norm_bwd) X(mrx_layer_norm_fwd) X(mrx_layer_norm_bwd)       \
    X(mrx_silu_gate_fwd) X(mrx_silu_gate_bwd) X(mrx_residual_add) X(mrx_linear_attn_fwd) X(mrx_linear_attn_bwd)                          \
    X(mrx_linear_attn_fwd_chunk_parallel) X(mrx_linear_attn_bwd_chunk_parallel)                                      \
    X(mrx_linear_attn_chunk_parallel_pays) X(mrx_linear_attn_norm_fwd) X(mrx_linear_attn_norm_bwd)                   \
    X(mrx_gated_linear_attn_fwd) X(mrx_gated_linear_attn_bwd) X(mrx_delta_rule_fwd) X(mrx_delta_rule_bwd)            \
    X(mrx_delta_rule_fwd_noalloc) X(mrx_deltanet_fwd) X(mrx_deltanet_bwd) X(mrx_linear_attn_step)                    \
    X(mrx_gated_linear_attn_step) X(mrx_delta_rule_step) X(mrx_causal_conv_silu_fwd) X(mrx_causal_conv_silu_bwd)     \
    X(mrx_mamba_elements_fwd) X(mrx_mamba_elements_bwd) X(mrx_decay_last) X(mrx_mamba_readout_fwd)                   \
    X(mrx_mamba_readout_bwd) X(mrx_deltanet_step) X(mrx_mingru_step) X(mrx_row_dense) X(mrx_dense_grads) X(mrx_dense_grads_workspace)                  \
    X(mrx_gated_recurrence_act) X(mrx_closed_row_dense) X(mrx_closed_gated_recurrence_act) X(mrx_gated_scan_pays) X(mrx_gated_scan_fwd) X(mrx_gated_scan_bwd)                                                                                       \
    X(mrx_dense_f32_workspace) X(mrx_dense_f32) X(mrx_dense_f32_input_grad_workspace) X(mrx_dense_f32_input_grad) X(mrx_lru_params_fwd)                       \
    X(mrx_lru_params_bwd) X(mrx_column_product_workspace) X(mrx_column_product) X(mrx_dense_rows_suit) X(mrx_dense_pack) X(mrx_dense_rows) X(mrx_dense_rows_input_grad)                          \
    X(mrx_lru_step) X(mrx_mlstm_step) X(mrx_linear_attn_norm_fwd_chunk_parallel) X(mrx_linear_attn_norm_bwd_chunk_parallel) \
    X(mrx_gated_linear_attn_fwd_chunk_parallel) X(mrx_gated_linear_attn_bwd_chunk_parallel)
struct {
#define MRX_MEMBER(name) decltype(&::name) name = nullptr;
    MRX_BOUND(MRX_MEMBER)
#undef MRX_MEMBER
} lib;

void bind(const py::dict &addresses)
{
#define MRX_TAKE(name) lib.name = reinterpret_cast<decltype(&::name)>(addresses[#name].cast<uintptr_t>());
    MRX_BOUND(MRX_TAKE)
#undef MRX_TAKE
}

void check(int status, const char *what)
{
    TORCH_CHECK(status == MRX_OK, what, " failed: ", lib.mrx_status_string(status), " (status ", status, ")");
}

// --------------------------------------------------------------------------------------------------- arguments
void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

template <typename P = void> P *ptr(const Tensor &t) { return t.defined() ? static_cast<P *>(t.data_ptr()) : nullptr; }
template <typename P = void> P *ptr(const OptTensor &t) { return t.has_value() ? ptr<P>(*t) : nullptr; }
float *fptr(const Tensor &t) { return ptr<float>(t); }
float *fptr(const OptTensor &t) { return ptr<float>(t); }

int code(ScalarType dt)
{
    switch (dt) {
    case at::kFloat: return MRX_F32;
    case at::kBFloat16: return MRX_BF16;
    case at::kComplexFloat: return MRX_C64;
    default: return -1;
    }
}

void chk(const Tensor &t, const char *name)
{
    TORCH_CHECK_VALUE(t.is_cuda(), name, " must live on the GPU (memorax_amd has no CPU path)");
    TORCH_CHECK_VALUE(t.is_contiguous(), name, " must be contiguous");
}
void chk(const Tensor &t, const char *name, ScalarType dt)
{
    chk(t, name);
    TORCH_CHECK_VALUE(t.scalar_type() == dt, name, " must be ", dt, ", got ", t.scalar_type());
}
void chk(const Tensor &t, const char *name, ScalarType dt, IntArrayRef shape)
{
    chk(t, name, dt);
    TORCH_CHECK_VALUE(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes());
}
void chk(const OptTensor &t, const char *name, ScalarType dt, IntArrayRef shape)
{
    if (t.has_value() && t->defined()) chk(*t, name, dt, shape);
}

// contiguous and on a 16-byte boundary; the tensor itself where it is that already (a parameter may be a view into a flat vector)
Tensor dense16(const Tensor &t)
{
    if (!t.defined()) return t;
    const Tensor c = t.contiguous();
    return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone();
}
Tensor dense16(const OptTensor &t) { return t.has_value() ? dense16(*t) : Tensor(); }

Tensor fresh(IntArrayRef shape, ScalarType dt, const Tensor &like)
{
    return at::detail::empty_cuda(shape, dt, like.device(), std::nullopt);
}
Tensor fresh_like(const Tensor &t) { return fresh(t.sizes(), t.scalar_type(), t); }

// Reset flags (B,T): bool, uint8 and float32 go to the kernels as they are, anything else as flag != 0.
struct Done {
    Tensor t;
    int dtype;
    Done(const Tensor &done, int64_t B, int64_t T)
    {
        TORCH_CHECK_VALUE(done.dim() == 2 && done.size(0) == B && done.size(1) == T, "done must have shape [", B, ", ", T, "], got ",
                          done.sizes());
        const auto dt = done.scalar_type();
        t = (dt == at::kBool || dt == at::kByte || dt == at::kFloat) ? done.contiguous() : done.ne(0).contiguous();
        dtype = dt == at::kFloat ? MRX_DONE_F32 : MRX_DONE_U8;
        TORCH_CHECK_VALUE(t.is_cuda(), "done must live on the GPU (memorax_amd has no CPU path)");
    }
    const void *p() const { return t.data_ptr(); }
};

int64_t chunk_size(ScalarType dt, bool delta) { return delta ? lib.mrx_delta_chunk_size(code(dt)) : lib.mrx_chunk_size(code(dt)); }

int compute_units(const Tensor &t) { return at::cuda::getDeviceProperties(t.get_device())->multiProcessorCount; }

// ----------------------------------------------------------------------------------- checks, allocation, launch
// ---- diagonal scans
struct ScanOut {
    Tensor h, h_last, P_last;
};

void chk_scan_dtype(ScalarType dt, bool complex, const char *what)
{
    TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16 || (complex && dt == at::kComplexFloat), what, " supports float32, ",
                      complex ? "complex64 and bfloat16" : "bfloat16");
}

// scratch for the scans that cut time into segments; undefined (a null pointer) where the shape is not served that way
Tensor scan_workspace(const Tensor &x, int64_t B, int64_t T, int64_t D, ScalarType dt, int what)
{
    const int64_t bytes = lib.mrx_scan_workspace(B, T, D, code(dt), what);
    return bytes ? fresh({bytes}, at::kByte, x) : Tensor();
}

ScanOut scan_fwd(const Tensor &a, const Tensor &b, const Tensor &done_, const OptTensor &h0, const OptTensor &P0, bool want_P)
{
    TORCH_CHECK_VALUE(b.dim() == 3, "b must be (B,T,D)");
    const int64_t B = b.size(0), T = b.size(1), D = b.size(2);
    const auto dt = b.scalar_type();
    chk_scan_dtype(dt, true, "linear_scan");
    const auto ct = dt == at::kBFloat16 ? at::kFloat : dt;   // the carries' type
    const bool ti = a.dim() == 1;
    if (ti) chk(a, "a", dt, {D});
    else chk(a, "a", dt, {B, T, D});
    chk(b, "b");
    chk(h0, "h0", ct, {B, D});
    chk(P0, "P0", ct, {B, D});
    const Done done(done_, B, T);
    ScanOut r{fresh_like(b), fresh({B, D}, ct, b), want_P ? fresh({B, D}, ct, b) : Tensor()};
    const Tensor workspace = scan_workspace(b, B, T, D, dt, 0);
    check(lib.mrx_linear_scan_fwd_segmented(stream(), ptr(a), ptr(b), done.p(), ptr(h0), ptr(P0), ptr(r.h), ptr(r.h_last), ptr(r.P_last), B, T, D,
                                  code(dt), done.dtype, ti, ptr(workspace)),
          "mrx_linear_scan_fwd");
    return r;
}

struct ScanGrads {
    Tensor da, db, dh0;
};

ScanGrads scan_bwd(const Tensor &a, const Tensor &h, const Tensor &done_, const OptTensor &h0, const Tensor &g, const OptTensor &g_last,
                   bool sum_da)
{
    TORCH_CHECK_VALUE(g.dim() == 3, "g must be (B,T,D)");
    const int64_t B = g.size(0), T = g.size(1), D = g.size(2);
    const auto dt = g.scalar_type();
    chk_scan_dtype(dt, true, "linear_scan");
    const auto ct = dt == at::kBFloat16 ? at::kFloat : dt;
    const bool ti = a.dim() == 1;
    if (ti) chk(a, "a", dt, {D});
    else chk(a, "a", dt, {B, T, D});
    chk(h, "h", dt, {B, T, D});
    chk(g, "g", dt);
    chk(h0, "h0", ct, {B, D});
    chk(g_last, "g_last", ct, {B, D});
    const Done done(done_, B, T);
    TORCH_CHECK_VALUE(ti || !sum_da, "sum_da belongs to a time-invariant a");
    ScanGrads r{sum_da ? fresh({B, D}, ct, g) : fresh_like(g), fresh_like(g), fresh({B, D}, ct, g)};
    const Tensor workspace = scan_workspace(g, B, T, D, dt, MRX_SCAN_BACKWARD | (sum_da ? MRX_SCAN_SUM_DA : 0));
    check(lib.mrx_linear_scan_bwd_segmented(stream(), ptr(a), ptr(h), done.p(), ptr(h0), ptr(g), ptr(g_last), ptr(r.da), ptr(r.db), ptr(r.dh0), B, T, D,
                                  code(dt), done.dtype, sum_da ? MRX_A_TIME_INVARIANT_SUM_DA : int(ti), ptr(workspace)),
          "mrx_linear_scan_bwd");
    return r;
}

Tensor scan_last(const Tensor &a, const Tensor &b, const Tensor &done_, const OptTensor &h0)
{
    TORCH_CHECK_VALUE(b.dim() == 3, "b must be (B,T,D)");
    const int64_t B = b.size(0), T = b.size(1), D = b.size(2);
    const auto dt = b.scalar_type();
    TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kComplexFloat, "linear_scan_last supports float32 and complex64");
    TORCH_CHECK_VALUE(a.dim() == 3 && a.size(0) == B && a.size(1) == T && a.size(2) > 0 && D % a.size(2) == 0,
                      "a must be (B,T,D/group), got ", a.sizes(), " for b ", b.sizes());
    chk(a, "a", dt);
    chk(b, "b", dt);
    chk(h0, "h0", dt, {B, D});
    const Done done(done_, B, T);
    Tensor h_last = fresh({B, D}, dt, b);
    check(lib.mrx_linear_scan_last(stream(), ptr(a), ptr(b), done.p(), ptr(h0), ptr(h_last), B, T, D, D / a.size(2), code(dt), done.dtype),
          "mrx_linear_scan_last");
    return h_last;
}

ScanOut mingru_fwd(const Tensor &z, const Tensor &x, const Tensor &done_, const OptTensor &h0, const OptTensor &P0, bool want_P)
{
    TORCH_CHECK_VALUE(z.dim() == 3, "z must be (B,T,D)");
    const int64_t B = z.size(0), T = z.size(1), D = z.size(2);
    const auto dt = z.scalar_type();
    chk_scan_dtype(dt, false, "mingru_scan");
    chk(z, "z");
    chk(x, "h_tilde", dt, z.sizes());
    chk(h0, "h0", at::kFloat, {B, D});
    chk(P0, "P0", at::kFloat, {B, D});
    const Done done(done_, B, T);
    ScanOut r{fresh_like(z), fresh({B, D}, at::kFloat, z), want_P ? fresh({B, D}, at::kFloat, z) : Tensor()};
    const Tensor workspace = scan_workspace(z, B, T, D, dt, MRX_SCAN_MINGRU);
    check(lib.mrx_mingru_scan_fwd_segmented(stream(), ptr(z), ptr(x), done.p(), fptr(h0), fptr(P0), ptr(r.h), fptr(r.h_last), fptr(r.P_last), B, T, D,
                                  code(dt), done.dtype, ptr(workspace)),
          "mrx_mingru_scan_fwd");
    return r;
}

ScanGrads mingru_bwd(const Tensor &z, const Tensor &x, const Tensor &h, const Tensor &done_, const OptTensor &h0, const Tensor &g,
                     const OptTensor &g_last)
{
    TORCH_CHECK_VALUE(g.dim() == 3, "g must be (B,T,D)");
    const int64_t B = g.size(0), T = g.size(1), D = g.size(2);
    const auto dt = g.scalar_type();
    chk_scan_dtype(dt, false, "mingru_scan");
    chk(z, "z", dt, g.sizes());
    chk(x, "h_tilde", dt, g.sizes());
    chk(h, "h", dt, g.sizes());
    chk(g, "g");
    chk(h0, "h0", at::kFloat, {B, D});
    chk(g_last, "g_last", at::kFloat, {B, D});
    const Done done(done_, B, T);
    ScanGrads r{fresh_like(g), fresh_like(g), fresh({B, D}, at::kFloat, g)};
    const Tensor workspace = scan_workspace(g, B, T, D, dt, MRX_SCAN_MINGRU | MRX_SCAN_BACKWARD);
    check(lib.mrx_mingru_scan_bwd_segmented(stream(), ptr(z), ptr(x), ptr(h), done.p(), fptr(h0), ptr(g), fptr(g_last), ptr(r.da), ptr(r.db),
                                  fptr(r.dh0), B, T, D, code(dt), done.dtype, ptr(workspace)),
          "mrx_mingru_scan_bwd");
    return r;
}

// ---- the mLSTM stabiliser
std::array<Tensor, 3> mlstm_gates_fwd(const Tensor &li, const Tensor &lf, const Tensor &done_, const OptTensor &m0, double g_floor)
{
    TORCH_CHECK_VALUE(li.dim() == 3, "log_i must be (B,T,H)");
    const int64_t B = li.size(0), T = li.size(1), H = li.size(2);
    chk(li, "log_i", at::kFloat);
    chk(lf, "log_f", at::kFloat, {B, T, H});
    chk(m0, "m0", at::kFloat, {B, H});
    const Done done(done_, B, T);
    std::array<Tensor, 3> r{fresh_like(li), fresh_like(li), fresh_like(li)};
    check(lib.mrx_mlstm_gates_fwd(stream(), fptr(li), fptr(lf), done.p(), fptr(m0), fptr(r[0]), fptr(r[1]), fptr(r[2]), B, T, H, done.dtype,
                                  (float)g_floor),
          "mrx_mlstm_gates_fwd");
    return r;
}

std::array<Tensor, 3> mlstm_gates_bwd(const Tensor &li, const Tensor &lf, const Tensor &done_, const OptTensor &m0, const Tensor &m,
                                      const OptTensor &dm, const OptTensor &dg, const OptTensor &dw, double g_floor, bool want_dm0)
{
    TORCH_CHECK_VALUE(li.dim() == 3, "log_i must be (B,T,H)");
    const int64_t B = li.size(0), T = li.size(1), H = li.size(2);
    chk(li, "log_i", at::kFloat);
    chk(lf, "log_f", at::kFloat, {B, T, H});
    chk(m, "m", at::kFloat, {B, T, H});
    chk(dm, "dm", at::kFloat, {B, T, H});
    chk(dg, "dg", at::kFloat, {B, T, H});
    chk(dw, "dw", at::kFloat, {B, T, H});
    chk(m0, "m0", at::kFloat, {B, H});
    const Done done(done_, B, T);
    std::array<Tensor, 3> r{fresh_like(li), fresh_like(li), want_dm0 ? fresh({B, H}, at::kFloat, li) : Tensor()};
    check(lib.mrx_mlstm_gates_bwd(stream(), fptr(li), fptr(lf), done.p(), fptr(m0), fptr(m), fptr(dm), fptr(dg), fptr(dw), fptr(r[0]),
                                  fptr(r[1]), fptr(r[2]), B, T, H, done.dtype, (float)g_floor),
          "mrx_mlstm_gates_bwd");
    return r;
}

// ---- norms and the gate
void chk_norm_dtype(ScalarType dt)
{
    TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16, "the norm kernels take float32 or bfloat16 arrays");
}

Tensor norm_fwd(const Tensor &x, const OptTensor &scale, const OptTensor &bias, double eps, std::optional<ScalarType> out_dtype, bool center)
{
    TORCH_CHECK_VALUE(x.dim() >= 1, "x must have a feature axis");
    const int64_t D = x.size(-1);
    const auto dt = x.scalar_type(), od = out_dtype.value_or(dt);
    chk_norm_dtype(dt);
    chk_norm_dtype(od);
    chk(x, "x");
    chk(scale, "scale", at::kFloat, {D});
    chk(bias, "bias", at::kFloat, {D});
    Tensor y = fresh(x.sizes(), od, x);
    if (x.numel() == 0) return y;
    const int64_t rows = x.numel() / D;
    if (center)
        check(lib.mrx_layer_norm_fwd(stream(), ptr(x), fptr(scale), fptr(bias), ptr(y), rows, D, code(dt), code(od), (float)eps),
              "mrx_layer_norm_fwd");
    else
        check(lib.mrx_rms_norm_fwd(stream(), ptr(x), fptr(scale), ptr(y), rows, D, code(dt), code(od), (float)eps), "mrx_rms_norm_fwd");
    return y;
}

struct NormGrads {
    Tensor dx, dscale, dbias;
};

NormGrads norm_bwd(const Tensor &x, const OptTensor &scale, const Tensor &dy, double eps, bool want_dparams, const OptTensor &dx_add,
                   bool center)
{
    TORCH_CHECK_VALUE(x.dim() >= 1, "x must have a feature axis");
    const int64_t D = x.size(-1);
    const auto dt = x.scalar_type(), yd = dy.scalar_type();
    chk_norm_dtype(dt);
    chk_norm_dtype(yd);
    chk(x, "x");
    chk(dy, "dy", yd, x.sizes());
    chk(dx_add, "dx_add", dt, x.sizes());
    chk(scale, "scale", at::kFloat, {D});
    NormGrads r{fresh_like(x), {}, {}};
    Tensor work;
    if (want_dparams) {
        r.dscale = fresh({D}, at::kFloat, x);
        if (center) r.dbias = fresh({D}, at::kFloat, x);
        work = fresh({(center ? 2 : 1) * MRX_RMS_NORM_PARTS, D}, at::kFloat, x);
    }
    if (x.numel() == 0) {   // dx (and dx_add) are empty
        if (r.dscale.defined()) r.dscale.zero_();
        if (r.dbias.defined()) r.dbias.zero_();
        return r;
    }
    const int64_t rows = x.numel() / D;
    if (center)
        check(lib.mrx_layer_norm_bwd(stream(), ptr(x), fptr(scale), ptr(dy), ptr(dx_add), ptr(r.dx), fptr(r.dscale), fptr(r.dbias), fptr(work),
                                     rows, D, code(dt), code(yd), (float)eps),
              "mrx_layer_norm_bwd");
    else
        check(lib.mrx_rms_norm_bwd(stream(), ptr(x), fptr(scale), ptr(dy), ptr(dx_add), ptr(r.dx), fptr(r.dscale), fptr(work), rows, D,
                                   code(dt), code(yd), (float)eps),
              "mrx_rms_norm_bwd");
    return r;
}

Tensor silu_gate_fwd(const Tensor &h, const Tensor &g)
{
    const auto dt = h.scalar_type();
    TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16, "silu_gate takes float32 or bfloat16 arrays");
    chk(h, "h");
    chk(g, "g", dt, h.sizes());
    Tensor y = fresh_like(h);
    if (h.numel()) check(lib.mrx_silu_gate_fwd(stream(), ptr(h), ptr(g), ptr(y), h.numel(), code(dt)), "mrx_silu_gate_fwd");
    return y;
}

std::array<Tensor, 2> silu_gate_bwd(const Tensor &h, const Tensor &g, const Tensor &dy)
{
    const auto dt = h.scalar_type();
    TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16, "silu_gate takes float32 or bfloat16 arrays");
    chk(h, "h");
    chk(g, "g", dt, h.sizes());
    chk(dy, "dy", dt, h.sizes());
    std::array<Tensor, 2> r{fresh_like(h), fresh_like(h)};
    if (h.numel())
        check(lib.mrx_silu_gate_bwd(stream(), ptr(h), ptr(g), ptr(dy), ptr(r[0]), ptr(r[1]), h.numel(), code(dt)), "mrx_silu_gate_bwd");
    return r;
}

// ---- chunked attention
struct Shape {
    int64_t B, T, H, dk, dv;
    ScalarType dt;
    Shape(const Tensor &q, const Tensor &k, const Tensor &v)
    {
        TORCH_CHECK_VALUE(q.dim() == 4 && v.dim() == 4, "q, k, v must be (B,T,H,d)");
        B = q.size(0), T = q.size(1), H = q.size(2), dk = q.size(3), dv = v.size(3);
        dt = q.scalar_type();
        TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16, "chunked kernels support float32 and bfloat16");
        chk(q, "q");
        chk(k, "k", dt, {B, T, H, dk});
        chk(v, "v", dt, {B, T, H, dv});
    }
    int64_t chunks(bool delta = false) const { return (T + chunk_size(dt, delta) - 1) / chunk_size(dt, delta); }
    std::array<int64_t, 4> state() const { return {B, H, dv, dk}; }
};

struct AttnOut {
    Tensor o, S_last, S_chk;
    bool parallel;   // S_chk is dense, from the pair of kernels that cuts the work along time
};

AttnOut linear_attn_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done_, const OptTensor &S0, int fmap, bool save_chk,
                        std::optional<bool> chunk_parallel)
{
    const Shape s(q, k, v);
    chk(S0, "S0", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    const bool par = chunk_parallel.has_value() ? *chunk_parallel : lib.mrx_linear_attn_chunk_parallel_pays(s.B, s.T, s.H, code(s.dt)) != 0;
    AttnOut r{fresh_like(v), fresh(s.state(), at::kFloat, q), {}, par};
    if (save_chk || par) r.S_chk = fresh({s.B, s.H, s.chunks(), s.dv, s.dk}, at::kFloat, q);
    if (par)
        check(lib.mrx_linear_attn_fwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S0), ptr(r.o), fptr(r.S_last),
                                                     fptr(r.S_chk), s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
              "mrx_linear_attn_fwd_chunk_parallel");
    else
        check(lib.mrx_linear_attn_fwd(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S0), ptr(r.o), fptr(r.S_last), fptr(r.S_chk), s.B, s.T,
                                      s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
              "mrx_linear_attn_fwd");
    if (!save_chk) r.S_chk = Tensor();
    return r;
}

// Whether the gated or the normalised form cuts the work along time, a workgroup per chunk: the library's rule, and on heads of up to
// 32 features ten chunks or more.  Six launches instead of two for a forward and backward pair cost the host 12 us (82 and 70 us
// from a slow host, 44 and 35 from a fast one); a sequential pair's chain costs 12 us a chunk in bfloat16 (64 features), 7 us up to 32
// features (slow host, bfloat16, 32 sequences: 8 chunks 100 -> 81 and 65 -> 83 us, 16 chunks 180 -> 81 and 112 -> 83 us, 32 chunks
// 334 -> 87 and 219 -> 82 us; float32 of 64 features, 128 sequences of 64 chunks 736 -> 505 us, 192 of 8 to 64 chunks level).
bool chunk_parallel_pays(const Shape &s)
{
    return lib.mrx_linear_attn_chunk_parallel_pays(s.B, s.T, s.H, code(s.dt)) != 0 && (std::max(s.dk, s.dv) > 32 || s.chunks() >= 10);
}

struct AttnGrads {
    Tensor dq, dk, dv, extra, dS0, dz0;   // extra: the gradient of the gate (gated: dg, delta rule: dbeta)
};

AttnGrads linear_attn_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done_, const Tensor &S_chk, const OptTensor &S_last,
                          const Tensor &dout, const OptTensor &dS_last, int fmap, bool want_dS0)
{
    const Shape s(q, k, v);
    chk(dout, "do", s.dt, v.sizes());
    chk(S_chk, "S_chk", at::kFloat, {s.B, s.H, s.chunks(), s.dv, s.dk});
    chk(S_last, "S_last", at::kFloat, s.state());
    chk(dS_last, "dS_last", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    AttnGrads r{fresh_like(q), fresh_like(k), fresh_like(v), {}, want_dS0 ? fresh(s.state(), at::kFloat, q) : Tensor(), {}};
    if (!(S_last.has_value() && S_last->defined())) {   // residuals of the chunk-parallel pair
        const Tensor ws = fresh_like(S_chk);
        check(lib.mrx_linear_attn_bwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S_chk), ptr(dout), fptr(dS_last),
                                                     ptr(r.dq), ptr(r.dk), ptr(r.dv), fptr(r.dS0), fptr(ws), s.B, s.T, s.H, s.dk, s.dv,
                                                     code(s.dt), done.dtype, fmap),
              "mrx_linear_attn_bwd_chunk_parallel");
        return r;
    }
    check(lib.mrx_linear_attn_bwd(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S_chk), fptr(S_last), ptr(dout), fptr(dS_last), ptr(r.dq),
                                  ptr(r.dk), ptr(r.dv), fptr(r.dS0), s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
          "mrx_linear_attn_bwd");
    return r;
}

struct NormAttnOut {
    Tensor o, den, S_last, z_last, S_chk, z_chk, ss;
    bool parallel;   // as in AttnOut
};

NormAttnOut linear_attn_norm_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done_, const OptTensor &S0,
                                 const OptTensor &z0, int fmap, double eps, bool save_chk, bool want_ss, bool chunk_parallel = false)
{
    const Shape s(q, k, v);
    chk(S0, "S0", at::kFloat, s.state());
    chk(z0, "z0", at::kFloat, {s.B, s.H, s.dk});
    const Done done(done_, s.B, s.T);
    NormAttnOut r;
    r.parallel = chunk_parallel && chunk_parallel_pays(s);
    r.o = fresh_like(v);
    r.den = fresh({s.B, s.H, s.T}, at::kFloat, q);
    r.S_last = fresh(s.state(), at::kFloat, q);
    r.z_last = fresh({s.B, s.H, s.dk}, at::kFloat, q);
    if (save_chk || r.parallel) {
        r.S_chk = fresh({s.B, s.H, s.chunks(), s.dv, s.dk}, at::kFloat, q);
        r.z_chk = fresh({s.B, s.H, s.chunks(), s.dk}, at::kFloat, q);
    }
    if (want_ss) r.ss = fresh({s.B, s.H, s.T}, at::kFloat, q);
    if (r.parallel)
        check(lib.mrx_linear_attn_norm_fwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S0), fptr(z0), ptr(r.o), fptr(r.den),
                                                          fptr(r.ss), fptr(r.S_last), fptr(r.z_last), fptr(r.S_chk), fptr(r.z_chk), s.B, s.T,
                                                          s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap, (float)eps),
              "mrx_linear_attn_norm_fwd_chunk_parallel");
    else
        check(lib.mrx_linear_attn_norm_fwd(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S0), fptr(z0), ptr(r.o), fptr(r.den), fptr(r.ss),
                                           fptr(r.S_last), fptr(r.z_last), fptr(r.S_chk), fptr(r.z_chk), s.B, s.T, s.H, s.dk, s.dv,
                                           code(s.dt), done.dtype, fmap, (float)eps),
              "mrx_linear_attn_norm_fwd");
    return r;
}

AttnGrads linear_attn_norm_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done_, const Tensor &S_chk,
                               const Tensor &z_chk, const Tensor &S_last, const Tensor &o, const Tensor &den, const Tensor &dout,
                               const OptTensor &dS_last, const OptTensor &dz_last, int fmap, double eps, bool want_d0, const OptTensor &d_ss,
                               bool parallel = false)
{
    const Shape s(q, k, v);
    chk(S_last, "S_last", at::kFloat, s.state());
    chk(dout, "do", s.dt, v.sizes());
    chk(o, "o", s.dt, v.sizes());
    chk(den, "den", at::kFloat, {s.B, s.H, s.T});
    chk(S_chk, "S_chk", at::kFloat, {s.B, s.H, s.chunks(), s.dv, s.dk});
    chk(z_chk, "z_chk", at::kFloat, {s.B, s.H, s.chunks(), s.dk});
    chk(dS_last, "dS_last", at::kFloat, s.state());
    chk(dz_last, "dz_last", at::kFloat, {s.B, s.H, s.dk});
    chk(d_ss, "d_ss", at::kFloat, {s.B, s.H, s.T});
    const Done done(done_, s.B, s.T);
    AttnGrads r{fresh_like(q), fresh_like(k), fresh_like(v), {}, want_d0 ? fresh(s.state(), at::kFloat, q) : Tensor(),
                want_d0 ? fresh({s.B, s.H, s.dk}, at::kFloat, q) : Tensor()};
    if (parallel) {
        const Tensor ws = fresh({s.B, s.H, s.chunks(), s.dv + 1, s.dk}, at::kFloat, q);
        check(lib.mrx_linear_attn_norm_bwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S_chk), fptr(z_chk), ptr(o), fptr(den),
                                                          ptr(dout), fptr(d_ss), fptr(dS_last), fptr(dz_last), ptr(r.dq), ptr(r.dk), ptr(r.dv),
                                                          fptr(r.dS0), fptr(r.dz0), fptr(ws), s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype,
                                                          fmap, (float)eps),
              "mrx_linear_attn_norm_bwd_chunk_parallel");
        return r;
    }
    check(lib.mrx_linear_attn_norm_bwd(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S_chk), fptr(S_last), fptr(z_chk), ptr(o), fptr(den),
                                       ptr(dout), fptr(d_ss), fptr(dS_last), fptr(dz_last), ptr(r.dq), ptr(r.dk), ptr(r.dv), fptr(r.dS0),
                                       fptr(r.dz0), s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap, (float)eps),
          "mrx_linear_attn_norm_bwd");
    return r;
}

AttnOut gated_linear_attn_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done_, const OptTensor &S0,
                              int fmap, bool save_chk, bool chunk_parallel = false)
{
    const Shape s(q, k, v);
    chk(g, "g", at::kFloat, {s.B, s.T, s.H});
    chk(S0, "S0", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    AttnOut r{fresh_like(v), fresh(s.state(), at::kFloat, q), {}, chunk_parallel && chunk_parallel_pays(s)};
    if (save_chk || r.parallel) r.S_chk = fresh({s.B, s.H, s.chunks(), s.dv, s.dk}, r.parallel ? at::kFloat : s.dt, q);
    if (r.parallel) {
        const Tensor dec = fresh({s.B, s.H, s.chunks()}, at::kFloat, q);
        check(lib.mrx_gated_linear_attn_fwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), fptr(g), done.p(), fptr(S0), ptr(r.o), fptr(r.S_last),
                                                           fptr(r.S_chk), fptr(dec), s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
              "mrx_gated_linear_attn_fwd_chunk_parallel");
        return r;
    }
    check(lib.mrx_gated_linear_attn_fwd(stream(), ptr(q), ptr(k), ptr(v), fptr(g), done.p(), fptr(S0), ptr(r.o), fptr(r.S_last), ptr(r.S_chk),
                                        s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
          "mrx_gated_linear_attn_fwd");
    return r;
}

AttnGrads gated_linear_attn_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done_, const Tensor &S_chk,
                                const Tensor &dout, const OptTensor &dS_last, int fmap, bool want_dS0, const OptTensor &S_last,
                                bool parallel = false)
{
    const Shape s(q, k, v);
    chk(g, "g", at::kFloat, {s.B, s.T, s.H});
    chk(dout, "do", s.dt, v.sizes());
    chk(S_chk, "S_chk", parallel ? at::kFloat : s.dt, {s.B, s.H, s.chunks(), s.dv, s.dk});
    chk(dS_last, "dS_last", at::kFloat, s.state());
    chk(S_last, "S_last", at::kFloat, s.state());
    TORCH_CHECK_VALUE(!ptr(dS_last) || ptr(S_last), "S_last is required with dS_last");
    const Done done(done_, s.B, s.T);
    AttnGrads r{fresh_like(q), fresh_like(k), fresh_like(v), fresh_like(g), want_dS0 ? fresh(s.state(), at::kFloat, q) : Tensor(), {}};
    if (parallel) {
        const Tensor ws = fresh({s.B * s.H * s.chunks() * (s.dv * s.dk + 1)}, at::kFloat, q);
        check(lib.mrx_gated_linear_attn_bwd_chunk_parallel(stream(), ptr(q), ptr(k), ptr(v), fptr(g), done.p(), fptr(S_chk), fptr(S_last), ptr(dout),
                                                           fptr(dS_last), ptr(r.dq), ptr(r.dk), ptr(r.dv), fptr(r.extra), fptr(r.dS0), fptr(ws),
                                                           s.B, s.T, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap),
              "mrx_gated_linear_attn_bwd_chunk_parallel");
        return r;
    }
    check(lib.mrx_gated_linear_attn_bwd(stream(), ptr(q), ptr(k), ptr(v), fptr(g), done.p(), ptr(S_chk), fptr(S_last), ptr(dout),
                                        fptr(dS_last), ptr(r.dq), ptr(r.dk), ptr(r.dv), fptr(r.extra), fptr(r.dS0), s.B, s.T, s.H, s.dk, s.dv,
                                        code(s.dt), done.dtype, fmap),
          "mrx_gated_linear_attn_bwd");
    return r;
}

// ---- delta rule
struct DeltaOut {
    Tensor o, S_last, S_chk, Tm_chk;
};

// out: an earlier call's results to write into instead of allocating (S_chk undefined there: no residuals).
// tm_scratch (only without residuals): whether the library is given a buffer for the triangular factors anyway, which lets it
// compute them chunk-parallel; unset: when it would use one (float32; bfloat16 with at most two sequences per compute unit).
DeltaOut delta_rule_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done_, const OptTensor &S0,
                        bool save_chk, const std::optional<std::array<OptTensor, 4>> &out, bool prologue, std::optional<bool> tm_scratch,
                        int factors, int resets)
{
    const Shape s(q, k, v);
    chk(beta, "beta", s.dt, {s.B, s.T, s.H});
    chk(S0, "S0", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    const int64_t C = chunk_size(s.dt, true), NC = s.chunks(true);
    DeltaOut r;
    if (out.has_value()) {
        auto take = [](const OptTensor &t) { return t.has_value() ? *t : Tensor(); };
        r = {take((*out)[0]), take((*out)[1]), take((*out)[2]), take((*out)[3])};
        chk((*out)[0], "out o", s.dt, v.sizes());
        chk((*out)[1], "out S_last", at::kFloat, s.state());
        chk((*out)[2], "out S_chk", s.dt, {s.B, s.H, NC, s.dv, s.dk});
        chk((*out)[3], "out Tm_chk", s.dt, {s.B, s.H, NC, C, C});
        TORCH_CHECK_VALUE(r.o.defined() && r.S_last.defined(), "out needs o and S_last");
    } else {
        r.o = fresh_like(v);
        r.S_last = fresh(s.state(), at::kFloat, q);
        if (save_chk) r.S_chk = fresh({s.B, s.H, NC, s.dv, s.dk}, s.dt, q);
        const bool factor_buffer =
            save_chk || (tm_scratch.has_value() ? *tm_scratch : s.dt == at::kFloat || s.B * s.H <= 2 * compute_units(q));
        if (factor_buffer) r.Tm_chk = fresh({s.B, s.H, NC, C, C}, s.dt, q);
    }
    check((prologue ? lib.mrx_deltanet_fwd : lib.mrx_delta_rule_fwd)(stream(), ptr(q), ptr(k), ptr(v), ptr(beta), done.p(), fptr(S0), ptr(r.o),
                                                                     fptr(r.S_last), ptr(r.S_chk), ptr(r.Tm_chk), s.B, s.T, s.H, s.dk, s.dv,
                                                                     code(s.dt), done.dtype, factors, resets),
          prologue ? "mrx_deltanet_fwd" : "mrx_delta_rule_fwd");
    return r;
}

AttnGrads delta_rule_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done_, const Tensor &S_chk,
                         const Tensor &Tm_chk, const Tensor &dout, const OptTensor &dS_last, bool want_dS0,
                         const std::optional<std::array<OptTensor, 5>> &out, bool prologue, int resets)
{
    const Shape s(q, k, v);
    const int64_t C = chunk_size(s.dt, true), NC = s.chunks(true);
    chk(Tm_chk, "Tm_chk", s.dt, {s.B, s.H, NC, C, C});
    chk(beta, "beta", s.dt, {s.B, s.T, s.H});
    chk(dout, "do", s.dt, v.sizes());
    chk(S_chk, "S_chk", s.dt, {s.B, s.H, NC, s.dv, s.dk});
    chk(dS_last, "dS_last", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    AttnGrads r;
    if (out.has_value()) {
        const auto &o = *out;
        for (int i = 0; i < 4; ++i) TORCH_CHECK_VALUE(ptr(o[i]), "out needs dq, dk, dv and dbeta");
        chk(o[0], "out dq", s.dt, q.sizes());
        chk(o[1], "out dk", s.dt, k.sizes());
        chk(o[2], "out dv", s.dt, v.sizes());
        chk(o[3], "out dbeta", s.dt, beta.sizes());
        chk(o[4], "out dS0", at::kFloat, s.state());
        r = {*o[0], *o[1], *o[2], *o[3], o[4].has_value() ? *o[4] : Tensor(), {}};
    } else {
        r = {fresh_like(q), fresh_like(k), fresh_like(v), fresh_like(beta), want_dS0 ? fresh(s.state(), at::kFloat, q) : Tensor(), {}};
    }
    check((prologue ? lib.mrx_deltanet_bwd : lib.mrx_delta_rule_bwd)(stream(), ptr(q), ptr(k), ptr(v), ptr(beta), done.p(), ptr(S_chk),
                                                                     ptr(Tm_chk), ptr(dout), fptr(dS_last), ptr(r.dq), ptr(r.dk), ptr(r.dv),
                                                                     ptr(r.extra), fptr(r.dS0), s.B, s.T, s.H, s.dk, s.dv, code(s.dt),
                                                                     done.dtype, resets),
          prologue ? "mrx_deltanet_bwd" : "mrx_delta_rule_bwd");
    return r;
}

std::array<Tensor, 2> delta_rule_fwd_noalloc(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done_,
                                             const OptTensor &S0, const OptTensor &o, const OptTensor &S_last)
{
    const Shape s(q, k, v);
    chk(beta, "beta", s.dt, {s.B, s.T, s.H});
    chk(S0, "S0", at::kFloat, s.state());
    const Done done(done_, s.B, s.T);
    chk(o, "out o", s.dt, v.sizes());
    chk(S_last, "out S_last", at::kFloat, s.state());
    std::array<Tensor, 2> r{o.has_value() ? *o : fresh_like(v), S_last.has_value() ? *S_last : fresh(s.state(), at::kFloat, q)};
    check(lib.mrx_delta_rule_fwd_noalloc(stream(), ptr(q), ptr(k), ptr(v), ptr(beta), done.p(), fptr(S0), ptr(r[0]), fptr(r[1]), s.B, s.T, s.H,
                                         s.dk, s.dv, code(s.dt), done.dtype),
          "mrx_delta_rule_fwd_noalloc");
    return r;
}

// ---- single time steps: q, k, v (B,H,d), done (B)
struct StepShape {
    int64_t B, H, dk, dv;
    ScalarType dt;
    StepShape(const Tensor &q, const Tensor &k, const Tensor &v)
    {
        TORCH_CHECK_VALUE(q.dim() == 3 && v.dim() == 3, "q must be (B,H,d), got ", q.sizes());
        B = q.size(0), H = q.size(1), dk = q.size(2), dv = v.size(2);
        dt = q.scalar_type();
        TORCH_CHECK_VALUE(dt == at::kFloat || dt == at::kBFloat16, "unsupported dtype ", dt);
        chk(q, "q");
        chk(k, "k", dt, {B, H, dk});
        chk(v, "v", dt, {B, H, dv});
    }
    std::array<int64_t, 4> state() const { return {B, H, dv, dk}; }
    Tensor next(const OptTensor &S, bool inplace, const Tensor &like) const
    {
        return inplace && S.has_value() ? *S : fresh(state(), at::kFloat, like);
    }
};

struct StepOut {
    Tensor o, S, z;
};

StepOut linear_attn_step(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done_, const OptTensor &S, const OptTensor &z,
                         int fmap, bool normalise, double eps, bool inplace)
{
    const StepShape s(q, k, v);
    chk(S, "S", at::kFloat, s.state());
    chk(z, "z", at::kFloat, {s.B, s.H, s.dk});
    const Done done(done_.reshape({s.B, 1}), s.B, 1);
    StepOut r{fresh_like(v), s.next(S, inplace, q), {}};
    if (normalise) r.z = inplace && z.has_value() ? *z : fresh({s.B, s.H, s.dk}, at::kFloat, q);
    check(lib.mrx_linear_attn_step(stream(), ptr(q), ptr(k), ptr(v), done.p(), fptr(S), normalise ? fptr(z) : nullptr, ptr(r.o), fptr(r.S),
                                   fptr(r.z), s.B, s.H, s.dk, s.dv, code(s.dt), done.dtype, fmap, (float)eps),
          "mrx_linear_attn_step");
    return r;
}

StepOut gated_linear_attn_step(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done_, const OptTensor &S,
                               int fmap, bool inplace)
{
    const StepShape s(q, k, v);
    chk(g, "g", at::kFloat, {s.B, s.H});
    chk(S, "S", at::kFloat, s.state());
    const Done done(done_.reshape({s.B, 1}), s.B, 1);
    StepOut r{fresh_like(v), s.next(S, inplace, q), {}};
    check(lib.mrx_gated_linear_attn_step(stream(), ptr(q), ptr(k), ptr(v), fptr(g), done.p(), fptr(S), ptr(r.o), fptr(r.S), s.B, s.H, s.dk,
                                         s.dv, code(s.dt), done.dtype, fmap),
          "mrx_gated_linear_attn_step");
    return r;
}

// prologue: k and beta are the raw projections of the DeltaNet cell
StepOut delta_rule_step(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done_, const OptTensor &S,
                        bool inplace, bool prologue)
{
    const StepShape s(q, k, v);
    chk(beta, "beta", s.dt, {s.B, s.H});
    chk(S, "S", at::kFloat, s.state());
    const Done done(done_.reshape({s.B, 1}), s.B, 1);
    StepOut r{fresh_like(v), s.next(S, inplace, q), {}};
    check((prologue ? lib.mrx_deltanet_step : lib.mrx_delta_rule_step)(stream(), ptr(q), ptr(k), ptr(v), ptr(beta), done.p(), fptr(S), ptr(r.o),
                                                                       fptr(r.S), s.B, s.H, s.dk, s.dv, code(s.dt), done.dtype),
          prologue ? "mrx_deltanet_step" : "mrx_delta_rule_step");
    return r;
}

// ---- acting: dense layers on few rows, the MinGRU cell's step
Tensor norm_param(const OptTensor &t) { return t.has_value() ? dense16(t->to(at::kFloat)) : Tensor(); }

// The operators know no forward mode: an input with a tangent is refused, as an autograd function without a jvp refuses it (also where
// gradients are switched off: no_grad leaves tangents on).
void refuse_tangent(const Tensor &t)
{
    TORCH_CHECK_NOT_IMPLEMENTED(!t.defined() || !t._fw_grad(0).defined(), "memorax_amd operators have no forward-mode derivative");
}
void refuse_tangent(const OptTensor &t)
{
    if (t.has_value()) refuse_tangent(*t);
}
// Nor do they know functorch's transforms: a history set on the wrapper of a batched tensor is lost when vmap unwraps it.
bool transformed(const Tensor &t)
{
    return t.defined() && t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched}));
}
bool transformed(const OptTensor &t) { return t.has_value() && transformed(*t); }
void refuse(const Tensor &t)
{
    refuse_tangent(t);
    TORCH_CHECK(!transformed(t), "memorax_amd operators do not run under functorch's transforms (vmap, grad, vjp, ...)");
}
void refuse(const OptTensor &t)
{
    if (t.has_value()) refuse(*t);
}
// A traced graph (torch.jit.trace) would hold a kernel's results as constants: what is a composition of array operations is traced as
// that, the rest refused.
bool tracing() { return torch::jit::tracer::isTracing(); }
void refuse_tracing() { TORCH_CHECK(!tracing(), "memorax_amd operators cannot be traced by torch.jit.trace"); }
void refuse(const std::vector<Tensor> &ts)
{
    for (const Tensor &t : ts) refuse(t);
}
void refuse(const std::vector<OptTensor> &ts)
{
    for (const OptTensor &t : ts) refuse(t);
}
template <typename... Ts> void refuse(const Ts &...ts) requires(sizeof...(Ts) > 1)
{
    refuse_tracing();
    (refuse(ts), ...);
}

// What an acting call reads and writes lies on the GPU of its rows: a layer left on the host, or on another GPU, is an error and no address.
void chk_beside(const Tensor &x, const Tensor &t)
{
    if (!t.defined()) return;
    TORCH_CHECK_VALUE(t.is_cuda(), "parameters and carries must live on the GPU (memorax_amd has no CPU path)");
    TORCH_CHECK_VALUE(t.device() == x.device(), "parameters and carries must live on the GPU of the rows, ", x.device(), ", got ", t.device());
}
void chk_beside(const Tensor &x, const OptTensor &t)
{
    if (t.has_value()) chk_beside(x, *t);
}
template <typename T> void chk_beside(const Tensor &x, const std::vector<T> &ts)
{
    for (const T &t : ts) chk_beside(x, t);
}
template <typename... Ts> void chk_beside(const Tensor &x, const Ts &...ts) requires(sizeof...(Ts) > 1)
{
    TORCH_CHECK_VALUE(x.is_cuda(), "x must live on the GPU (memorax_amd has no CPU path)");
    (chk_beside(x, ts), ...);
}

// norm: 0 none, 1 RMS, 2 layer norm.  The results keep x's leading axes; residual (float32, x's leading axes): added to the one
// layer's result.
std::vector<Tensor> row_dense(const Tensor &x_, int norm, const OptTensor &scale_, const OptTensor &nbias_, double eps, bool round_norm,
                              std::vector<Tensor> weights, std::vector<OptTensor> biases, ScalarType product, ScalarType out_dtype,
                              const OptTensor &residual_, const OptTensor &weight2_ = std::nullopt, const OptTensor &skip_ = std::nullopt,
                              Tensor *skip_out = nullptr)
{
    refuse(x_, scale_, nbias_, weights, biases, residual_, weight2_, skip_);
    chk_beside(x_, scale_, nbias_, weights, biases, residual_, weight2_, skip_);
    const Tensor x = dense16(x_), scale = norm_param(scale_), nbias = norm_param(nbias_), weight2 = dense16(weight2_), skip = dense16(skip_),
                 residual = residual_.has_value() ? residual_->contiguous() : Tensor();
    for (Tensor &w : weights) w = dense16(w);
    for (OptTensor &b : biases)
        if (b.has_value()) b = b->contiguous();
    TORCH_CHECK_VALUE(x.dim() >= 2 && !weights.empty() && weights.size() <= MRX_ROW_DENSE_LAYERS && biases.size() == weights.size(),
                      "row_dense takes rows and 1 to ", MRX_ROW_DENSE_LAYERS, " layers");
    const int64_t K = x.size(-1), rows = x.numel() / K;
    chk(x, "x");
    if (scale.defined()) chk(scale, "scale", at::kFloat, {K});
    if (nbias.defined()) chk(nbias, "bias of the norm", at::kFloat, {K});
    const auto wd = weights[0].scalar_type();
    auto bd = at::kFloat;
    std::array<const void *, MRX_ROW_DENSE_LAYERS> w{}, b{};
    std::array<void *, MRX_ROW_DENSE_LAYERS> y{};
    std::array<int64_t, MRX_ROW_DENSE_LAYERS> n{};
    std::vector<Tensor> out;
    out.reserve(weights.size());
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    bool first_bias = true;
    for (size_t l = 0; l < weights.size(); ++l) {
        n[l] = weights[l].size(0);
        chk(weights[l], "weight", wd, {n[l], weight2.defined() ? K - weight2.size(1) : K});
        if (biases[l].has_value()) {
            if (std::exchange(first_bias, false)) bd = biases[l]->scalar_type();
            chk(*biases[l], "bias", bd, {n[l]});
        }
        shape.back() = n[l];
        out.push_back(fresh(shape, out_dtype, x));
        w[l] = ptr(weights[l]), b[l] = ptr(biases[l]), y[l] = ptr(out[l]);
    }
    if (residual.defined()) chk(residual, "residual", at::kFloat, out[0].sizes());
    if (weight2.defined()) chk(weight2, "weight2", wd, {n[0], weight2.size(1)});
    if (skip.defined()) chk(skip, "skip", at::kFloat, {K});
    if (skip.defined()) *skip_out = fresh(x.sizes(), at::kFloat, x);
    check(lib.mrx_row_dense(stream(), ptr(x), fptr(scale), fptr(nbias), norm, round_norm, w.data(), b.data(), y.data(), n.data(),
                            (int)weights.size(), fptr(residual), rows, K, code(x.scalar_type()), code(wd), code(bd), code(out_dtype),
                            code(product), (float)eps, ptr(weight2), weight2.defined() ? weights[0].size(1) : 0, fptr(skip),
                            skip_out ? fptr(*skip_out) : nullptr),
          "mrx_row_dense");
    return out;
}

// A pre-norm residual block around an LRU cell, one acting step: x (B,1,F) float32, the carry's leaves (B,1,N) complex64
// -> y, h, P.  params: nu_log, theta_log, gamma_log, B_real, B_imag, C_real, C_imag, D.
std::tuple<Tensor, Tensor, Tensor> lru_act(const Tensor &x, int norm, const OptTensor &scale, const OptTensor &nbias, double eps,
                                           std::vector<Tensor> params, const Tensor &done_, const Tensor &h_, const Tensor &P_)
{
    TORCH_CHECK_VALUE(x.dim() == 3 && x.size(1) == 1 && params.size() == 8, "lru_act takes one time step");
    refuse(x, scale, nbias, params, done_, h_, P_);
    chk_beside(x, scale, nbias, params, done_, h_, P_);
    const int64_t B = x.size(0), N = params[0].size(0);
    for (Tensor &t : params) t = dense16(t);
    for (int i = 0; i < 3; ++i) chk(params[i], "parameter", at::kFloat, {N});
    const Tensor h = h_.contiguous(), P = P_.contiguous();
    chk(h, "h", at::kComplexFloat, {B, 1, N});
    chk(P, "P", at::kComplexFloat, {B, 1, N});
    const Done done(done_, B, 1);
    Tensor skip;
    const auto u = row_dense(x, norm, scale, nbias, eps, false, {params[3], params[4]}, {std::nullopt, std::nullopt}, at::kFloat, at::kFloat,
                             std::nullopt, std::nullopt, params[7], &skip);
    const Tensor hn = fresh_like(h), Pn = fresh_like(P), row = fresh({B, 1, 2 * N}, at::kFloat, x);
    check(lib.mrx_lru_step(stream(), fptr(u[0]), fptr(u[1]), fptr(params[0]), fptr(params[1]), fptr(params[2]), done.p(), ptr(h), ptr(P), ptr(hn),
                           ptr(Pn), fptr(row), B, N, done.dtype),
          "mrx_lru_step");
    return {row_dense(row, 0, std::nullopt, std::nullopt, 0.0, false, {params[5]}, {std::nullopt}, at::kFloat, at::kFloat, skip, params[6])[0], hn, Pn};
}

// The same around an mLSTM cell; params: up, conv weight and bias, query, key, value, i_gate and f_gate (weight, bias), norm_weight,
// learnable_skip, output projection; the carry's leaves C (B,1,H,D,D), log_f, n (B,1,H,D,1), m.
std::vector<Tensor> mlstm_act(const Tensor &x, int norm, const OptTensor &scale, const OptTensor &nbias, double eps, std::vector<Tensor> p,
                              const Tensor &done_, const std::vector<Tensor> &carry, double g_floor)
{
    TORCH_CHECK_VALUE(x.dim() == 3 && x.size(1) == 1 && p.size() == 13 && carry.size() == 4, "mlstm_act takes one time step");
    refuse(x, scale, nbias, p, done_, carry);
    chk_beside(x, scale, nbias, p, done_, carry);
    const int64_t B = x.size(0), H = p[3].size(0), D = p[3].size(1), W = H * D, K = p[1].size(2);
    for (Tensor &t : p) t = dense16(t);
    chk(p[1], "conv weight", at::kFloat, {W, 1, K});
    chk(p[2], "conv bias", at::kFloat, {W});
    for (int i = 3; i < 6; ++i) chk(p[i], "block-diagonal map", at::kFloat, {H, D, D});
    for (int i : {6, 8}) chk(p[i], "gate weight", at::kFloat, {H, 3 * W}), chk(p[i + 1], "gate bias", at::kFloat, {H});
    chk(p[10], "norm_weight", at::kFloat, {H, D});
    chk(p[11], "learnable_skip", at::kFloat, {W});
    const Tensor C = dense16(carry[0]), lf = carry[1].contiguous(), n = carry[2].contiguous(), m = carry[3].contiguous();
    chk(C, "C", at::kFloat, {B, 1, H, D, D});
    chk(n, "n", at::kFloat, {B, 1, H, D, 1});
    chk(lf, "log_f", at::kFloat, {B, 1, H, 1, 1});
    chk(m, "m", at::kFloat, {B, 1, H, 1, 1});
    const Done done(done_, B, 1);
    const auto up = row_dense(x, norm, scale, nbias, eps, false, {p[0]}, {std::nullopt}, at::kFloat, at::kFloat, std::nullopt)[0];
    const Tensor Co = fresh_like(C), lfo = fresh_like(lf), no = fresh_like(n), mo = fresh_like(m), y = fresh({B, 1, W}, at::kFloat, x);
    TORCH_CHECK_VALUE(up.size(2) == 2 * W, "up projection");
    check(lib.mrx_mlstm_step(stream(), fptr(up), fptr(p[1]), fptr(p[2]), fptr(p[3]), fptr(p[4]), fptr(p[5]), fptr(p[6]), fptr(p[7]), fptr(p[8]),
                             fptr(p[9]), fptr(p[10]), fptr(p[11]), done.p(), fptr(C), fptr(lf), fptr(n), fptr(m), fptr(Co), fptr(lfo), fptr(no),
                             fptr(mo), fptr(y), B, H, D, K, done.dtype, (float)g_floor),
          "mrx_mlstm_step");
    return {row_dense(y, 0, std::nullopt, std::nullopt, 0.0, false, {p[12]}, {std::nullopt}, at::kFloat, at::kFloat, x)[0], Co, lfo, no, mo};
}

// z, h~, gate (B,1,D), done (B,1), the carry's leaves (B,1,D) float32 -> y, log_state, log_decay
std::tuple<Tensor, Tensor, Tensor> mingru_step(const Tensor &z, const Tensor &x, const OptTensor &gate, const Tensor &done_,
                                               const Tensor &log_state, const Tensor &log_decay, bool in_place)
{
    TORCH_CHECK_VALUE(z.dim() == 3 && z.size(1) == 1, "mingru_step takes one time step");
    refuse(z, x, gate, done_, log_state, log_decay);
    chk_beside(z, x, gate, done_, log_state, log_decay);
    const int64_t B = z.size(0), D = z.size(2);
    const auto dt = z.scalar_type();
    chk_scan_dtype(dt, false, "mingru_step");
    chk(z, "z");
    chk(x, "h_tilde", dt, z.sizes());
    chk(gate, "gate", dt, z.sizes());
    chk(log_state, "log_state", at::kFloat, z.sizes());
    chk(log_decay, "log_decay", at::kFloat, z.sizes());
    const Done done(done_, B, 1);
    const Tensor y = fresh_like(z), ls = in_place ? log_state : fresh_like(log_state), ld = in_place ? log_decay : fresh_like(log_decay);
    check(lib.mrx_mingru_step(stream(), ptr(z), ptr(x), ptr(gate), done.p(), fptr(log_state), fptr(log_decay), ptr(y), fptr(ls), fptr(ld), B, D,
                              code(dt), done.dtype),
          "mrx_mingru_step");
    return {y, ls, ld};
}

// Pre-norm residual blocks, one acting step each: x (B,1,K) float32 -> x + block(norm(x)) and what the cell carries on.  One call from Python
// instead of one for each launch, with a dozen checks and views between them.
// A gated recurrence: weights and biases of z, h~, gate and the closing layer, the carry's leaves (B,1,N) -> y, z, log_state, log_decay
std::tuple<Tensor, Tensor, Tensor, Tensor> gated_act(const Tensor &x, int norm, const OptTensor &scale, const OptTensor &nbias, double eps,
                                                     const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, ScalarType product,
                                                     const Tensor &done_, const Tensor &log_state, const Tensor &log_decay, bool in_place)
{
    TORCH_CHECK_VALUE(x.dim() == 3 && x.size(1) == 1 && weights.size() == 4 && biases.size() == 4, "gated_act takes one time step");
    refuse(x, scale, nbias, weights, biases, done_, log_state, log_decay);
    chk_beside(x, scale, nbias, weights, biases, done_, log_state, log_decay);
    const int64_t B = x.size(0), K = x.size(2), N = weights[0].size(0);
    auto fits = [](const Tensor &t) { return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    const auto wd = weights[0].scalar_type();
    bool whole = K % 8 == 0 && K <= 512 && N % 4 == 0 && B > 0 && fits(x) && fits(log_state) && fits(log_decay) &&
                 (product == at::kBFloat16 ? wd == at::kFloat || wd == at::kBFloat16 : wd == at::kFloat);
    for (int l = 0; l < 3; ++l)
        whole = whole && !biases[l].has_value() && weights[l].scalar_type() == wd && fits(weights[l]) && weights[l].sizes() == IntArrayRef({N, K});
    Tensor z, y, ls, ld;
    if (whole) {
        const Tensor sc = norm_param(scale), nb = norm_param(nbias);
        chk(x, "x", at::kFloat);
        if (sc.defined()) chk(sc, "scale", at::kFloat, {K});
        if (nb.defined()) chk(nb, "bias of the norm", at::kFloat, {K});
        chk(log_state, "log_state", at::kFloat, {B, 1, N});
        chk(log_decay, "log_decay", at::kFloat, {B, 1, N});
        const Done done(done_, B, 1);
        z = fresh({B, 1, N}, product, x), y = fresh({B, 1, N}, product, x);
        ls = in_place ? log_state : fresh_like(log_state), ld = in_place ? log_decay : fresh_like(log_decay);
        check(lib.mrx_gated_recurrence_act(stream(), fptr(x), fptr(sc), fptr(nb), norm, ptr(weights[0]), ptr(weights[1]), ptr(weights[2]), done.p(),
                                           fptr(log_state), fptr(log_decay), ptr(z), ptr(y), fptr(ls), fptr(ld), B, K, N, code(wd), code(product),
                                           done.dtype, (float)eps),
              "mrx_gated_recurrence_act");
    } else {
        auto u = row_dense(x, norm, scale, nbias, eps, false, {weights[0], weights[1], weights[2]}, {biases[0], biases[1], biases[2]}, product, product,
                           std::nullopt);
        z = u[0];
        std::tie(y, ls, ld) = mingru_step(z, u[1], u[2], done_, log_state, log_decay, in_place);
    }
    return {row_dense(y, 0, std::nullopt, std::nullopt, 0.0, false, {weights[3]}, {biases[3]}, product, at::kFloat, x)[0], z, ls, ld};
}

// A matrix state: weights and biases of q, k, v (, beta: the delta rule with its prologue; without it linear attention with the elu + 1 map and
// its normaliser z (B,1,H,D)) and of the closing layer, behind the RMS norm of the read-out; projections handed on in `dtype`;
// S (B,1,H,D,D) -> y, S, z
std::tuple<Tensor, Tensor, OptTensor> state_act(const Tensor &x, int norm, const OptTensor &scale, const OptTensor &nbias, double eps,
                                                std::vector<Tensor> weights, std::vector<OptTensor> biases, const Tensor &out_scale, double out_eps,
                                                ScalarType product, ScalarType dtype, const Tensor &done, const Tensor &S, const OptTensor &z, double den_eps,
                                                bool in_place)
{
    TORCH_CHECK_VALUE(x.dim() == 3 && x.size(1) == 1 && weights.size() == (z.has_value() ? 4u : 5u) && biases.size() == weights.size() && S.dim() == 5,
                      "state_act takes one time step");
    refuse(x, scale, nbias, weights, biases, out_scale, done, S, z);
    chk_beside(x, scale, nbias, weights, biases, out_scale, done, S, z);
    const int64_t B = x.size(0), H = S.size(2), D = S.size(3);
    const Tensor out_w = weights.back();
    const OptTensor out_b = biases.back();
    weights.pop_back(), biases.pop_back();
    auto u = row_dense(x, norm, scale, nbias, eps, false, weights, biases, product, dtype, std::nullopt);
    for (int i = 0; i < 3; ++i) u[i] = u[i].view({B, H, D});
    auto carried = [](const Tensor &t) { return t.select(1, 0).to(at::kFloat).contiguous(); };
    const bool own = in_place && S.scalar_type() == at::kFloat && S.is_contiguous() && (!z.has_value() || (z->scalar_type() == at::kFloat && z->is_contiguous()));
    const Tensor S_ = carried(S);
    StepOut r = z.has_value() ? linear_attn_step(u[0], u[1], u[2], done, S_, carried(*z), MRX_FMAP_ELU1, true, den_eps, own)
                              : delta_rule_step(u[0], u[1], u[2], u[3].view({B, H}), done, S_, own, true);
    const Tensor y = row_dense(r.o.view({B, 1, H * D}), 1, out_scale, std::nullopt, out_eps, dtype == at::kBFloat16, {out_w}, {out_b}, product, at::kFloat, x)[0];
    return {y, own ? S : r.S.unsqueeze(1), own ? z : z.has_value() ? OptTensor(r.z.unsqueeze(1)) : std::nullopt};
}

// Copies x and done into the buffers of a recorded step by one launch; false, and nothing done, where they are not float32 rows and flags as
// those buffers hold them (another shape, type, layout or device, gradients recorded): what a copy makes of these is the caller's then.
bool place_inputs(const Tensor &x, const Tensor &x_to, const Tensor &done, const Tensor &done_to)
{
    auto fits = [](const Tensor &t, const Tensor &to) {
        return t.is_cuda() && t.device() == to.device() && t.get_device() == c10::hip::getCurrentHIPStream().device_index() && t.sizes() == to.sizes() &&
               t.is_contiguous() && t.has_storage() && !t.is_neg() && t.numel() > 0 && !t.key_set().has(c10::DispatchKey::Python) && !transformed(t) &&
               !t._fw_grad(0).defined() && !(at::GradMode::is_enabled() && t.requires_grad());
    };
    if (tracing() || !fits(x, x_to) || !fits(done, done_to)) return false;
    const bool flags = done.scalar_type() == at::kBool || done.scalar_type() == at::kFloat;
    if (x.scalar_type() != at::kFloat || x_to.scalar_type() != at::kFloat || !flags || done_to.scalar_type() != at::kBool) return false;
    if ((reinterpret_cast<uintptr_t>(x.data_ptr()) | reinterpret_cast<uintptr_t>(x_to.data_ptr())) % 16) return false;
    check(lib.mrx_place_inputs(stream(), fptr(x), fptr(x_to), x.numel(), ptr(done), ptr(done_to), done.numel(),
                               done.scalar_type() == at::kFloat ? MRX_DONE_F32 : MRX_DONE_U8),
          "mrx_place_inputs");
    return true;
}

// ------------------------------------------------------------------------------------------------ autograd nodes
bool differentiable(const Tensor &t) { return t.defined() && t.requires_grad(); }
bool differentiable(const OptTensor &t) { return t.has_value() && differentiable(*t); }

template <typename... Ts> bool need_grad(const Ts &...ts)
{
    refuse_tracing();
    (refuse(ts), ...);
    return at::GradMode::is_enabled() && (differentiable(ts) || ...);
}

// Gradients that say so when they are differentiated again, instead of passing for constants.
variable_list refuse_second(variable_list &&grads)
{
    variable_list defined;
    for (Tensor &g : grads)
        if (g.defined()) defined.push_back(g.detach().set_requires_grad(true));
    const auto error = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that is differentiable once", (int64_t)defined.size());
    defined = (*error)(std::move(defined));
    size_t i = 0;
    for (Tensor &g : grads)
        if (g.defined()) g = defined[i++];
    return std::move(grads);
}

// One node type for every operator: Op holds what is no tensor of the graph (flags, scalars, the reset flags) and
//     static constexpr int SAVED          how many tensors the backward reads
//     static const char *name()
//     static constexpr bool ONCE          (where it is declared) differentiating the gradients again is an error
//     variable_list backward(node, saved, grads)
template <class Op> struct OpNode final : torch::autograd::Node {
    Op op;
    std::array<SavedVariable, Op::SAVED> saved;
    std::array<bool, Op::SAVED> output{};

    void keep(int i, const Tensor &t, bool is_output = false)
    {
        saved[i] = SavedVariable(t, is_output);
        output[i] = is_output;
    }
    variable_list apply(variable_list &&grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        std::array<Tensor, Op::SAVED> s;
        for (int i = 0; i < Op::SAVED; ++i) s[i] = saved[i].unpack(output[i] ? shared_from_this() : nullptr);
        variable_list out;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            out = op.backward(*this, s, grads);
        }
        if constexpr (requires { Op::ONCE; })
            if (at::GradMode::is_enabled() && std::any_of(grads.begin(), grads.end(), [](const Tensor &g) { return differentiable(g); }))
                return refuse_second(std::move(out));
        return out;
    }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto &s : saved) s.reset_data();
        if constexpr (requires(Op & o) { o.release(); }) op.release();
    }
    std::string name() const override { return Op::name(); }
    bool wants(size_t i) const { return task_should_compute_output(i); }
};

template <class Op, typename... Ts> std::shared_ptr<OpNode<Op>> record(Op &&op, const Ts &...inputs)
{
    auto node = std::shared_ptr<OpNode<Op>>(new OpNode<Op>(), torch::autograd::deleteNode);
    node->op = std::move(op);
    node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
    return node;
}


Tensor unwrap(const OptTensor &t) { return t.has_value() ? *t : Tensor(); }
OptTensor some(const Tensor &t) { return t.defined() ? OptTensor(t) : std::nullopt; }
// contiguous and in the given type; the tensor itself where it is that already
Tensor as(const Tensor &t, ScalarType dt) { return t.defined() ? t.to(dt).contiguous() : t; }
Tensor grad_or_zeros(const Tensor &g, const Tensor &like) { return g.defined() ? g.contiguous() : at::zeros_like(like); }
Tensor unless(bool skip, const Tensor &t) { return skip ? Tensor() : t; }

// The sum over the rows of a (B,D) float32 or complex64 array: one launch of the library's column sum up to 512 rows (64 x 184 4.1 and 1.9 us, complex64
// 192 x 184 5.6 and 2.1, 512 x 256 8.4 and 2.8).  Beyond, its chains of sums grow longer than the array library's: 2048 x 64 errs by 1.4e-7
// and 1.1e-7 against float64, 512 x 64 by 0.9e-7 and 1.0e-7.
constexpr int64_t SUM_ROWS = 512;
Tensor sum_rows(const Tensor &x)
{
    const bool complex = x.scalar_type() == at::kComplexFloat;
    if ((!complex && x.scalar_type() != at::kFloat) || x.numel() == 0 || x.size(0) > SUM_ROWS) return x.sum(0);
    const Tensor out = fresh({x.size(1)}, x.scalar_type(), x);
    check(lib.mrx_column_sum(stream(), static_cast<const float *>(ptr(x)), static_cast<float *>(ptr(out)), x.size(0), x.size(1) * (complex ? 2 : 1)),
          "mrx_column_sum");
    return out;
}

struct LinearScanOp {
    static constexpr int SAVED = 3;   // a, h, h0
    static const char *name() { return "MemoraxLinearScanBackward"; }
    Tensor done;
    variable_list backward(OpNode<LinearScanOp> &node, std::array<Tensor, 3> &s, variable_list &grads)
    {
        const Tensor &a = s[0], &h = s[1];
        const bool ti = a.dim() == 1;   // a broadcast coefficient: the kernel sums its gradient over time, the rest is (B,D)
        auto r = scan_bwd(a, h, done, some(s[2]), grad_or_zeros(grads[0], h), some(as(grads[1], s[2].defined() ? s[2].scalar_type() : carry(h))),
                          ti);
        if (ti && node.wants(0)) r.da = sum_rows(r.da).to(a.scalar_type());
        return {unless(!node.wants(0), r.da), unless(!node.wants(1), r.db), unless(!node.wants(2), r.dh0)};
    }
    static ScalarType carry(const Tensor &h) { return h.scalar_type() == at::kBFloat16 ? at::kFloat : h.scalar_type(); }
};

std::tuple<Tensor, Tensor, Tensor> linear_scan(const Tensor &a, const Tensor &b, const Tensor &done, const OptTensor &h0, const OptTensor &P0)
{
    refuse(done, P0);
    const bool need = need_grad(a, b, h0);
    Tensor a_, h0_;
    ScanOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        auto carried = [&](const OptTensor &t) {   // bfloat16 arrays: float32 carries
            return !t.has_value() ? Tensor() : b.scalar_type() == at::kBFloat16 ? as(*t, at::kFloat) : t->contiguous();
        };
        a_ = a.contiguous();
        h0_ = carried(h0);
        r = scan_fwd(a_, b.contiguous(), done, some(h0_), some(carried(P0)), true);
    }
    if (need) {
        auto node = record(LinearScanOp{done}, a, b, unwrap(h0));
        torch::autograd::set_history(r.h, node);
        torch::autograd::set_history(r.h_last, node);
        node->keep(0, a_);
        node->keep(1, r.h, true);
        node->keep(2, h0_);
    }
    return {r.h, r.h_last, r.P_last};
}

struct MinGruOp {
    static constexpr int SAVED = 4;   // z, h~, h, h0
    static const char *name() { return "MemoraxMinGruScanBackward"; }
    Tensor done;
    variable_list backward(OpNode<MinGruOp> &node, std::array<Tensor, 4> &s, variable_list &grads)
    {
        auto r = mingru_bwd(s[0], s[1], s[2], done, some(s[3]), grad_or_zeros(grads[0], s[2]), some(as(grads[1], at::kFloat)));
        return {unless(!node.wants(0), r.da), unless(!node.wants(1), r.db), unless(!node.wants(2), r.dh0)};
    }
};

std::tuple<Tensor, Tensor, Tensor> mingru_scan(const Tensor &z, const Tensor &x, const Tensor &done, const OptTensor &h0, const OptTensor &P0)
{
    refuse(done, P0);
    const bool need = need_grad(z, x, h0);
    Tensor z_, x_, h0_;
    ScanOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        z_ = z.contiguous();
        x_ = as(x, z.scalar_type());
        h0_ = as(unwrap(h0), at::kFloat);   // the carries are float32 whatever the arrays are
        r = mingru_fwd(z_, x_, done, some(h0_), some(as(unwrap(P0), at::kFloat)), true);
    }
    if (need) {
        auto node = record(MinGruOp{done}, z, x, unwrap(h0));
        torch::autograd::set_history(r.h, node);
        torch::autograd::set_history(r.h_last, node);
        node->keep(0, z_);
        node->keep(1, x_);
        node->keep(2, r.h, true);
        node->keep(3, h0_);
    }
    return {r.h, r.h_last, r.P_last};
}

struct LinearAttentionOp {
    static constexpr int SAVED = 5;   // q, k, v, S_chk, S_last (undefined: the chunk-parallel pair ran)
    static const char *name() { return "MemoraxLinearAttentionBackward"; }
    Tensor done;
    int fmap;
    bool parallel;
    variable_list backward(OpNode<LinearAttentionOp> &node, std::array<Tensor, 5> &s, variable_list &grads)
    {
        auto r = linear_attn_bwd(s[0], s[1], s[2], done, s[3], parallel ? std::nullopt : some(s[4]), grad_or_zeros(grads[0], s[2]),
                                 some(as(grads[1], at::kFloat)), fmap, node.wants(3));
        return {r.dq, r.dk, r.dv, r.dS0};
    }
};

// Acting (one time step, no gradients: memoroid.py:93-109 with T = 1) goes to the single-step kernels; in_place lets them
// update the carried state where it lies, which they do only on the caller's own array (a converted copy is a new one already).
std::tuple<Tensor, Tensor> linear_attention(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const OptTensor &S0, int fmap,
                                            bool in_place)
{
    refuse(done);
    const bool need = need_grad(q, k, v, S0);
    Tensor q_, k_, v_, S0_;
    AttnOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        q_ = q.contiguous(), k_ = k.contiguous(), v_ = v.contiguous();
        S0_ = as(unwrap(S0), at::kFloat);
        if (q_.size(1) == 1 && !need) {
            auto st = linear_attn_step(q_.select(1, 0), k_.select(1, 0), v_.select(1, 0), done.select(1, 0), some(S0_), std::nullopt, fmap, false,
                                       1e-6, in_place && S0.has_value() && S0_.is_same(*S0));
            return {st.o.unsqueeze(1), st.S};
        }
        r = linear_attn_fwd(q_, k_, v_, done, some(S0_), fmap, need, std::nullopt);
    }
    if (need) {
        auto node = record(LinearAttentionOp{done, fmap, r.parallel}, q, k, v, unwrap(S0));
        torch::autograd::set_history(r.o, node);
        torch::autograd::set_history(r.S_last, node);
        node->keep(0, q_);
        node->keep(1, k_);
        node->keep(2, v_);
        node->keep(3, r.S_chk);
        if (!r.parallel) node->keep(4, r.S_last, true);
    }
    return {r.o, r.S_last};
}

struct NormalisedOp {
    static constexpr int SAVED = 8;   // q, k, v, o, den, S_chk, z_chk, S_last
    static const char *name() { return "MemoraxNormalisedLinearAttentionBackward"; }
    Tensor done;
    int fmap;
    double eps;
    bool has_ss, parallel;
    variable_list backward(OpNode<NormalisedOp> &node, std::array<Tensor, 8> &s, variable_list &grads)
    {
        auto r = linear_attn_norm_bwd(s[0], s[1], s[2], done, s[5], s[6], s[7], s[3], s[4], grad_or_zeros(grads[0], s[2]),
                                      some(as(grads[1], at::kFloat)), some(as(grads[2], at::kFloat)), fmap, eps, node.wants(3) || node.wants(4),
                                      has_ss ? some(as(grads[3], at::kFloat)) : std::nullopt, parallel);
        return {r.dq, r.dk, r.dv, unless(!node.wants(3), r.dS0), unless(!node.wants(4), r.dz0)};
    }
};

std::tuple<Tensor, Tensor, Tensor, OptTensor> normalised_linear_attention(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done,
                                                                          const OptTensor &S0, const OptTensor &z0, int fmap, double eps,
                                                                          bool want_ss, bool in_place)
{
    refuse(done);
    const bool need = need_grad(q, k, v, S0, z0);
    Tensor q_, k_, v_;
    NormAttnOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        q_ = q.contiguous(), k_ = k.contiguous(), v_ = v.contiguous();
        const Tensor S0_ = as(unwrap(S0), at::kFloat), z0_ = as(unwrap(z0), at::kFloat);
        if (q_.size(1) == 1 && !need) {
            const bool own = in_place && S0.has_value() && S0_.is_same(*S0) && z0.has_value() && z0_.is_same(*z0);
            auto st = linear_attn_step(q_.select(1, 0), k_.select(1, 0), v_.select(1, 0), done.select(1, 0), some(S0_), some(z0_), fmap, true,
                                       eps, own);
            OptTensor ss;
            if (want_ss) ss = st.o.to(at::kFloat).square().sum(-1).unsqueeze(-1);   // (B,H,1)
            return {st.o.unsqueeze(1), st.S, st.z, ss};
        }
        r = linear_attn_norm_fwd(q_, k_, v_, done, some(S0_), some(z0_), fmap, eps, need, want_ss, true);
    }
    if (need) {
        auto node = record(NormalisedOp{done, fmap, eps, want_ss, r.parallel}, q, k, v, unwrap(S0), unwrap(z0));
        torch::autograd::set_history(r.o, node);
        torch::autograd::set_history(r.S_last, node);
        torch::autograd::set_history(r.z_last, node);
        if (want_ss) torch::autograd::set_history(r.ss, node);
        node->keep(0, q_);
        node->keep(1, k_);
        node->keep(2, v_);
        node->keep(3, r.o, true);
        node->keep(4, r.den);
        node->keep(5, r.S_chk);
        node->keep(6, r.z_chk);
        node->keep(7, r.S_last, true);
    }
    return {r.o, r.S_last, r.z_last, some(r.ss)};
}

struct GatedOp {
    static constexpr int SAVED = 6;   // q, k, v, g, S_chk, S_last
    static const char *name() { return "MemoraxGatedLinearAttentionBackward"; }
    Tensor done;
    int fmap;
    bool parallel;
    variable_list backward(OpNode<GatedOp> &node, std::array<Tensor, 6> &s, variable_list &grads)
    {
        auto r = gated_linear_attn_bwd(s[0], s[1], s[2], s[3], done, s[4], grad_or_zeros(grads[0], s[2]), some(as(grads[1], at::kFloat)), fmap,
                                       node.wants(4), some(s[5]), parallel);
        return {r.dq, r.dk, r.dv, r.extra, r.dS0};
    }
};

std::tuple<Tensor, Tensor> gated_linear_attention(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done,
                                                  const OptTensor &S0, int fmap, bool in_place)
{
    refuse(done);
    const bool need = need_grad(q, k, v, g, S0);
    Tensor q_, k_, v_, g_;
    AttnOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        q_ = q.contiguous(), k_ = k.contiguous(), v_ = v.contiguous(), g_ = as(g, at::kFloat);
        const Tensor S0_ = as(unwrap(S0), at::kFloat);
        if (q_.size(1) == 1 && !need) {
            auto st = gated_linear_attn_step(q_.select(1, 0), k_.select(1, 0), v_.select(1, 0), g_.select(1, 0), done.select(1, 0), some(S0_), fmap,
                                             in_place && S0.has_value() && S0_.is_same(*S0));
            return {st.o.unsqueeze(1), st.S};
        }
        r = gated_linear_attn_fwd(q_, k_, v_, g_, done, some(S0_), fmap, need, true);
    }
    if (need) {
        auto node = record(GatedOp{done, fmap, r.parallel}, q, k, v, g, unwrap(S0));
        torch::autograd::set_history(r.o, node);
        torch::autograd::set_history(r.S_last, node);
        node->keep(0, q_);
        node->keep(1, k_);
        node->keep(2, v_);
        node->keep(3, g_);
        node->keep(4, r.S_chk);
        node->keep(5, r.S_last, true);
    }
    return {r.o, r.S_last};
}

struct DeltaOp {
    static constexpr int SAVED = 6;   // q, k, v, beta, S_chk, Tm_chk
    static const char *name() { return "MemoraxDeltaRuleBackward"; }
    Tensor done;
    bool prologue;
    int resets;
    variable_list backward(OpNode<DeltaOp> &node, std::array<Tensor, 6> &s, variable_list &grads)
    {
        auto r = delta_rule_bwd(s[0], s[1], s[2], s[3], done, s[4], s[5], grad_or_zeros(grads[0], s[2]), some(as(grads[1], at::kFloat)),
                                node.wants(4), std::nullopt, prologue, resets);
        return {r.dq, r.dk, r.dv, r.extra, r.dS0};
    }
};

std::tuple<Tensor, Tensor> delta_rule(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done,
                                      const OptTensor &S0, bool prologue, int resets, bool in_place)
{
    refuse(done);
    const bool need = need_grad(q, k, v, beta, S0);
    Tensor q_, k_, v_, b_;
    DeltaOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        q_ = q.contiguous(), k_ = k.contiguous(), v_ = v.contiguous(), b_ = beta.contiguous();
        const Tensor S0_ = as(unwrap(S0), at::kFloat);
        if (q_.size(1) == 1 && !need) {
            auto st = delta_rule_step(q_.select(1, 0), k_.select(1, 0), v_.select(1, 0), b_.select(1, 0), done.select(1, 0), some(S0_),
                                      in_place && S0.has_value() && S0_.is_same(*S0), prologue);
            return {st.o.unsqueeze(1), st.S};
        }
        r = delta_rule_fwd(q_, k_, v_, b_, done, some(S0_), need, std::nullopt, prologue, std::nullopt, MRX_FACTORS_AUTO, resets);
    }
    if (need) {
        auto node = record(DeltaOp{done, prologue, resets}, q, k, v, beta, unwrap(S0));
        torch::autograd::set_history(r.o, node);
        torch::autograd::set_history(r.S_last, node);
        node->keep(0, q_);
        node->keep(1, k_);
        node->keep(2, v_);
        node->keep(3, b_);
        node->keep(4, r.S_chk);
        node->keep(5, r.Tm_chk);
    }
    return {r.o, r.S_last};
}

struct MlstmGatesOp {
    static constexpr int SAVED = 4;   // log_i, log_f, m, m0
    static const char *name() { return "MemoraxMlstmGatesBackward"; }
    Tensor done;
    double g_floor;
    variable_list backward(OpNode<MlstmGatesOp> &node, std::array<Tensor, 4> &s, variable_list &grads)
    {
        auto r = mlstm_gates_bwd(s[0], s[1], done, some(s[3]), s[2], some(as(grads[0], at::kFloat)), some(as(grads[1], at::kFloat)),
                                 some(as(grads[2], at::kFloat)), g_floor, node.wants(2));
        return {r[0], r[1], r[2]};
    }
};

std::tuple<Tensor, Tensor, Tensor> mlstm_gates(const Tensor &log_i, const Tensor &log_f, const Tensor &done, const OptTensor &m0, double g_floor)
{
    refuse(done);
    const bool need = need_grad(log_i, log_f, m0);
    Tensor li, lf, m0_;
    std::array<Tensor, 3> r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        li = as(log_i, at::kFloat), lf = as(log_f, at::kFloat), m0_ = as(unwrap(m0), at::kFloat);
        r = mlstm_gates_fwd(li, lf, done, some(m0_), g_floor);
    }
    if (need) {
        auto node = record(MlstmGatesOp{done, g_floor}, log_i, log_f, unwrap(m0));
        for (auto &t : r) torch::autograd::set_history(t, node);
        node->keep(0, li);
        node->keep(1, lf);
        node->keep(2, r[0], true);
        node->keep(3, m0_);
    }
    return {r[0], r[1], r[2]};
}

struct SiluGateOp {
    static constexpr int SAVED = 2;   // h, g
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxSiluGateBackward"; }
    variable_list backward(OpNode<SiluGateOp> &, std::array<Tensor, 2> &s, variable_list &grads)
    {
        if (!grads[0].defined()) return {Tensor(), Tensor()};
        auto r = silu_gate_bwd(s[0], s[1], as(grads[0], s[0].scalar_type()));
        return {r[0], r[1]};
    }
};

Tensor silu_gate(const Tensor &h, const Tensor &g)
{
    if (tracing()) {
        refuse_tangent(h), refuse_tangent(g);
        const auto dt = c10::promoteTypes(h.scalar_type(), g.scalar_type());
        return (h.to(at::kFloat) * at::silu(g.to(at::kFloat))).to(dt == at::kBFloat16 ? dt : at::kFloat);
    }
    const bool need = need_grad(h, g);
    Tensor hc, gc, y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        auto dt = c10::promoteTypes(h.scalar_type(), g.scalar_type());
        if (dt != at::kFloat && dt != at::kBFloat16) dt = at::kFloat;
        hc = as(h, dt), gc = as(g, dt);
        y = silu_gate_fwd(hc, gc);
    }
    if (need) {
        auto node = record(SiluGateOp{}, h, g);
        torch::autograd::set_history(y, node);
        node->keep(0, hc);
        node->keep(1, gc);
    }
    return y;
}

// A gated recurrence between its projections and its closing layer (scan.hip, GATE).
struct GatedScanOp {
    static constexpr int SAVED = 5;   // z, h~, gate, h, the states at both ends
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxGatedScanBackward"; }
    Tensor done;
    ScalarType carried;
    variable_list backward(OpNode<GatedScanOp> &node, std::array<Tensor, SAVED> &s, variable_list &grads)
    {
        const Tensor &z = s[0];
        const int64_t B = z.size(0), T = z.size(1), D = z.size(2);
        const Tensor dy = grads[0].defined() ? as(grads[0], z.scalar_type()) : at::zeros_like(z);
        chk(s[1], "h_tilde", z.scalar_type(), z.sizes());
        chk(s[2], "gate", z.scalar_type(), z.sizes());
        chk(s[3], "h", z.scalar_type(), z.sizes());
        chk(z, "z");
        chk(s[4], "ends", at::kFloat, {2, B, D});
        chk(dy, "dy", z.scalar_type(), z.sizes());
        Tensor g_last = as(grads[1], at::kFloat);
        if (!lib.mrx_gated_scan_pays(B, T, D, code(z.scalar_type()), true)) {   // the gate's backward, and then the scan's
            const auto d = silu_gate_bwd(dense16(s[3]), dense16(s[2]), dense16(dy));
            const Tensor first = s[4].select(0, 0);
            if (g_last.defined()) g_last = g_last.view({B, D}) / s[4].select(0, 1);
            auto r = mingru_bwd(z, s[1], s[3], done, first, d[0], some(g_last));
            return {unless(!node.wants(0), r.da), unless(!node.wants(1), r.db), unless(!node.wants(2), d[1]),
                    node.wants(3) ? r.dh0.mul_(first).view({B, 1, D}).to(carried) : Tensor()};
        }
        const Tensor dz = fresh_like(z), dx = fresh_like(z), dg = fresh_like(z), dls = node.wants(3) ? fresh({B, D}, at::kFloat, z) : Tensor();
        const Done flags(done, B, T);
        check(lib.mrx_gated_scan_bwd(stream(), ptr(z), ptr(s[1]), ptr(s[2]), ptr(s[3]), flags.p(), fptr(s[4]), ptr(dy), fptr(g_last), ptr(dz), ptr(dx), ptr(dg),
                                     fptr(dls), B, T, D, code(z.scalar_type()), flags.dtype),
              "mrx_gated_scan_bwd");
        return {unless(!node.wants(0), dz), unless(!node.wants(1), dx), unless(!node.wants(2), dg), dls.defined() ? dls.view({B, 1, D}).to(carried) : dls};
    }
};

// z, h~, gate (B,T,D) of one type, the carry's leaves (B,1,D) -> y = h silu(gate), log_state, log_decay
std::tuple<Tensor, Tensor, Tensor> gated_scan(const Tensor &z, const Tensor &x, const Tensor &gate, const Tensor &done, const Tensor &log_state,
                                              const Tensor &log_decay)
{
    refuse(done, log_decay);
    const bool need = need_grad(z, x, gate, log_state);
    TORCH_CHECK_VALUE(z.dim() == 3 && log_state.dim() == 3 && log_decay.dim() == 3, "z must be (B,T,D), the carry (B,1,D)");
    const int64_t B = z.size(0), T = z.size(1), D = z.size(2);
    const auto dt = z.scalar_type();
    chk_scan_dtype(dt, false, "gated_scan");
    // long sequences over few columns run in segments, which know nothing of gates: the operations this stands for; a carry of more than one step likewise
    if (log_state.size(1) != 1 || log_decay.size(1) != 1 || lib.mrx_scan_workspace(B, T, D, code(dt), MRX_SCAN_MINGRU) ||
        (need && lib.mrx_scan_workspace(B, T, D, code(dt), MRX_SCAN_MINGRU | MRX_SCAN_BACKWARD))) {
        const auto [h, h_last, P_last] = mingru_scan(z, x, done, log_state.exp().select(1, 0), log_decay.exp().select(1, 0));
        return {silu_gate(h, gate), h_last.unsqueeze(1).log(), P_last.unsqueeze(1).log()};
    }
    Tensor z_, x_, g_, h, y, ls_out, ld_out, ends;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        z_ = z.contiguous(), x_ = as(x, dt), g_ = as(gate, dt);
        const Tensor ls = as(log_state.select(1, 0), at::kFloat), ld = as(log_decay.select(1, 0), at::kFloat);
        chk(z_, "z");
        chk(x_, "h_tilde", dt, z.sizes());
        chk(g_, "gate", dt, z.sizes());
        chk(ls, "log_state", at::kFloat, {B, D});
        chk(ld, "log_decay", at::kFloat, {B, D});
        const Done flags(done, B, T);
        h = fresh_like(z_);
        if (lib.mrx_gated_scan_pays(B, T, D, code(dt), false)) {
            y = fresh_like(z_), ls_out = fresh({B, 1, D}, at::kFloat, z_), ld_out = fresh({B, 1, D}, at::kFloat, z_);
            if (need) ends = fresh({2, B, D}, at::kFloat, z_);
            check(lib.mrx_gated_scan_fwd(stream(), ptr(z_), ptr(x_), ptr(g_), flags.p(), fptr(ls), fptr(ld), ptr(h), ptr(y), fptr(ls_out), fptr(ld_out), fptr(ends), B,
                                         T, D, code(dt), flags.dtype),
                  "mrx_gated_scan_fwd");
        } else {   // the scan, and then the gate
            ends = fresh({2, B, D}, at::kFloat, z_);
            Tensor first = ends.select(0, 0), last = ends.select(0, 1);
            at::exp_out(first, ls);
            const Tensor decay = ld.exp(), decay_last = fresh_like(decay);
            check(lib.mrx_mingru_scan_fwd(stream(), ptr(z_), ptr(x_), flags.p(), fptr(first), fptr(decay), ptr(h), fptr(last), fptr(decay_last), B, T, D, code(dt),
                                          flags.dtype),
                  "mrx_mingru_scan_fwd");
            y = silu_gate_fwd(h, dense16(g_));
            ls_out = last.unsqueeze(1).log(), ld_out = decay_last.unsqueeze(1).log();
        }
    }
    if (need) {
        auto node = record(GatedScanOp{done, log_state.scalar_type()}, z, x, gate, log_state);
        torch::autograd::set_history(y, node);
        torch::autograd::set_history(ls_out, node);
        const Tensor *kept[] = {&z_, &x_, &g_, &h, &ends};
        for (int i = 0; i < GatedScanOp::SAVED; ++i) node->keep(i, *kept[i]);
    }
    return {y, ls_out, ld_out};
}

// x + branch for a float32 stream and a bfloat16 branch; the node is the array library's own, so derivatives of any order are what
// its sum's are, and so is everything the kernel does not take.
Tensor residual_add(const Tensor &x, const Tensor &branch)
{
    auto plain = [](const Tensor &t) {
        return t.is_cuda() && t.is_contiguous() && t.has_storage() && !t.is_neg() && !t._fw_grad(0).defined() &&
               !transformed(t) && !t.key_set().has(c10::DispatchKey::Python) &&
               reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    };
    if (tracing() || x.scalar_type() != at::kFloat || branch.scalar_type() != at::kBFloat16 || x.sizes() != branch.sizes() || x.numel() == 0 ||
        x.device() != branch.device() || !plain(x) || !plain(branch))
        return at::add(x, branch);
    const Tensor y = fresh_like(x);
    check(lib.mrx_residual_add(stream(), fptr(x), ptr(branch), fptr(y), x.numel()), "mrx_residual_add");
    if (at::GradMode::is_enabled() && (differentiable(x) || differentiable(branch))) {
        auto node = std::shared_ptr<torch::autograd::generated::AddBackward0>(new torch::autograd::generated::AddBackward0(),
                                                                              torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, branch));
        node->alpha = 1;
        node->self_scalar_type = at::kFloat;
        node->other_scalar_type = at::kBFloat16;
        torch::autograd::set_history(y, node);
    }
    return y;
}

// RMS norm (center false) or layer norm; fork: the input is handed on beside its norm -- (x, norm(x)) -- so that the
// gradients of both meet in the norm's backward kernel instead of in a pass of their own.
struct NormOp {
    static constexpr int SAVED = 2;   // x, scale
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxNormBackward"; }
    double eps;
    bool center, fork;
    variable_list backward(OpNode<NormOp> &node, std::array<Tensor, 2> &s, variable_list &grads)
    {
        const Tensor &x = s[0], dres = fork ? grads[0] : Tensor(), &dy = grads[fork];
        if (!dy.defined()) return {dres, Tensor(), Tensor()};   // the norm's branch was not used
        const Tensor dyc = dy.scalar_type() == at::kFloat || dy.scalar_type() == at::kBFloat16 ? dy.contiguous() : as(dy, at::kFloat);
        auto r = norm_bwd(x, some(s[1]), dyc, eps, node.wants(1) || node.wants(2), some(as(dres, x.scalar_type())), center);
        return {r.dx, unless(!node.wants(1), r.dscale), unless(!node.wants(2), r.dbias)};
    }
};

std::tuple<Tensor, Tensor> norm(const Tensor &x, const OptTensor &scale, const OptTensor &bias, double eps, std::optional<ScalarType> out_dtype,
                                bool center, bool fork)
{
    if (tracing()) {
        refuse_tangent(x), refuse_tangent(scale), refuse_tangent(bias);
        const Tensor xf = x.to(at::kFloat), w = scale.has_value() ? scale->to(at::kFloat) : Tensor(), b = bias.has_value() ? bias->to(at::kFloat) : Tensor();
        const Tensor y = center ? at::layer_norm(xf, x.sizes().slice(x.dim() - 1), some(w), some(b), eps)
                                : at::rms_norm(xf, x.sizes().slice(x.dim() - 1), some(w), eps);
        return {x, y.to(out_dtype.value_or(x.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat))};
    }
    const bool need = need_grad(x, scale, bias);
    Tensor xc, sc, y, res;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        xc = x.scalar_type() == at::kFloat || x.scalar_type() == at::kBFloat16 ? x.contiguous() : as(x, at::kFloat);
        sc = as(unwrap(scale), at::kFloat);
        y = norm_fwd(xc, some(sc), some(as(unwrap(bias), at::kFloat)), eps, out_dtype, center);
        if (fork)   // x under a second name, with x's version counter: writing to either is noticed by the saved tensor
            res = xc.scalar_type() != x.scalar_type()
                      ? xc.to(x.scalar_type())
                      : Tensor(xc.unsafeGetTensorImpl()->shallow_copy_and_detach(torch::autograd::impl::version_counter(xc), false));
    }
    if (need) {
        auto node = record(NormOp{eps, center, fork}, x, unwrap(scale), unwrap(bias));
        if (fork) torch::autograd::set_history(res, node);
        torch::autograd::set_history(y, node);
        node->keep(0, xc);
        node->keep(1, sc);
    }
    return {fork ? res : x, y};
}

// ---- dense layers (memorax_amd/dense.py): the array library's products in a shape it runs well
constexpr int64_t SLICE_ROWS = 2048, MAX_SLICES = 128;   // rows per slice of the weight-gradient product

// Into how many slices the rows of a weight-gradient product are cut: none while the result has tiles enough to fill the
// device or the rows are few.
int64_t weight_gradient_slices(int64_t rows, int64_t n_out, int64_t n_in)
{
    if (rows < 4 * SLICE_ROWS || rows < 32 * std::max(n_out, n_in)) return 1;
    int64_t s = 1;
    while (s < MAX_SLICES && rows % (2 * s) == 0 && rows / (2 * s) >= SLICE_ROWS) s *= 2;
    return s;
}

bool half(ScalarType dt) { return dt == at::kBFloat16 || dt == at::kHalf; }
ScalarType wide(ScalarType dt) { return half(dt) ? at::kFloat : dt; }

// dy^T x for dy (rows, n_out), x (rows, n_in); float32 from 16-bit operands
Tensor weight_gradient(const Tensor &dy, const Tensor &x)
{
    const int64_t rows = dy.size(0), n_out = dy.size(1), n_in = x.size(1);
    const int64_t s = dy.is_cuda() ? weight_gradient_slices(rows, n_out, n_in) : 1;
    // a ragged batch: its even part in slices, the rest by itself
    const int64_t even = rows - rows % (4 * SLICE_ROWS);
    if (dy.is_cuda() && rows != even && s < weight_gradient_slices(even, n_out, n_in))
        return weight_gradient(dy.narrow(0, 0, even), x.narrow(0, 0, even)) +
               at::mm(dy.narrow(0, even, rows - even).t(), x.narrow(0, even, rows - even));
    if (s == 1) return at::mm(dy.t(), x).to(wide(dy.scalar_type()));
    const Tensor a = dy.reshape({s, rows / s, n_out}).transpose(1, 2), b = x.reshape({s, rows / s, n_in});
    return (half(dy.scalar_type()) ? at::bmm(a, b, at::kFloat) : at::bmm(a, b)).sum(0);
}

// Gradients of dense layers that read the rows x (rows, K), of dys[l] (rows, n_l): the input's (undefined unless wanted), then
// each layer's weight and bias gradients (views of one float32 block; undefined unless wanted / without a bias).  The weights are read
// for the input's gradient only.
std::vector<Tensor> dense_grads(const Tensor &x, const std::vector<Tensor> &dys, const std::vector<Tensor> &weights, const std::vector<bool> &has_bias,
                                bool want_dx, ScalarType dx_dtype, bool want_params)
{
    const size_t L = dys.size();
    TORCH_CHECK_VALUE(L >= 1 && L <= MRX_DENSE_LAYERS && (weights.size() == L || !want_dx) && has_bias.size() == L, "dense_grads takes 1 to ", MRX_DENSE_LAYERS, " layers");
    const int64_t rows = x.size(0), K = x.size(1);
    const auto dt = x.scalar_type();
    chk(x, "x");
    std::array<const void *, MRX_DENSE_LAYERS> dy{}, w{};
    std::array<int64_t, MRX_DENSE_LAYERS> n{};
    unsigned bias = 0;
    int64_t total = 0;
    for (size_t l = 0; l < L; ++l) {
        TORCH_CHECK_VALUE(dys[l].dim() == 2, "dy must be (rows, n)");
        n[l] = dys[l].size(1);
        chk(dys[l], "dy", dt, {rows, n[l]});
        if (want_dx) chk(weights[l], "weight", dt, {n[l], K});
        dy[l] = ptr(dys[l]), w[l] = want_dx ? ptr(weights[l]) : nullptr;
        total += n[l] * (K + has_bias[l]);
        if (has_bias[l]) bias |= 1u << l;
    }
    const Tensor dx = want_dx ? fresh({rows, K}, dx_dtype, x) : Tensor();
    Tensor params, work;
    if (want_params) {
        params = fresh({(total + 3) / 4 * 4}, at::kFloat, x);
    }
    if (want_params || dt == at::kFloat)   // (where a float32 input gradient has its weights)
        if (const int64_t floats = lib.mrx_dense_grads_workspace(rows, K, n.data(), (int)L, code(dt), bias)) work = fresh({floats}, at::kFloat, x);
    check(lib.mrx_dense_grads(stream(), ptr(x), dy.data(), w.data(), n.data(), (int)L, ptr(dx), fptr(params), fptr(work), rows, K, code(dt),
                              code(dx_dtype), bias),
          "mrx_dense_grads");
    std::vector<Tensor> out(1 + 2 * L);
    out[0] = dx;
    if (want_params) {
        int64_t at = 0;
        for (size_t l = 0; l < L; ++l, at += n[l - 1] * K) out[1 + l] = params.narrow(0, at, n[l] * K).view({n[l], K});
        for (size_t l = 0; l < L; ++l)
            if (has_bias[l]) out[1 + L + l] = params.narrow(0, at, n[l]), at += n[l];
    }
    return out;
}

// The dtype the array library's autocast would run a product on x in.
std::optional<ScalarType> autocast_dtype(const Tensor &x)
{
    if (x.is_cuda() && x.is_floating_point() && at::autocast::is_autocast_enabled(at::kCUDA)) return at::autocast::get_autocast_dtype(at::kCUDA);
    return std::nullopt;
}

// What the library's kernels form of a group of dense layers on `rows` rows of K features, `widest` the most outputs of a layer and `outputs` those of all; the
// rest are the array library's products.
// bfloat16.  Parameters: while they are bound by reading the rows, i.e. up to widths where the array library's larger tiles take over (us,
// here / there: 131072 x 256 -> 3 x 256 105 / 277, 11455 x 128 -> 3 x 256 26 / 225, 32768 x 1024 -> 1024 148 / 121).  The input: several layers at
// once, as narrow (68200 x 128 -> 3 x 64 + 2 25 / 69, 131072 x 256 -> 3 x 256 + 4 118 / 150), or few rows, where the host's calls are what it costs.
// float32, on the bfloat16 matrix units (split_bf16.h).  Times in graphs, i.e. without the 20 us of the host that a product of the array library costs beside;
// sizes are taken where these are no longer here, and groups up to 512 x 512 on few rows, whose gradient of the input has always been one call of the host's.
//   forward     1024 x 128 -> 3 x 128 15 / 18, 1024 x 256 -> 3 x 256 19 / 21, 4096 x 512 -> 512 30 / 31, 4096 x 512 -> 3 x 512 50 / 63, 4096 x 1024 -> 1024 62 / 77;
//               not 256 x 512 -> 512 21 / 15, 1024 x 512 -> 3 x 512 33 / 28, 1024 x 1024 -> 1024 38 / 28
//   parameters  1024 x 256 -> 3 x 256 28 / 32, 12288 x 128 -> 256 28 / 28, 32768 x 256 -> 256 45 / 43, 131072 x 256 -> 3 x 256 + 4 412 / 414; groups 4096 x 512 -> 3 x 512
//               76 / 80, 32768 x 256 -> 1024 + 512 + 512 + 8 259 / 289; with a bias 8192 x 512 -> 512 51 / 76, 32768 x 512 -> 256 74 / 100, without 50 / 58 and 73 / 75; not
//               1024 x 512 -> 3 x 512 52 / 32, 4096 x 512 -> 512 38 / 30, 16384 x 1024 -> 1024 246 / 238
//   input       4096 x 1024 -> 1024 62 / 69, 32768 x 256 -> 256 35 / 43, 131072 x 256 -> 3 x 256 + 4 303 / 504; groups 4096 x 256 -> 3 x 256 29 / 32, 1024 x 256 ->
//               3 x 256 25 / 19, 1024 x 512 -> 3 x 512 43 / 31, 256 x 512 -> 3 x 512 43 / 23; not 12288 x 128 -> 256 21 / 17, 4096 x 512 -> 512 29 / 24, 1024 x 1024 -> 3 x 1024 88 / 62
// Sums of fewer than SPLIT_TERMS products stay float32's, whose error is that of their few additions.
constexpr int64_t SPLIT_TERMS = 64, SPLIT_WIDEST = 1 << 20;
// What mrx_dense_grads and mrx_dense_f32 take: features of a row and outputs of a layer up to DENSE_WIDEST, rows that 32 bits count.
constexpr int64_t DENSE_WIDEST = 1 << 16;
struct DenseRoutes {
    bool forward, params, input;
};
DenseRoutes dense_routes(ScalarType dt, int64_t rows, int64_t K, int64_t widest, int64_t outputs, int64_t layers)
{
    if (K % 8 != 0 || rows >= (1ll << 31) || K > DENSE_WIDEST || widest > DENSE_WIDEST || layers > MRX_DENSE_LAYERS) return {};
    const int64_t size = K * widest;
    const bool group = layers > 1, many = rows >= 4096, more = rows >= 8192;
    if (dt == at::kBFloat16) return {false, size <= 512 * 512, group && ((K <= 256 && widest <= 256) || (rows <= 4096 && size <= 512 * 512))};
    if (dt != at::kFloat || size > SPLIT_WIDEST) return {};
    const bool small = size <= 256 * 256, middle = size <= 512 * 512;
    return {K >= SPLIT_TERMS && (small || many), rows >= SPLIT_TERMS && (small || (middle && (group ? many : more))),
            outputs >= SPLIT_TERMS && ((group && middle) || (many && rows * K * outputs >= 1ll << 31))};
}

// Layers in bfloat16 whose weights fit the registers of a compute unit: the rows pass all of them once, in either direction (dense_rows.hip).
struct RowLayers {
    int suit = 0;                  // MRX_DENSE_ROWS_*
    std::vector<Tensor> weights;   // bfloat16, as the products read them
    Tensor transposed;             // (K, outputs of the wide layers): what the gradient of the input reads
};

// Outputs of layers whose parameters the kernels read where they lie -- dense, of the types that `suits` names, beside x -- or nothing.
template <typename Suits>
bool plain_layers(const Tensor &x, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, Suits suits, std::array<int64_t, MRX_DENSE_LAYERS> &n)
{
    auto plain = [&](const Tensor &t) {
        return t.device() == x.device() && t.has_storage() && !t.is_neg() && !t.key_set().has(c10::DispatchKey::Python);
    };
    if (!x.is_cuda() || !plain(x) || x.dim() < 2 || x.numel() == 0 || weights.size() > MRX_DENSE_LAYERS) return false;
    const int64_t K = x.size(-1);
    const auto wd = weights[0].scalar_type();
    std::optional<ScalarType> bd;
    for (size_t l = 0; l < weights.size(); ++l) {
        const Tensor &w = weights[l];
        if (!plain(w) || w.scalar_type() != wd || !suits(wd) || w.dim() != 2 || w.size(1) != K || !w.is_contiguous() ||
            reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 != 0)
            return false;
        n[l] = w.size(0);
        if (!biases[l].has_value()) continue;
        if (!plain(*biases[l]) || !biases[l]->is_contiguous() || biases[l]->dim() != 1 || biases[l]->numel() != n[l] || !suits(biases[l]->scalar_type())) return false;
        if (bd.value_or(biases[l]->scalar_type()) != biases[l]->scalar_type()) return false;
        bd = biases[l]->scalar_type();
    }
    return true;
}

// Whether these layers on x -- the rows in bfloat16 -- are such; their weights are not looked at beyond type, shape and place.
int row_layers(const Tensor &x, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, bool cast)
{
    std::array<int64_t, MRX_DENSE_LAYERS> n{};
    if (x.scalar_type() != at::kBFloat16 ||
        !plain_layers(x, weights, biases, [&](ScalarType dt) { return dt == at::kBFloat16 || (cast && dt == at::kFloat); }, n))
        return 0;
    return lib.mrx_dense_rows_suit(x.numel() / x.size(-1), x.size(-1), n.data(), (int)weights.size());
}

// The outputs of float32 layers on float32 rows (dense_split.hip), residual: added to the one layer's; nothing where the library does not serve them or -- unless
// `any` size is to be -- they are the array library's (dense_routes).
std::vector<Tensor> dense_f32(const Tensor &x_, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, const Tensor &residual,
                              bool any = false, const Tensor &skip = Tensor(), const Tensor &skip_x = Tensor())
{
    std::vector<Tensor> out;
    std::array<int64_t, MRX_DENSE_LAYERS> n{};
    if (x_.scalar_type() != at::kFloat || !plain_layers(x_, weights, biases, [](ScalarType dt) { return dt == at::kFloat; }, n)) return out;
    const int64_t K = x_.size(-1), rows = x_.numel() / K, floats = lib.mrx_dense_f32_workspace(n.data(), (int)weights.size(), K);
    const int64_t widest = *std::max_element(n.begin(), n.end()), outputs = std::accumulate(n.begin(), n.end(), int64_t(0));
    if (!floats || rows >= (1ll << 31) || (!any && !dense_routes(at::kFloat, rows, K, widest, outputs, (int64_t)weights.size()).forward)) return out;
    const Tensor x = dense16(x_), work = fresh({floats}, at::kFloat, x);
    std::array<const void *, MRX_DENSE_LAYERS> w{}, b{};
    std::array<void *, MRX_DENSE_LAYERS> y{};
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    for (size_t l = 0; l < weights.size(); ++l) {
        shape.back() = n[l];
        out.push_back(fresh(shape, at::kFloat, x));
        w[l] = ptr(weights[l]), b[l] = ptr(biases[l]), y[l] = ptr(out[l]);
    }
    check(lib.mrx_dense_f32(stream(), fptr(x), w.data(), b.data(), y.data(), n.data(), (int)out.size(), fptr(residual), fptr(skip), fptr(skip_x), rows, K,
                            fptr(work)),
          "mrx_dense_f32");
    return out;
}

// The weights of such layers for the products: cast, and transposed where the input's gradient will be wanted.
RowLayers pack_layers(int suit, const std::vector<Tensor> &weights, bool transpose)
{
    RowLayers r;
    r.suit = suit, r.weights = weights;
    const int64_t K = weights[0].size(1);
    const bool cast = weights[0].scalar_type() != at::kBFloat16;
    transpose = transpose && (suit & MRX_DENSE_ROWS_INPUT);
    if (!cast && !transpose) return r;
    std::array<const void *, MRX_DENSE_LAYERS> w{};
    std::array<void *, MRX_DENSE_LAYERS> copies{};
    std::array<int64_t, MRX_DENSE_LAYERS> n{};
    int64_t total = 0, wide = 0;
    for (size_t l = 0; l < weights.size(); ++l) {
        n[l] = weights[l].size(0), total += n[l] * K, w[l] = ptr(weights[l]);
        if (n[l] > 8) wide += n[l];
    }
    if (cast) {
        const Tensor all = fresh({total}, at::kBFloat16, weights[0]);
        int64_t at = 0;
        for (size_t l = 0; l < weights.size(); ++l, at += n[l - 1] * K) r.weights[l] = all.narrow(0, at, n[l] * K).view({n[l], K}), copies[l] = ptr(r.weights[l]);
    }
    if (transpose) r.transposed = fresh({K, wide}, at::kBFloat16, weights[0]);
    check(lib.mrx_dense_pack(stream(), w.data(), n.data(), (int)weights.size(), K, code(weights[0].scalar_type()), copies.data(), ptr(r.transposed)),
          "mrx_dense_pack");
    return r;
}

// The outputs of such layers on the rows x (bfloat16, dense); residual: the one layer's result added to it, in float32.
std::vector<Tensor> dense_rows(const Tensor &x, const RowLayers &layers, const std::vector<OptTensor> &biases, const Tensor &residual)
{
    std::vector<Tensor> out;
    std::array<const void *, MRX_DENSE_LAYERS> w{}, b{};
    std::array<void *, MRX_DENSE_LAYERS> y{};
    std::array<int64_t, MRX_DENSE_LAYERS> n{};
    auto bd = at::kFloat;
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    for (size_t l = 0; l < layers.weights.size(); ++l) {
        shape.back() = n[l] = layers.weights[l].size(0);
        out.push_back(fresh(shape, residual.defined() ? at::kFloat : at::kBFloat16, x));
        w[l] = ptr(layers.weights[l]), b[l] = ptr(biases[l]), y[l] = ptr(out[l]);
        if (biases[l].has_value()) bd = biases[l]->scalar_type();
    }
    check(lib.mrx_dense_rows(stream(), ptr(x), w.data(), b.data(), y.data(), n.data(), (int)out.size(), fptr(residual), x.numel() / x.size(-1),
                             x.size(-1), code(bd)),
          "mrx_dense_rows");
    return out;
}

// Several dense layers on one input: one cast of it, and the gradients with respect to it accumulated by the products
// themselves (each adds onto the sum so far) instead of by a pass per layer.
struct DenseOp {
    static constexpr int SAVED = 1;   // x as the products read it; the weights follow in `weights`
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxDenseBackward"; }
    std::vector<SavedVariable> weights;
    SavedVariable transposed;   // of a group whose input's gradient is mrx_dense_rows_input_grad's; else undefined
    std::vector<bool> has_bias;
    ScalarType x_dtype;
    bool onto = false;   // the one layer's result was added to a float32 residual, whose gradient follows the others
    variable_list backward(OpNode<DenseOp> &node, std::array<Tensor, 1> &s, variable_list &grads)
    {
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        const Tensor &x = s[0], x2 = x.reshape({-1, x.size(-1)}), across = node.wants(0) ? transposed.unpack() : Tensor();
        const size_t n = weights.size();
        const auto dt = x.scalar_type();
        variable_list out(1 + 2 * n + onto);
        if (onto) out.back() = grads[0];
        std::vector<Tensor> dys, ws;   // of the layers whose outputs were used: the others cost no products
        std::vector<size_t> used;
        std::vector<bool> bias;
        int64_t widest = 0, outputs = 0;
        bool want_params = false, regular = x.is_cuda() && (dt == at::kFloat || dt == at::kBFloat16) && x2.size(1) % 8 == 0 && x2.numel() > 0;
        for (size_t l = 0; l < n; ++l) {
            if (!grads[l].defined()) continue;
            ws.push_back(weights[l].unpack());
            dys.push_back((onto && across.defined() && grads[l].scalar_type() == at::kFloat ? grads[l] : grads[l].to(dt)).reshape({-1, ws.back().size(0)}).contiguous());
            used.push_back(l);
            bias.push_back(has_bias[l] && node.wants(1 + n + l));
            widest = std::max(widest, ws.back().size(0)), outputs += ws.back().size(0);
            want_params = want_params || node.wants(1 + l) || bias.back();
            regular = regular && ws.back().device() == x.device() && ws.back().scalar_type() == dt && ws.back().is_contiguous() && ws.back().size(0) > 0 && reinterpret_cast<uintptr_t>(ws.back().data_ptr()) % 16 == 0;
        }
        if (used.empty()) return out;
        regular = regular && used.size() <= MRX_DENSE_LAYERS && x2.is_contiguous() && reinterpret_cast<uintptr_t>(x2.data_ptr()) % 16 == 0;
        const bool rows_dx = across.defined() && used.size() == n && regular && input_from_rows(dys, ws, across, x2.size(1), want_params, out);
        for (Tensor &dy : dys) dy = dy.to(dt);   // (a residual stream's gradient: unless that has left its rounded copy)
        const DenseRoutes routes = regular ? dense_routes(dt, x2.size(0), x2.size(1), widest, outputs, (int64_t)used.size()) : DenseRoutes{};
        const bool own_params = want_params && routes.params, own_dx = node.wants(0) && !rows_dx && routes.input && (x_dtype == at::kFloat || x_dtype == at::kBFloat16);
        if (own_params || own_dx) {
            auto r = dense_grads(x2, dys, ws, bias, own_dx, x_dtype, own_params);
            if (own_dx) out[0] = r[0];
            for (size_t i = 0; i < used.size(); ++i) out[1 + used[i]] = r[1 + i], out[1 + n + used[i]] = r[1 + used.size() + i];
        }
        for (size_t i = 0; i < used.size(); ++i) {
            const size_t l = used[i];
            if (node.wants(0) && !own_dx && !rows_dx) {
                if (i > 0) out[0].addmm_(dys[i], ws[i]);
                else out[0] = at::mm(dys[i], ws[i]);
            }
            if (own_params) continue;
            if (node.wants(1 + l)) out[1 + l] = weight_gradient(dys[i], x2);
            if (bias[i]) out[1 + n + l] = dys[i].sum({0}, false, wide(dt));
        }
        if (out[0].defined()) out[0] = out[0].view(x.sizes()).to(x_dtype);
        return out;
    }
    // The input's gradient as the rows' way past the transposed weights `across`, where those are what the forward has saved (a hook on saved
    // tensors may hand on others); a float32 dy is left rounded where the parameters want it.
    static bool input_from_rows(std::vector<Tensor> &dys, const std::vector<Tensor> &ws, const Tensor &across, int64_t K, bool want_params, variable_list &out)
    {
        int64_t wide = 0;
        for (const Tensor &w : ws) wide += w.size(0) > 8 ? w.size(0) : 0;
        if (across.device() != dys[0].device() || across.scalar_type() != at::kBFloat16 || across.sizes() != IntArrayRef({K, wide}) || !across.is_contiguous() ||
            reinterpret_cast<uintptr_t>(across.data_ptr()) % 16)
            return false;
        std::array<const void *, MRX_DENSE_LAYERS> dy{};
        std::array<int64_t, MRX_DENSE_LAYERS> n{};
        const void *narrow = nullptr;
        for (size_t l = 0; l < dys.size(); ++l) {
            n[l] = ws[l].size(0), dy[l] = ptr(dys[l]);
            if (reinterpret_cast<uintptr_t>(dy[l]) % 16) return false;
            if (n[l] <= 8) narrow = ptr(ws[l]);
        }
        const auto dt = dys[0].scalar_type();
        const Tensor copy = dt == at::kFloat && want_params ? fresh(dys[0].sizes(), at::kBFloat16, dys[0]) : Tensor();
        out[0] = fresh({dys[0].size(0), K}, at::kBFloat16, dys[0]);
        check(lib.mrx_dense_rows_input_grad(stream(), dy.data(), n.data(), (int)dys.size(), ptr(across), narrow, ptr(out[0]), ptr(copy),
                                            dys[0].size(0), K, code(dt)),
              "mrx_dense_rows_input_grad");
        if (copy.defined()) dys[0] = copy;
        return true;
    }
    void release()
    {
        for (auto &w : weights) w.reset_data();
        transposed.reset_data();
    }
};

// Whether the row kernel beats the array library's products on rows of (at most) K features, for layers whose weights hold `weights`
// elements together.  It reads every weight once per 16 or 32 rows, so beyond a few hundred MFLOP a layer the library's larger tiles take
// over, and above 512 features its tiles are the small ones whatever the rows.  Plain layers, device time here / the library's (which costs
// the host 19 us a layer, 30 under autocast, against 5-7 for one launch): rows x K x n, float32 1024 x 256 x 256 6.5 / 5.8 us, 4096 x 256 x
// 256 12 / 10, 16384 x 256 x 256 34 / 22, 4096 x 512 x 1024 63 / 36, 256 x 1024 x 256 15 / 5.6, 16384 x 1024 x 4096 2227 / 966; bfloat16
// products of float32 rows and weights 4096 x 256 x 256 7 / 9, 16384 x 256 x 256 15 / 16, 4096 x 512 x 1024 33 / 15, 16384 x 1024 x 4096
// 1208 / 131.
// fused: an acting block, whose composition has a norm, casts, a sum and a dozen calls more.  Whole blocks in a graph / host-issued, fused
// over composed (gated recurrence, float32): 1024 x 512 62 / 76 and 61 / 74, 2048 x 512 96 / 80 and 91 / 134, 4096 x 512 153 / 129 and
// 147 / 135, 64 x 1024 38 / 47 and 39 / 135, 256 x 1024 65 / 60 and 62 / 134, 1024 x 1024 194 / 109 and 182 / 133, 32 x 2048 67 / 57 and
// 64 / 136; bfloat16 4096 x 512 110 / 87, 1024 x 1024 166 / 75, 32 x 2048 65 / 76.
constexpr int64_t ROW_DENSE_ROWS = 16384, ROW_DENSE_K = 512;
bool rows_pay(int64_t rows, int64_t K, int64_t weights, int64_t layers, bool fused, bool bf16)
{
    if (rows > ROW_DENSE_ROWS) return false;
    if (K <= ROW_DENSE_K) return rows * weights <= layers << 28;
    return fused && K <= (bf16 ? 2048 : 1024) && rows * weights <= layers << 27;
}

// The layers of an acting block: what the row kernel multiplies with as it is (half: bfloat16 products, under autocast), where that pays.
bool row_layers_suit(int64_t rows, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, bool half)
{
    auto suits = [](const Tensor &t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; };
    int64_t widest = 0, elements = 0;
    for (const Tensor &w : weights) {
        if (w.scalar_type() != weights[0].scalar_type() || !(half ? suits(w) : w.scalar_type() == at::kFloat) || w.dim() != 2 || w.size(1) % 8 != 0)
            return false;
        widest = std::max(widest, w.size(1)), elements += w.numel();
    }
    for (const OptTensor &b : biases)
        if (b.has_value() && !suits(*b)) return false;
    return rows_pay(rows, widest, elements, (int64_t)weights.size(), true, half);   // (which takes no more features than the kernel does)
}

// Dense maps of one input head by head (block-diagonal matrices given by their blocks (H, o, d)): x (..., H d) -> (..., H o) each.
// Batched products over strided views in both directions, so that a head's values -- infinities and NaN among them -- meet its own block
// alone; the weights' gradients are the diagonal blocks of the whole dy^T x, an element of which reads one feature of each side.  As the array
// library's einsum forms them (a batched product over every row for a result of 16 to 64 features a side, permutations around it) forward
// and backward of three maps on 32768 rows take 312 us (four heads of 16) to 531 us (four of 64) and the host 390 us; here 106 to 282 and
// 170.  (One product with the whole matrix, zeros included, takes 100 to 411 and 213, and lets heads see each other.)
struct HeadMapsOp {
    static constexpr int SAVED = 1;   // x; the maps follow in `maps`
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxHeadMapsBackward"; }
    std::vector<SavedVariable> maps;
    variable_list backward(OpNode<HeadMapsOp> &node, std::array<Tensor, 1> &s, variable_list &grads)
    {
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        const Tensor &x = s[0];
        variable_list out(1 + maps.size());
        std::vector<Tensor> dys;
        std::vector<size_t> wanted;
        for (size_t l = 0; l < maps.size(); ++l) {
            if (!grads[l].defined()) continue;
            const Tensor map = maps[l].unpack();
            const int64_t H = map.size(0), o = map.size(1), d = map.size(2);
            const Tensor dy = grads[l].reshape({-1, H * o}).contiguous(), heads = dy.view({-1, H, o}).transpose(0, 1);
            if (node.wants(0)) {
                const bool first = !out[0].defined();
                if (first) out[0] = fresh(x.sizes(), x.scalar_type(), x);
                Tensor dx = out[0].view({-1, H, d}).transpose(0, 1);
                if (first) at::bmm_out(dx, heads, map);
                else dx.baddbmm_(heads, map);
            }
            if (node.wants(1 + l)) dys.push_back(dy), wanted.push_back(l);
        }
        if (wanted.empty()) return out;
        const Tensor x2 = x.reshape({-1, x.size(-1)}).contiguous();
        int64_t widest = 0;
        for (const Tensor &dy : dys) widest = std::max(widest, dy.size(1));
        std::vector<Tensor> whole;
        if (reinterpret_cast<uintptr_t>(x2.data_ptr()) % 16 == 0 &&
            dense_routes(x2.scalar_type(), x2.size(0), x2.size(1), widest, widest, (int64_t)dys.size()).params) {
            whole = dense_grads(x2, dys, {}, std::vector<bool>(dys.size(), false), false, x2.scalar_type(), true);
            whole.erase(whole.begin());
        } else {
            for (const Tensor &dy : dys) whole.push_back(weight_gradient(dy, x2));
        }
        for (size_t i = 0; i < wanted.size(); ++i) {
            const auto map = maps[wanted[i]].unpack();
            const int64_t H = map.size(0);
            out[1 + wanted[i]] = whole[i].view({H, map.size(1), H, map.size(2)}).diagonal(0, 0, 2).permute({2, 0, 1}).contiguous();
        }
        return out;
    }
    void release()
    {
        for (auto &m : maps) m.reset_data();
    }
};

std::vector<Tensor> head_maps(const Tensor &x, const std::vector<Tensor> &maps)
{
    bool need = need_grad(x);
    for (const Tensor &m : maps) need = need_grad(m) || need;
    TORCH_CHECK_VALUE(x.is_cuda() && x.dim() >= 2 && x.scalar_type() == at::kFloat && x.numel() > 0, "head_maps takes float32 rows on the GPU");
    c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
    std::vector<Tensor> out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        for (const Tensor &m : maps) {
            TORCH_CHECK_VALUE(m.dim() == 3 && m.scalar_type() == at::kFloat && m.size(0) * m.size(2) == x.size(-1), "a map must be float32 (H, o, d) with H d = ",
                              x.size(-1), ", got ", m.sizes());
            const int64_t H = m.size(0), o = m.size(1), d = m.size(2);
            c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
            shape.back() = H * o;
            out.push_back(fresh(shape, at::kFloat, x));
            Tensor y = out.back().view({-1, H, o}).transpose(0, 1);
            at::bmm_out(y, x.reshape({-1, H, d}).transpose(0, 1), m.transpose(1, 2));
        }
    }
    if (need) {
        auto node = std::shared_ptr<OpNode<HeadMapsOp>>(new OpNode<HeadMapsOp>(), torch::autograd::deleteNode);
        torch::autograd::edge_list edges = torch::autograd::collect_next_edges(x);
        for (const Tensor &m : maps) edges.push_back(torch::autograd::impl::gradient_edge(m));
        node->set_next_edges(std::move(edges));
        for (Tensor &y : out) torch::autograd::set_history(y, node);
        node->keep(0, x);
        for (const Tensor &m : maps) node->op.maps.emplace_back(m, false);
    }
    return out;
}

// Few rows without gradients: the layers as one launch of the row kernel, where it takes the arrays as they are.
bool rows_suit(const Tensor &x, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, std::optional<ScalarType> cast)
{
    const int64_t K = x.size(-1);
    auto suits = [](ScalarType dt) { return dt == at::kFloat || dt == at::kBFloat16; };
    auto fits = [](const Tensor &t) { return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    const auto wd = weights[0].scalar_type();
    if (!x.is_cuda() || x.dim() < 2 || x.numel() == 0 || weights.size() > MRX_ROW_DENSE_LAYERS || K % 8 != 0) return false;
    int64_t elements = 0;
    for (const Tensor &w : weights) elements += w.numel();
    if (!rows_pay(x.numel() / K, K, elements, (int64_t)weights.size(), false, cast.has_value() || wd == at::kBFloat16) || !suits(x.scalar_type()) || !suits(wd) || !fits(x)) return false;
    if (cast.has_value() ? *cast != at::kBFloat16 : wd != x.scalar_type()) return false;
    for (size_t l = 0; l < weights.size(); ++l) {
        if (weights[l].scalar_type() != wd || weights[l].dim() != 2 || weights[l].size(1) != K || weights[l].size(0) == 0 || !fits(weights[l])) return false;
        if (biases[l].has_value() && (biases[l]->scalar_type() != wd || !biases[l]->is_contiguous())) return false;
    }
    return true;
}

// Records the node of layers on x, which went into the products as xc with the weights ws.
void record_dense(const Tensor &x, const Tensor &xc, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases,
                  const std::vector<Tensor> &ws, const Tensor &transposed, const OptTensor &residual, std::vector<Tensor> &out)
{
    auto node = std::shared_ptr<OpNode<DenseOp>>(new OpNode<DenseOp>(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges = torch::autograd::collect_next_edges(x);
    for (const Tensor &w : weights) edges.push_back(torch::autograd::impl::gradient_edge(w));
    for (const OptTensor &b : biases) edges.push_back(b.has_value() ? torch::autograd::impl::gradient_edge(*b) : torch::autograd::Edge());
    if (residual.has_value()) edges.push_back(torch::autograd::impl::gradient_edge(*residual));
    node->set_next_edges(std::move(edges));
    node->op.x_dtype = x.scalar_type();
    if (transposed.defined()) node->op.transposed = SavedVariable(transposed, false);
    node->op.onto = residual.has_value();
    for (Tensor &y : out) torch::autograd::set_history(y, node);
    node->keep(0, xc);
    for (size_t l = 0; l < ws.size(); ++l) {
        node->op.weights.emplace_back(ws[l], false);
        node->op.has_bias.push_back(biases[l].has_value());
    }
}

std::vector<Tensor> dense_group(const Tensor &x, const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases)
{
    TORCH_CHECK_VALUE(!weights.empty() && biases.size() == weights.size(), "dense_group takes one bias (or None) per weight");
    std::vector<Tensor> out;
    out.reserve(weights.size());
    bool others = tracing() || transformed(x);
    for (size_t l = 0; l < weights.size(); ++l) others = others || transformed(weights[l]) || transformed(biases[l]);
    if (others) {   // the array library's layers, which vmap, the functional gradients and the tracer know
        refuse_tangent(x);
        for (size_t l = 0; l < weights.size(); ++l) {
            refuse_tangent(weights[l]), refuse_tangent(biases[l]);
            out.push_back(at::linear(x, weights[l], biases[l]));
        }
        return out;
    }
    const auto cast = autocast_dtype(x);
    bool need = need_grad(x);
    for (size_t l = 0; l < weights.size(); ++l) need = need_grad(weights[l], biases[l]) || need;   // every one is looked at
    c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
    std::vector<Tensor> ws;
    Tensor xc, transposed;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        if (!need && rows_suit(x, weights, biases, cast)) {
            const auto product = cast.value_or(x.scalar_type());
            return row_dense(x, 0, std::nullopt, std::nullopt, 0.0, false, weights, biases, product, product, std::nullopt);
        }
        xc = cast.has_value() ? x.to(*cast) : x;
        const int suit = row_layers(xc, weights, biases, cast.has_value());
        if (suit & MRX_DENSE_ROWS_FORWARD) {
            xc = dense16(xc);
            auto layers = pack_layers(suit, weights, need_grad(x) && x.scalar_type() == at::kBFloat16);
            out = dense_rows(xc, layers, biases, Tensor());
            ws = std::move(layers.weights), transposed = layers.transposed;
        } else if (need && weights.size() > 1 && (out = dense_f32(xc, weights, biases, Tensor()), !out.empty())) {
            ws = weights;   // (a layer by itself has torch.nn.Linear's results bit for bit, and so has any without gradients)
        } else {
            for (size_t l = 0; l < weights.size(); ++l) {
                ws.push_back(cast.has_value() ? weights[l].to(*cast) : weights[l]);
                out.push_back(at::linear(xc, ws[l], biases[l].has_value() && cast.has_value() ? OptTensor(biases[l]->to(*cast)) : biases[l]));
            }
        }
    }
    if (need) record_dense(x, xc, weights, biases, ws, transposed, OptTensor(), out);
    return out;
}

// residual + dense(x): the layer that closes a residual branch of a float32 stream, under autocast or in bfloat16 as one launch: the
// layer's own result rounded to bfloat16, the sum in float32, as one after the other; the array library's sum of a layer's output otherwise.
Tensor dense_onto(const Tensor &residual, const Tensor &x, const Tensor &weight, const OptTensor &bias)
{
    auto composed = [&]() {
        const Tensor y = dense_group(x, {weight}, {bias})[0];
        return residual.is_cuda() && residual.scalar_type() == at::kFloat && y.scalar_type() == at::kBFloat16 ? residual_add(residual, y) : at::add(residual, y);
    };
    if (tracing() || transformed(x) || transformed(weight) || transformed(bias) || transformed(residual) || x.dim() < 2 || weight.dim() != 2 ||
        residual.scalar_type() != at::kFloat || residual._fw_grad(0).defined() || !residual.has_storage() || residual.is_neg() ||
        residual.key_set().has(c10::DispatchKey::Python) || residual.device() != x.device() || !residual.is_contiguous() ||
        reinterpret_cast<uintptr_t>(residual.data_ptr()) % 16 != 0)
        return composed();
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = weight.size(0);
    const auto cast = autocast_dtype(x);
    const auto product = cast.has_value() ? *cast : x.scalar_type();
    if (residual.sizes() != IntArrayRef(shape) || (product != at::kBFloat16 && (cast.has_value() || product != at::kFloat))) return composed();
    const bool need_x = need_grad(x), need_params = need_grad(weight, bias);
    const bool need = (at::GradMode::is_enabled() && differentiable(residual)) || need_x || need_params;
    RowLayers layers;
    Tensor xc;
    std::vector<Tensor> out;
    {
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        at::AutoDispatchBelowADInplaceOrView below;
        xc = x.to(product);
        const int suit = row_layers(xc, {weight}, {bias}, cast.has_value());
        if (product == at::kFloat && need) {
            out = dense_f32(xc, {weight}, {bias}, residual);
            layers.weights = {weight};
        }
        if (suit & MRX_DENSE_ROWS_RESIDUAL) {
            xc = dense16(xc);
            layers = pack_layers(suit, {weight}, need_x && x.scalar_type() == at::kBFloat16);
            out = dense_rows(xc, layers, {bias}, residual);
        }
    }
    if (out.empty()) return composed();
    if (need) record_dense(x, xc, {weight}, {bias}, layers.weights, layers.transposed, residual, out);
    return out[0];
}

// ---- the LRU cell (lru_cells.hip around dense_split.hip and scan.hip)
struct LruOp {
    enum { X, H, H0, PARAMS, D_ = PARAMS + 7, DECAY, WB, WC, SAVED };   // the parameters in the order of lru_cells.hip, the skip vector behind them
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxLruBackward"; }
    Tensor done;
    bool onto;   // a residual was added to the result
    variable_list backward(OpNode<LruOp> &node, std::array<Tensor, SAVED> &s, variable_list &grads)
    {
        for (int i = 0; i < SAVED; ++i) {   // a hook on saved tensors may hand them on in another layout
            s[i] = dense16(s[i]);
            chk(s[i], "saved tensor", i == H || i == H0 || i == DECAY ? at::kComplexFloat : at::kFloat);
        }
        const Tensor &x = s[X], &h = s[H];
        const int64_t B = x.size(0), T = x.size(1), F = x.size(2), N = h.size(2), rows = B * T;
        variable_list out(10 + onto);   // x, eight parameters, h0 (, the residual)
        if (onto) out.back() = grads[0];
        const Tensor dy = dense16(grad_or_zeros(grads[0], x)).view({rows, F}), x2 = x.view({rows, F});
        const auto read = dense_grads(at::view_as_real(h).view({rows, 2 * N}), {dy}, {s[WC]}, {false}, true, at::kFloat, true);
        const auto r = scan_bwd(s[DECAY], h, done, some(s[H0]), at::view_as_complex(read[0].view({B, T, N, 2})), some(as(grads[1], at::kComplexFloat)), true);
        const Tensor du = at::view_as_real(r.db).view({rows, 2 * N}), dwb = dense_grads(x2, {du}, {}, {false}, false, at::kFloat, true)[1];
        out[9] = r.dh0;
        if (node.wants(0)) {
            const int64_t n = 2 * N;
            const Tensor work = fresh({lib.mrx_dense_f32_input_grad_workspace(&n, 1, F)}, at::kFloat, x);
            const void *dys = ptr(du), *ws = ptr(s[WB]);
            out[0] = fresh_like(x);
            check(lib.mrx_dense_f32_input_grad(stream(), &dys, &ws, &n, 1, fptr(s[D_]), fptr(dy), fptr(out[0]), rows, F, fptr(work)), "mrx_dense_f32_input_grad");
        }
        if (node.wants(1 + 7)) {
            const int64_t floats = lib.mrx_column_product_workspace(rows, F);
            const Tensor work = floats ? fresh({floats}, at::kFloat, x) : Tensor();
            out[1 + 7] = fresh({F}, at::kFloat, x);
            check(lib.mrx_column_product(stream(), fptr(dy), fptr(x2), fptr(out[1 + 7]), fptr(work), rows, F), "mrx_column_product");
        }
        const Tensor decay = sum_rows(r.da);
        const float *params[7];
        float *dparams[7];
        for (int i = 0; i < 7; ++i) {
            params[i] = fptr(s[PARAMS + i]);
            out[1 + i] = fresh_like(s[PARAMS + i]);
            dparams[i] = fptr(out[1 + i]);
        }
        check(lib.mrx_lru_params_bwd(stream(), params, ptr(decay), fptr(dwb), fptr(read[1]), dparams, N, F), "mrx_lru_params_bwd");
        return out;
    }
};

// x (B,T,F) float32 through the cell, residual (nullable, as x) added; p: nu_log, theta_log, gamma_log, B_real, B_imag, C_real, C_imag, D; the
// carry's leaves (B,N) complex64.  y, and the carry's leaves afterwards.  F and 2 N multiples of eight.
std::tuple<Tensor, Tensor, Tensor> lru_layer(const Tensor &x_, const OptTensor &residual_, const std::vector<Tensor> &p, const Tensor &done, const Tensor &h0_,
                                             const Tensor &P0_)
{
    TORCH_CHECK_VALUE(x_.dim() == 3 && p.size() == 8 && p[3].dim() == 2, "lru_layer: x (B,T,F) and eight parameters");
    const int64_t B = x_.size(0), T = x_.size(1), F = x_.size(2), N = p[3].size(0);
    TORCH_CHECK_VALUE(F % 8 == 0 && N % 4 == 0 && B * T > 0, "lru_layer takes a multiple of eight features and of four states");
    refuse(done, P0_);
    bool need = need_grad(x_, residual_, h0_);
    for (const Tensor &t : p) need = need_grad(t) || need;
    chk_beside(x_, residual_, p, done, h0_, P0_);
    Tensor x, residual, h0, decay, wb, wc, y;
    std::vector<Tensor> q;
    ScanOut r;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        x = dense16(x_), residual = dense16(residual_), h0 = h0_.contiguous();
        for (const Tensor &t : p) q.push_back(dense16(t));
        chk(x, "x", at::kFloat);
        if (residual.defined()) chk(residual, "residual", at::kFloat, x.sizes());
        const float *params[8];
        const char *names[] = {"nu_log", "theta_log", "gamma_log", "B_real", "B_imag", "C_real", "C_imag", "D"};
        const std::vector<int64_t> shapes[] = {{N}, {N}, {N}, {N, F}, {N, F}, {F, N}, {F, N}, {F}};
        for (int i = 0; i < 8; ++i) chk(q[i], names[i], at::kFloat, shapes[i]), params[i] = fptr(q[i]);
        decay = fresh({N}, at::kComplexFloat, x), wb = fresh({2 * N, F}, at::kFloat, x), wc = fresh({F, 2 * N}, at::kFloat, x);
        check(lib.mrx_lru_params_fwd(stream(), params, ptr(decay), fptr(wb), fptr(wc), N, F), "mrx_lru_params_fwd");
        const auto u = dense_f32(x, {wb}, {std::nullopt}, Tensor(), true);
        TORCH_CHECK_VALUE(!u.empty(), "lru_layer: sizes that the float32 products do not serve");
        r = scan_fwd(decay, at::view_as_complex(u[0].view({B, T, N, 2})), done, some(h0), some(P0_.contiguous()), true);
        y = dense_f32(at::view_as_real(r.h).view({B, T, 2 * N}), {wc}, {std::nullopt}, residual, true, q[7], x)[0];
    }
    if (need) {
        auto node = std::shared_ptr<OpNode<LruOp>>(new OpNode<LruOp>(), torch::autograd::deleteNode);
        node->op.done = done, node->op.onto = residual_.has_value();
        torch::autograd::edge_list edges = torch::autograd::collect_next_edges(x_);
        for (const Tensor &t : p) edges.push_back(torch::autograd::impl::gradient_edge(t));
        edges.push_back(torch::autograd::impl::gradient_edge(h0_));
        if (residual_.has_value()) edges.push_back(torch::autograd::impl::gradient_edge(*residual_));
        node->set_next_edges(std::move(edges));
        torch::autograd::set_history(y, node);
        torch::autograd::set_history(r.h_last, node);
        node->keep(LruOp::X, x);
        node->keep(LruOp::H, r.h);
        node->keep(LruOp::H0, h0);
        for (int i = 0; i < 8; ++i) node->keep(LruOp::PARAMS + i, q[i]);
        node->keep(LruOp::DECAY, decay);
        node->keep(LruOp::WB, wb);
        node->keep(LruOp::WC, wc);
    }
    return {y, r.h_last, r.P_last};
}

// ---- causal depthwise convolution over time with silu behind it (conv_cells.hip)
// x (B,T,C) as the kernels walk it: its own rows where they are dense or the leading columns of wider ones
Tensor as_rows(const Tensor &x)
{
    TORCH_CHECK_VALUE(x.dim() == 3 && x.is_cuda() && x.scalar_type() == at::kFloat, "causal_conv_silu takes (B,T,C) float32 arrays on the GPU");
    const bool rows = x.stride(2) == 1 && x.stride(1) % 4 == 0 && x.stride(0) == x.size(1) * x.stride(1) && ((uintptr_t)x.data_ptr()) % 16 == 0;
    return rows ? x : dense16(x);
}

struct ConvSiluOp {
    static constexpr int SAVED = 3;   // x, weight, bias
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxCausalConvSiluBackward"; }
    variable_list backward(OpNode<ConvSiluOp> &, std::array<Tensor, 3> &s, variable_list &grads)
    {
        if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor()};
        const Tensor x = as_rows(s[0]), weight = dense16(s[1]), bias = dense16(s[2]);   // a hook may hand them on in another layout
        chk(weight, "weight", at::kFloat), chk(bias, "bias", at::kFloat);
        const int64_t B = x.size(0), T = x.size(1), C = x.size(2), K = weight.size(2);
        const Tensor dy = grads[0].contiguous(), dx = fresh(x.sizes(), at::kFloat, x), params = fresh({C * (K + 1)}, at::kFloat, x),
                     work = fresh({MRX_CONV_PARTS, C * (K + 1)}, at::kFloat, x);
        check(lib.mrx_causal_conv_silu_bwd(stream(), fptr(x), x.stride(1), fptr(weight), fptr(bias), fptr(dy), fptr(dx), C, fptr(params),
                                           fptr(work), B, T, C, K),
              "mrx_causal_conv_silu_bwd");
        return {dx, params.narrow(0, 0, C * K).view({C, 1, K}), params.narrow(0, C * K, C)};
    }
};

// x (B,T,C) float32, dense or the leading columns of wider rows; weight (C,1,K), bias (C).
Tensor causal_conv_silu(const Tensor &x_, const Tensor &weight_, const Tensor &bias_)
{
    TORCH_CHECK_VALUE(x_.dim() == 3 && weight_.dim() == 3 && x_.is_cuda() && x_.scalar_type() == at::kFloat,
                      "causal_conv_silu takes (B,T,C) float32 arrays on the GPU");
    const int64_t B = x_.size(0), T = x_.size(1), C = x_.size(2), K = weight_.size(2);
    const bool need = need_grad(x_, weight_, bias_);
    Tensor x, y, weight, bias;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        weight = dense16(weight_), bias = dense16(bias_);
        chk(weight, "weight", at::kFloat, {C, 1, K});
        chk(bias, "bias", at::kFloat, {C});
        x = as_rows(x_);
        y = fresh({B, T, C}, at::kFloat, x);
        check(lib.mrx_causal_conv_silu_fwd(stream(), fptr(x), x.stride(1), fptr(weight), fptr(bias), fptr(y), B, T, C, K), "mrx_causal_conv_silu_fwd");
    }
    if (need) {
        auto node = record(ConvSiluOp{}, x_, weight_, bias_);
        torch::autograd::set_history(y, node);
        node->keep(0, x);
        node->keep(1, weight);
        node->keep(2, bias);
    }
    return y;
}

// ---- the mLSTM cell around its recurrence (mlstm_cells.hip); k, q, n, u, num of B T H d elements in that order
struct MlstmGateRowsOp {
    static constexpr int SAVED = 6;   // q, k, v, wi, wf, log_f
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxMlstmGateRowsBackward"; }
    variable_list backward(OpNode<MlstmGateRowsOp> &, std::array<Tensor, 6> &s, variable_list &grads)
    {
        for (Tensor &t : s) t = dense16(t), chk(t, "saved tensor", at::kFloat);   // a hook may hand them on in another layout
        const int64_t H = s[0].size(2), d = s[0].size(3), n = 3 * H * H * d, columns = MRX_MLSTM_GATE_COLUMNS(H, d);
        const Tensor di = grad_or_zeros(grads[0], s[5]), df = grad_or_zeros(grads[1], s[5]), dq = fresh_like(s[0]), dk = fresh_like(s[1]), dv = fresh_like(s[2]),
                     params = fresh({columns}, at::kFloat, di), work = fresh({MRX_MLSTM_GATE_PARTS, columns}, at::kFloat, di);
        check(lib.mrx_mlstm_gate_rows_bwd(stream(), fptr(s[0]), fptr(s[1]), fptr(s[2]), fptr(s[3]), fptr(s[4]), fptr(s[5]), fptr(di), fptr(df), fptr(dq), fptr(dk),
                                          fptr(dv), fptr(params), fptr(work), s[0].size(0) * s[0].size(1), H, d),
              "mrx_mlstm_gate_rows_bwd");
        return {dq, dk, dv, params.narrow(0, 0, n).view({H, -1}), params.narrow(0, 2 * n, H), params.narrow(0, n, n).view({H, -1}), params.narrow(0, 2 * n + H, H)};
    }
};

// q, k, v (B,T,H,d), weights (H, 3 H d), biases (H) -> log_i, log_f (B,T,H)
std::tuple<Tensor, Tensor> mlstm_gate_rows(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &wi, const Tensor &bi, const Tensor &wf, const Tensor &bf)
{
    TORCH_CHECK_VALUE(q.dim() == 4, "mlstm_gate_rows takes heads of (B,T,H,d)");
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), d = q.size(3);
    const bool need = need_grad(q, k, v, wi, bi, wf, bf);
    std::array<Tensor, 7> s;
    Tensor log_i, log_f;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        s = {dense16(q), dense16(k), dense16(v), dense16(wi), dense16(wf), dense16(bi), dense16(bf)};
        for (int i = 0; i < 7; ++i) chk(s[i], "input", at::kFloat, i < 3 ? IntArrayRef({B, T, H, d}) : i < 5 ? IntArrayRef({H, 3 * H * d}) : IntArrayRef({H}));
        log_i = fresh({B, T, H}, at::kFloat, q), log_f = fresh({B, T, H}, at::kFloat, q);
        check(lib.mrx_mlstm_gate_rows_fwd(stream(), fptr(s[0]), fptr(s[1]), fptr(s[2]), fptr(s[3]), fptr(s[5]), fptr(s[4]), fptr(s[6]), fptr(log_i), fptr(log_f),
                                          B * T, H, d),
              "mrx_mlstm_gate_rows_fwd");
    }
    if (need) {
        auto node = record(MlstmGateRowsOp{}, q, k, v, wi, bi, wf, bf);
        torch::autograd::set_history(log_i, node);
        torch::autograd::set_history(log_f, node);
        for (int i = 0; i < 5; ++i) node->keep(i, s[i]);
        node->keep(5, log_f, true);
    }
    return {log_i, log_f};
}

struct MlstmKeysOp {
    static constexpr int SAVED = 3;   // k, w, g
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxMlstmKeysBackward"; }
    variable_list backward(OpNode<MlstmKeysOp> &, std::array<Tensor, 3> &s, variable_list &grads)
    {
        for (Tensor &t : s) t = dense16(t), chk(t, "saved tensor", at::kFloat);   // a hook may hand them on in another layout
        const int64_t H = s[0].size(2), d = s[0].size(3);
        const Tensor dk_in = dense16(grad_or_zeros(grads[0], s[0])), da = dense16(grad_or_zeros(grads[1], s[0])), dk = fresh_like(s[0]), dw = fresh_like(s[1]),
                     dg = fresh_like(s[2]);
        check(lib.mrx_mlstm_keys_bwd(stream(), fptr(s[0]), fptr(s[1]), fptr(s[2]), fptr(dk_in), fptr(da), fptr(dk), fptr(dw), fptr(dg),
                                     s[0].size(0) * s[0].size(1), H, d),
              "mrx_mlstm_keys_bwd");
        return {dk, dw, dg};
    }
};

// k (B,T,H,d), w and g (B,T,H) -> k_in like k and a (B,T,H d)
std::tuple<Tensor, Tensor> mlstm_keys(const Tensor &k_, const Tensor &w_, const Tensor &g_)
{
    TORCH_CHECK_VALUE(k_.dim() == 4, "mlstm_keys takes keys of (B,T,H,d)");
    const int64_t B = k_.size(0), T = k_.size(1), H = k_.size(2), d = k_.size(3);
    const bool need = need_grad(k_, w_, g_);
    Tensor k, w, g, k_in, a;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        k = dense16(k_), w = dense16(w_), g = dense16(g_);
        chk(k, "k", at::kFloat), chk(w, "w", at::kFloat, {B, T, H}), chk(g, "g", at::kFloat, {B, T, H});
        k_in = fresh_like(k), a = fresh({B, T, H * d}, at::kFloat, k);
        check(lib.mrx_mlstm_keys_fwd(stream(), fptr(k), fptr(w), fptr(g), fptr(k_in), fptr(a), B * T, H, d), "mrx_mlstm_keys_fwd");
    }
    if (need) {
        auto node = record(MlstmKeysOp{}, k_, w_, g_);
        torch::autograd::set_history(k_in, node);
        torch::autograd::set_history(a, node);
        node->keep(0, k);
        node->keep(1, w);
        node->keep(2, g);
    }
    return {k_in, a};
}

struct MlstmReadOp {
    enum { NUM, Q, N, M, SCALE, SKIP, U, Z, SAVED };
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxMlstmReadBackward"; }
    double eps;
    variable_list backward(OpNode<MlstmReadOp> &, std::array<Tensor, SAVED> &s, variable_list &grads)
    {
        if (!grads[0].defined()) return variable_list(SAVED);
        for (int i = 0; i < SAVED; ++i) {
            s[i] = i == Z ? as_rows(s[i]) : dense16(s[i]);   // a hook may hand them on in another layout
            if (i != Z) chk(s[i], "saved tensor", at::kFloat);
        }
        const int64_t B = s[NUM].size(0), T = s[NUM].size(1), H = s[NUM].size(2), d = s[NUM].size(3), W = H * d;
        const Tensor dy = dense16(grads[0]), dnum = fresh_like(s[NUM]), dq = fresh_like(s[Q]), dn = fresh_like(s[N]), dm = fresh_like(s[M]), du = fresh_like(s[U]),
                     dz = fresh({B, T, W}, at::kFloat, dy), params = fresh({2 * W}, at::kFloat, dy), work = fresh({2, MRX_MLSTM_PARTS, W}, at::kFloat, dy);
        check(lib.mrx_mlstm_read_bwd(stream(), fptr(s[NUM]), fptr(s[Q]), fptr(s[N]), fptr(s[M]), fptr(s[SCALE]), fptr(s[SKIP]), fptr(s[U]), fptr(s[Z]),
                                     s[Z].stride(1), fptr(dy), fptr(dnum), fptr(dq), fptr(dn), fptr(dm), fptr(du), fptr(dz), fptr(params), fptr(work), B * T, H,
                                     d, (float)eps),
              "mrx_mlstm_read_bwd");
        return {dnum, dq, dn, dm, params.narrow(0, 0, W).view({H, d}), params.narrow(0, W, W), du, dz};
    }
};

// num and q (B,T,H,d), n, u and z (B,T,H d), z dense or columns of wider rows, m (B,T,H), scale (H,d), skip (H d) -> (B,T,H d)
Tensor mlstm_read(const Tensor &num, const Tensor &q, const Tensor &n, const Tensor &m, const Tensor &scale, const Tensor &skip, const Tensor &u, const Tensor &z,
                  double eps)
{
    TORCH_CHECK_VALUE(num.dim() == 4, "mlstm_read takes numerators of (B,T,H,d)");
    const int64_t B = num.size(0), T = num.size(1), H = num.size(2), d = num.size(3), W = H * d;
    const bool need = need_grad(num, q, n, m, scale, skip, u, z);
    std::array<Tensor, MlstmReadOp::SAVED> s;
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        s = {dense16(num), dense16(q), dense16(n), dense16(m), dense16(scale), dense16(skip), dense16(u), as_rows(z)};
        chk(s[0], "num", at::kFloat), chk(s[1], "q", at::kFloat, {B, T, H, d}), chk(s[2], "n", at::kFloat, {B, T, W}), chk(s[3], "m", at::kFloat, {B, T, H});
        chk(s[4], "scale", at::kFloat, {H, d}), chk(s[5], "skip", at::kFloat, {W}), chk(s[6], "u", at::kFloat, {B, T, W});
        TORCH_CHECK_VALUE(z.sizes() == u.sizes(), "z must have the shape of u");
        y = fresh({B, T, W}, at::kFloat, num);
        check(lib.mrx_mlstm_read_fwd(stream(), fptr(s[0]), fptr(s[1]), fptr(s[2]), fptr(s[3]), fptr(s[4]), fptr(s[5]), fptr(s[6]), fptr(s[7]), s[7].stride(1),
                                     fptr(y), B * T, H, d, (float)eps),
              "mrx_mlstm_read_fwd");
    }
    if (need) {
        auto node = record(MlstmReadOp{eps}, num, q, n, m, scale, skip, u, z);
        torch::autograd::set_history(y, node);
        for (int i = 0; i < MlstmReadOp::SAVED; ++i) node->keep(i, s[i]);
    }
    return y;
}

// ---- the Mamba cell between its projections: elements, recurrence, gated read-out (conv_cells.hip)
struct MambaSizes {
    int64_t B, T, H, P, N, K, W;   // W = H * P, the hidden width; up holds (hidden | z): rows of 2 W
};

struct MambaOp {
    enum { UP, BIN, CIN, DTIN, CONVW, CONVB, DTB, ALOG, D_, SCALE, V, K_, Q, G, O, SCHK, DECAY0, SLAST, SAVED };
    static constexpr bool ONCE = true;
    static const char *name() { return "MemoraxMambaBackward"; }
    Tensor done;
    MambaSizes n;
    double eps;
    variable_list backward(OpNode<MambaOp> &node, std::array<Tensor, SAVED> &s, variable_list &grads)
    {
        for (Tensor &t : s) {   // a hook on saved tensors may hand them on in another layout
            t = dense16(t);
            if (t.defined()) chk(t, "saved tensor", at::kFloat);
        }
        const Tensor dy = grad_or_zeros(grads[0], s[V].view({n.B, n.T, n.W})), &up = s[UP];
        const Tensor d_up = fresh_like(up), d_o = fresh_like(s[O]), dscale = fresh({n.W}, at::kFloat, up);
        Tensor work = fresh({MRX_RMS_NORM_PARTS, n.W}, at::kFloat, up);
        check(lib.mrx_mamba_readout_bwd(stream(), fptr(s[O]), fptr(s[V]), fptr(up) + n.W, 2 * n.W, fptr(s[D_]), fptr(s[SCALE]), fptr(dy),
                                        fptr(d_o), fptr(d_up) + n.W, 2 * n.W, fptr(dscale), fptr(work), n.B * n.T, n.H, n.P, (float)eps),
              "mrx_mamba_readout_bwd");
        auto r = gated_linear_attn_bwd(s[Q], s[K_], s[V], s[G], done, s[SCHK], d_o, some(as(grads[1], at::kFloat)), 0, node.wants(10), s[SLAST], parallel);
        const Tensor &decay0 = s[DECAY0];
        Tensor ddecay0;
        if (grads[2].defined()) {   // the decay leaf handed on: it depends on every g from the last reset on
            const Tensor behind = done.ne(0).to(at::kInt).flip(1).cumsum(1).flip(1);   // resets at or after each step
            const Tensor live = (behind - done.ne(0).to(at::kInt)).eq(0).to(at::kFloat).unsqueeze(-1), intact = behind.slice(1, 0, 1).eq(0).to(at::kFloat);
            const Tensor total = (s[G] * live).sum(1).exp() * grads[2].to(at::kFloat);   // (B,H), per unit of the decay it started from
            ddecay0 = total * intact;
            r.extra = r.extra + live * ((at::where(intact.ne(0), decay0, at::ones_like(decay0)) * total).unsqueeze(1));
        }
        const int64_t C = n.W + 2 * n.H * n.N, cols = C * (n.K + 1) + 2 * n.H + n.W / 4;
        const Tensor params = fresh({cols}, at::kFloat, up), db_in = fresh_like(s[BIN]), dc_in = fresh_like(s[CIN]), ddt = fresh_like(s[DTIN]);
        work = fresh({MRX_CONV_PARTS, cols}, at::kFloat, up);
        check(lib.mrx_mamba_elements_bwd(stream(), fptr(up), 2 * n.W, fptr(s[BIN]), fptr(s[CIN]), fptr(s[DTIN]), fptr(s[CONVW]), fptr(s[CONVB]),
                                         fptr(s[DTB]), fptr(s[ALOG]), fptr(s[D_]), fptr(r.dv), fptr(r.dk), fptr(r.dq), fptr(r.extra), fptr(d_o),
                                         fptr(d_up), 2 * n.W, fptr(db_in), fptr(dc_in), fptr(ddt), fptr(params), fptr(work), n.B, n.T, n.H, n.P,
                                         n.N, n.K),
              "mrx_mamba_elements_bwd");
        auto part = [&, at = int64_t(0)](int64_t len) mutable { return params.narrow(0, std::exchange(at, at + len), len); };
        const Tensor dw = part(C * n.K).view({C, 1, n.K}), dcb = part(C), ddtb = part(n.H), dA = part(n.H), dD = part(n.W / 4).view({n.H, n.P / 4}).sum(1);
        return {d_up, db_in, dc_in, ddt, dw, dcb, ddtb, dA, dD, dscale, r.dS0, ddecay0};
    }
    bool parallel;
};

// up (B,T,2HP), b_in, c_in (B,T,HN), dt_in (B,T,H) and the cell's parameters, all float32 -> y (B,T,HP) before the output
// projection, S_last (B,H,P,N), decay_last (B,H).  Acting (one step, no gradients) runs the single-step kernel.
std::tuple<Tensor, Tensor, Tensor> mamba_mix(const Tensor &up, const Tensor &b_in, const Tensor &c_in, const Tensor &dt_in, const Tensor &conv_w_,
                                             const Tensor &conv_b_, const Tensor &dt_bias_, const Tensor &A_log_, const Tensor &D_,
                                             const Tensor &scale_, const Tensor &done_, const Tensor &S0, const Tensor &decay0, double eps,
                                             bool in_place)
{
    TORCH_CHECK_VALUE(up.dim() == 3 && S0.dim() == 4 && conv_w_.dim() == 3, "mamba_mix: up (B,T,2HP), S0 (B,H,P,N), conv_w (C,1,K)");
    MambaSizes n{up.size(0), up.size(1), S0.size(1), S0.size(2), S0.size(3), conv_w_.size(2), S0.size(1) * S0.size(2)};
    const int64_t C = n.W + 2 * n.H * n.N;
    refuse(done_);
    const bool need = need_grad(up, b_in, c_in, dt_in, conv_w_, conv_b_, dt_bias_, A_log_, D_, scale_, S0, decay0);
    Tensor conv_w, conv_b, dt_bias, A_log, D, scale;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        conv_w = dense16(conv_w_), conv_b = dense16(conv_b_), dt_bias = dense16(dt_bias_), A_log = dense16(A_log_), D = dense16(D_),
        scale = dense16(scale_);
    }
    chk(up, "up", at::kFloat, {n.B, n.T, 2 * n.W});
    chk(b_in, "b_in", at::kFloat, {n.B, n.T, n.H * n.N});
    chk(c_in, "c_in", at::kFloat, {n.B, n.T, n.H * n.N});
    chk(dt_in, "dt_in", at::kFloat, {n.B, n.T, n.H});
    chk(conv_w, "conv_w", at::kFloat, {C, 1, n.K});
    chk(conv_b, "conv_b", at::kFloat, {C});
    chk(dt_bias, "dt_bias", at::kFloat, {n.H});
    chk(A_log, "A_log", at::kFloat, {n.H});
    chk(D, "D", at::kFloat, {n.H});
    chk(scale, "scale", at::kFloat, {n.W});
    Tensor v, k, q, g, o, S_chk, S_last, y, decay0_, decay_last;
    bool parallel = false;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor S0_ = as(S0, at::kFloat);
        decay0_ = as(decay0, at::kFloat);
        chk(decay0_, "decay0", at::kFloat, {n.B, n.H});
        const Done done(done_, n.B, n.T);
        v = fresh({n.B, n.T, n.H, n.P}, at::kFloat, up), k = fresh({n.B, n.T, n.H, n.N}, at::kFloat, up), q = fresh_like(k), g = fresh_like(dt_in);
        check(lib.mrx_mamba_elements_fwd(stream(), fptr(up), 2 * n.W, fptr(b_in), fptr(c_in), fptr(dt_in), fptr(conv_w), fptr(conv_b),
                                         fptr(dt_bias), fptr(A_log), fptr(v), fptr(k), fptr(q), fptr(g), n.B, n.T, n.H, n.P, n.N, n.K),
              "mrx_mamba_elements_fwd");
        if (n.T == 1 && !need) {
            auto st = gated_linear_attn_step(q.select(1, 0), k.select(1, 0), v.select(1, 0), g.select(1, 0), done.t.select(1, 0), S0_, 0,
                                             in_place && S0_.is_same(S0));
            o = st.o, S_last = st.S;
        } else {
            auto r = gated_linear_attn_fwd(q, k, v, g, done.t, S0_, 0, need, true);
            parallel = r.parallel;
            o = r.o, S_last = r.S_last, S_chk = r.S_chk;
        }
        y = fresh({n.B, n.T, n.W}, at::kFloat, up);
        check(lib.mrx_mamba_readout_fwd(stream(), fptr(o), fptr(v), fptr(up) + n.W, 2 * n.W, fptr(D), fptr(scale), fptr(y), n.B * n.T, n.H, n.P,
                                        (float)eps),
              "mrx_mamba_readout_fwd");
        decay_last = fresh({n.B, n.H}, at::kFloat, up);
        check(lib.mrx_decay_last(stream(), fptr(g), done.p(), fptr(decay0_), fptr(decay_last), n.B, n.T, n.H, done.dtype), "mrx_decay_last");
    }
    if (need) {
        auto node = record(MambaOp{done_, n, eps, parallel}, up, b_in, c_in, dt_in, conv_w_, conv_b_, dt_bias_, A_log_, D_, scale_, S0, decay0);
        torch::autograd::set_history(y, node);
        torch::autograd::set_history(S_last, node);
        torch::autograd::set_history(decay_last, node);
        const Tensor *kept[] = {&up, &b_in, &c_in, &dt_in, &conv_w, &conv_b, &dt_bias, &A_log, &D, &scale, &v, &k, &q, &g, &o, &S_chk, &decay0_};
        for (int i = 0; i < MambaOp::SLAST; ++i) node->keep(i, *kept[i]);
        node->keep(MambaOp::SLAST, S_last, true);
    }
    return {y, S_last, decay_last};
}

// Whether a hook waits in a torch module or below it, or one of the methods that fused operations stand for was replaced on an instance (as
// adapters and accelerators do).  An acting step asks on every call: from Python the walk over the eighteen modules of a small block pair
// takes 7 us of a step of 88.  deep: below it too.
bool any_hook(PyObject *module, bool deep)
{
    static PyObject *const hooks[] = {PyUnicode_InternFromString("_forward_hooks"), PyUnicode_InternFromString("_forward_pre_hooks"),
                                      PyUnicode_InternFromString("_backward_hooks"), PyUnicode_InternFromString("_backward_pre_hooks")};
    static PyObject *const methods[] = {PyUnicode_InternFromString("forward"), PyUnicode_InternFromString("scan"),
                                        PyUnicode_InternFromString("read"), PyUnicode_InternFromString("elements")};
    static PyObject *const children = PyUnicode_InternFromString("_modules");
    PyObject **const at = _PyObject_GetDictPtr(module);
    if (!at || !*at) return false;   // None, or no torch module
    for (PyObject *name : hooks) {
        PyObject *const held = PyDict_GetItem(*at, name);
        if (held && PyDict_Check(held) && PyDict_Size(held) > 0) return true;
    }
    for (PyObject *name : methods)
        if (PyDict_GetItem(*at, name)) return true;
    if (!deep) return false;
    PyObject *const below = PyDict_GetItem(*at, children);
    if (!below || !PyDict_Check(below)) return false;
    PyObject *key, *child;
    for (Py_ssize_t pos = 0; PyDict_Next(below, &pos, &key, &child);)
        if (any_hook(child, true)) return true;
    return false;
}

// ---- a run of acting blocks
PyObject *held(PyObject *module, const char *dict, const char *name)   // a borrowed reference, or none
{
    PyObject **const at = module ? _PyObject_GetDictPtr(module) : nullptr;
    if (!at || !*at) return nullptr;
    PyObject *const of = dict ? PyDict_GetItemString(*at, dict) : *at;
    PyObject *const found = of && PyDict_Check(of) ? PyDict_GetItemString(of, name) : nullptr;
    return found == Py_None ? nullptr : found;
}
PyObject *child(PyObject *module, const char *name) { return held(module, "_modules", name); }
Tensor param(PyObject *module, const char *name)
{
    PyObject *const p = held(module, "_parameters", name);
    return p ? py::cast<Tensor>(py::handle(p)) : Tensor();
}

// One block as the kernels read it.
struct ActBlock {
    enum Kind { DELTA = 0, LINEAR = 1, GATED = 2 } kind;
    int norm = 0;                     // of the block: 1 RMS, 2 layer norm
    Tensor scale, nbias;
    double eps = 0;
    std::vector<Tensor> w, b;         // of the opening layers and, last, of the closing one; b undefined where there is none
    Tensor out_scale;                 // the norm of the read-out
    double out_eps = 0, den_eps = 0;
    ScalarType dtype;                 // of the projections and the read-out
    Tensor carry[2];                  // S (, z); log_state, log_decay
    Tensor next[2], z;
    std::vector<int64_t> n;
    int64_t H = 0, D = 0, N = 0;
};

// Whether a stack's run of blocks on x (B,1,F) float32 takes this one: everything as it lies there, no copy and no conversion.  What is refused here goes
// the usual way, block by block, errors included.
bool act_block(ActBlock &k, const Tensor &x, const py::tuple &spec, const py::tuple &types, ScalarType product)
{
    // (kind, model, norm, carry, dtype, den_eps): model a cell, or a gated recurrence; types: Dense, Linear, RMSNorm, LayerNorm
    k.kind = (ActBlock::Kind)spec[0].cast<int>();
    PyObject *const model = spec[1].ptr(), *const norm = spec[2].ptr();
    auto is = [&](PyObject *o, int i) { return o && (PyObject *)Py_TYPE(o) == py::handle(types[i]).ptr(); };
    const int64_t B = x.size(0), F = x.size(2);
    bool fits = true;
    auto plain = [&](const Tensor &t, ScalarType dt, IntArrayRef shape) {
        fits = fits && t.defined() && t.scalar_type() == dt && t.device() == x.device() && t.sizes() == shape && t.is_contiguous() && t.has_storage() &&
               !t.is_neg() && !t.key_set().has(c10::DispatchKey::Python) && !transformed(t) && !t._fw_grad(0).defined() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
        return fits;
    };
    auto number = [&](PyObject *o, const char *name) {
        PyObject *const v = held(o, nullptr, name);
        if (!v || !PyFloat_Check(v)) fits = false;
        return fits ? PyFloat_AsDouble(v) : 0.0;
    };
    if (is(norm, 2)) {
        k.norm = 1, k.scale = param(norm, "scale");
    } else if (is(norm, 3)) {
        k.norm = 2, k.scale = param(norm, "weight"), k.nbias = param(norm, "bias");
        if (!k.scale.defined()) return false;
    } else {
        return false;
    }
    k.eps = number(norm, "eps");
    if (!plain(k.scale, at::kFloat, {F}) || (k.nbias.defined() && !plain(k.nbias, at::kFloat, {F}))) return false;
    std::vector<PyObject *> layers;
    if (k.kind == ActBlock::GATED) {
        PyObject *const cell = child(model, "cell");
        layers = {child(cell, "z"), child(cell, "h"), child(model, "gate"), child(model, "out")};
    } else {
        layers = {child(model, "query"), child(model, "key"), child(model, "value")};
        if (k.kind == ActBlock::DELTA) layers.push_back(child(model, "beta"));
        layers.push_back(child(model, "output_projection"));
        PyObject *const out_norm = child(model, "norm");
        if (!is(out_norm, 2)) return false;
        k.out_scale = param(out_norm, "scale"), k.out_eps = number(out_norm, "eps");
    }
    std::vector<OptTensor> biases;
    for (PyObject *layer : layers) {
        if (!is(layer, 0) && !is(layer, 1)) return false;
        k.w.push_back(param(layer, "weight")), k.b.push_back(param(layer, "bias"));
        if (!k.w.back().defined()) return false;
        biases.push_back(some(k.b.back()));
    }
    const auto wd = k.w[0].scalar_type();
    if (!row_layers_suit(B, k.w, biases, product == at::kBFloat16)) return false;
    const size_t opening = k.w.size() - 1;
    const int64_t read = k.w[opening].size(1);
    auto bd = at::kFloat;   // of the opening layers' biases
    bool first_bias = true;
    for (size_t l = 0; l <= opening; ++l) {
        k.n.push_back(k.w[l].size(0));
        if (!plain(k.w[l], wd, {k.n[l], l < opening ? F : read})) return false;
        if (!k.b[l].defined()) continue;
        const auto dt = k.b[l].scalar_type();
        if (l < opening && std::exchange(first_bias, false)) bd = dt;
        if ((l < opening && dt != bd) || !plain(k.b[l], dt, {k.n[l]})) return false;
    }
    if (F > 512 || k.n[opening] != F || read % 8 != 0 || read > 2048) return false;
    const py::tuple carry = spec[3];
    if (carry.size() > 2) return false;
    for (size_t i = 0; i < carry.size(); ++i) k.carry[i] = carry[i].cast<Tensor>();
    k.N = k.n[0];
    if (k.kind == ActBlock::GATED) {
        k.dtype = product;
        for (int l = 0; l < 3; ++l)
            if (k.b[l].defined() || k.n[l] != k.N) return false;
        return k.N % 4 == 0 && read == k.N && carry.size() == 2 && plain(k.carry[0], at::kFloat, {B, 1, k.N}) && plain(k.carry[1], at::kFloat, {B, 1, k.N});
    }
    k.dtype = spec[4].cast<ScalarType>(), k.den_eps = spec[5].cast<double>();
    if (carry.size() != (k.kind == ActBlock::LINEAR ? 2u : 1u) || k.carry[0].dim() != 5) return false;
    k.H = k.carry[0].size(2), k.D = k.carry[0].size(3);
    if (!plain(k.carry[0], at::kFloat, {B, 1, k.H, k.D, k.D}) || (k.kind == ActBlock::LINEAR && !plain(k.carry[1], at::kFloat, {B, 1, k.H, k.D}))) return false;
    for (int l = 0; l < 3; ++l)
        if (k.n[l] != k.H * k.D) return false;
    return plain(k.out_scale, at::kFloat, {read}) && read == k.N && (k.kind == ActBlock::LINEAR || k.n[3] == k.H) && (k.dtype == at::kFloat || k.dtype == at::kBFloat16) &&
           k.D <= 64 && k.D % (k.dtype == at::kBFloat16 ? 8 : 4) == 0;
}

// Whether the closing layer (K -> F) in the launch of what it opens -- layers of n columns, or a gated recurrence's -- takes less time than before it.  Each
// workgroup of the opening (act_chain.hip: 16 rows and 256 or, gated, 64 columns of three layers) forms the closing layer for its rows again, at the price of reading all
// of its weights; what is saved is a launch and a trip to memory.  Behind 512 MB of other traffic, us, apart / as one, weights and products in bfloat16 unless said:
//     beyond a workgroup for each compute unit      qkv 512 wide 64 features 2048 rows 20.8 / 21.3, gated 512 wide 1024 rows 17.2 / 21.2, 1024 wide 23.6 / 37.7
//     gated recurrences, by the bytes of weights a workgroup reads
//                                                   256 wide 256 features 32 rows 12.2 / 11.8, weights in float32 (448 KB) 15.2 / 15.3, 512 wide (704 KB) 17.9 / 19.3;
//                                                   float32 products 1024 wide 128 features 256 rows (352 KB) 19.4 / 18.8, 256 wide 256 features (448 KB) 16.4 / 18.2
//     other layers, half the compute units at work  256 wide 256 features 1024 rows 14.0 / 11.8, weights in float32 512 wide 512 rows (768 KB) 18.5 / 18.2;
//                                                   float32 products 512 wide 128 features 512 rows (384 KB) 19.0 / 17.5, 256 wide 256 features 1024 rows (512 KB) 19.5 / 20.5
//     fewer: apart, the closing layer has more workgroups than rows fill here, and its weights come in by all of them
//                                                   256 wide 256 features 32 rows 9.4 / 10.7, 128 features 9.2 / 7.4, 64 wide 256 features 8.9 / 8.7;
//                                                   float32 products 64 wide 128 features 9.1 / 9.9, 256 wide 64 features 10.8 / 10.2
bool chain_pays(int64_t B, int64_t F, int64_t K, IntArrayRef n, bool gated, int64_t weight_bytes, bool bf16, int64_t units)
{
    int64_t columns = 0;
    for (const int64_t c : n) columns += (c + 15) / 16 * 16;
    const int64_t groups = gated ? (n[0] + 63) / 64 : (columns + 255) / 256, wgs = (B + 15) / 16 * groups;
    if (wgs > units) return false;
    const int64_t read = weight_bytes * F * (K + (gated ? 192 : std::min<int64_t>(columns, 256)));
    if (gated) return read <= (bf16 ? 448 : 352) << 10;
    if (2 * wgs >= units) return read <= (bf16 ? 768 : 384) << 10;
    return F <= (bf16 ? 128 : 64) || (bf16 && groups == 1);
}

void run_act(const Tensor &x0, std::vector<ActBlock> &blocks, const Done &done, ScalarType product, bool in_place, Tensor &y)
{
    const int64_t B = x0.size(0), F = x0.size(2);
    void *const st = stream();
    const int pc = code(product);
    auto bytes = [](int64_t n, ScalarType dt) { return (n * (int64_t)c10::elementSize(dt) + 255) / 256 * 256; };
    // one allocation for everything between the blocks: what a block hands its closing layer lies in one half, what the next block writes meanwhile in the
    // other, and so do the residual streams
    int64_t part = 0;
    for (const ActBlock &k : blocks) {
        int64_t need = bytes(B * k.N, k.dtype);
        if (k.kind != ActBlock::GATED)
            for (size_t l = 0; l + 1 < k.n.size(); ++l) need += bytes(B * k.n[l], k.dtype);
        part = std::max(part, need);
    }
    part += bytes(B * F, at::kFloat);
    const Tensor scratch = fresh({2 * part}, at::kByte, x0);
    y = fresh(x0.sizes(), at::kFloat, x0);

    struct {
        bool any = false;
        mrx_closing c{};
        int wd = 0;
    } pending;
    const float *x = fptr(x0);
    auto close = [&] {   // the last block's closing layer in a launch of its own
        const mrx_closing &c = pending.c;
        const void *w = c.weight, *b = c.bias;
        void *out = c.out;
        check(lib.mrx_row_dense(st, c.rows, c.scale, nullptr, c.norm, c.round_norm, &w, &b, &out, &F, 1, c.residual, B, c.K, c.row_dtype, pending.wd,
                                c.bias_dtype, MRX_F32, pc, c.eps, nullptr, 0, nullptr, nullptr),
              "mrx_row_dense");
        pending.any = false;
    };
    // opens a block on what the pending closing layer leaves, in one launch if that pays and is taken
    const int64_t units = compute_units(x0);
    auto open = [&](const ActBlock &k, int wd, auto chained, auto alone) {
        if (pending.any) {
            x = pending.c.out;
            if (F <= 256 && pending.wd == wd &&
                chain_pays(B, F, pending.c.K, IntArrayRef(k.n).slice(0, k.n.size() - 1), k.kind == ActBlock::GATED, wd == MRX_F32 ? 4 : 2, product == at::kBFloat16,
                           units)) {
                const int rc = chained(&pending.c);
                if (rc != MRX_ERR_UNSUPPORTED) {
                    check(rc, "mrx_closing");
                    pending.any = false;
                    return;
                }
            }
            close();
        }
        alone();
    };
    for (size_t i = 0; i < blocks.size(); ++i) {
        ActBlock &k = blocks[i];
        char *at = static_cast<char *>(scratch.data_ptr()) + (i % 2) * part;
        auto take = [&](int64_t n, ScalarType dt) {
            char *const p = at;
            at += bytes(n, dt);
            return static_cast<void *>(p);
        };
        float *const stream_out = static_cast<float *>(take(B * F, at::kFloat));
        const int wd = code(k.w[0].scalar_type());
        const size_t last = k.w.size() - 1;
        for (int j = 0; j < 2; ++j)
            if (k.carry[j].defined()) k.next[j] = in_place ? k.carry[j] : fresh_like(k.carry[j]);
        void *rows;
        if (k.kind == ActBlock::GATED) {
            k.z = fresh({B, 1, k.N}, product, x0);
            rows = take(B * k.N, product);
            auto launch = [&](const mrx_closing *c) {
                return lib.mrx_closed_gated_recurrence_act(st, c, c ? nullptr : x, fptr(k.scale), fptr(k.nbias), k.norm, ptr(k.w[0]), ptr(k.w[1]), ptr(k.w[2]),
                                                           done.p(), fptr(k.carry[0]), fptr(k.carry[1]), ptr(k.z), rows, fptr(k.next[0]), fptr(k.next[1]), B, F,
                                                           k.N, wd, pc, done.dtype, (float)k.eps);
            };
            open(k, wd, launch, [&] { check(launch(nullptr), "mrx_closed_gated_recurrence_act"); });
        } else {
            std::array<const void *, MRX_ROW_DENSE_LAYERS> w{}, b{};
            std::array<void *, MRX_ROW_DENSE_LAYERS> u{};
            int bd = MRX_F32;
            for (size_t l = 0; l < last; ++l) {
                w[l] = ptr(k.w[l]), b[l] = ptr(k.b[l]), u[l] = take(B * k.n[l], k.dtype);
                if (k.b[l].defined()) bd = code(k.b[l].scalar_type());
            }
            open(k, wd, [&](const mrx_closing *c) {
                return lib.mrx_closed_row_dense(st, c, fptr(k.scale), fptr(k.nbias), k.norm, w.data(), b.data(), u.data(), k.n.data(), (int)last, B, F, wd, bd,
                                                code(k.dtype), pc, (float)k.eps);
            }, [&] {
                check(lib.mrx_row_dense(st, x, fptr(k.scale), fptr(k.nbias), k.norm, 0, w.data(), b.data(), u.data(), k.n.data(), (int)last, nullptr, B, F, MRX_F32,
                                        wd, bd, code(k.dtype), pc, (float)k.eps, nullptr, 0, nullptr, nullptr),
                      "mrx_row_dense");
            });
            rows = take(B * k.N, k.dtype);
            if (k.kind == ActBlock::DELTA)
                check(lib.mrx_deltanet_step(st, u[0], u[1], u[2], u[3], done.p(), fptr(k.carry[0]), rows, fptr(k.next[0]), B, k.H, k.D, k.D, code(k.dtype),
                                            done.dtype),
                      "mrx_deltanet_step");
            else
                check(lib.mrx_linear_attn_step(st, u[0], u[1], u[2], done.p(), fptr(k.carry[0]), fptr(k.carry[1]), rows, fptr(k.next[0]), fptr(k.next[1]), B, k.H,
                                               k.D, k.D, code(k.dtype), done.dtype, MRX_FMAP_ELU1, (float)k.den_eps),
                      "mrx_linear_attn_step");
        }
        pending.any = true, pending.wd = wd;
        pending.c = mrx_closing{rows, fptr(k.out_scale), ptr(k.w[last]), ptr(k.b[last]), x, i + 1 == blocks.size() ? fptr(y) : stream_out, k.N,
                                k.kind != ActBlock::GATED, k.kind != ActBlock::GATED && k.dtype == at::kBFloat16, code(k.dtype),
                                k.b[last].defined() ? code(k.b[last].scalar_type()) : MRX_F32, (float)k.out_eps};
    }
    close();
}

// The leading blocks of `specs` that the kernels take as they are, on x (B,1,F): how many, what leaves the last of them, and each one's next carry (with
// a gated recurrence's z behind it).
py::tuple stack_act(const Tensor &x, const py::list &specs, const py::tuple &types, const Tensor &done_, bool in_place)
{
    const ScalarType product = autocast_dtype(x).value_or(at::kFloat);
    std::vector<ActBlock> blocks;
    blocks.reserve(specs.size());
    if (!tracing() && !x.key_set().has(c10::DispatchKey::Python) && !transformed(x) && !transformed(done_) && x.dim() == 3 && x.size(1) == 1 && x.is_cuda() &&
        x.scalar_type() == at::kFloat && x.is_contiguous() && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && !x._fw_grad(0).defined() &&
        !done_._fw_grad(0).defined() && !done_.key_set().has(c10::DispatchKey::Python) &&
        (product == at::kFloat || product == at::kBFloat16) && done_.device() == x.device() && done_.dim() == 2 && done_.size(0) == x.size(0) && done_.size(1) == 1)
        for (const auto &spec : specs) {
            blocks.emplace_back();
            if (act_block(blocks.back(), x, py::reinterpret_borrow<py::tuple>(spec), types, product)) continue;
            blocks.pop_back();
            break;
        }
    py::list carries;
    if (blocks.empty()) return py::make_tuple(0, x, carries);
    Tensor y;
    {
        py::gil_scoped_release free;
        run_act(x, blocks, Done(done_, x.size(0), 1), product, in_place, y);
    }
    for (const ActBlock &k : blocks) {
        if (k.kind == ActBlock::GATED) carries.append(py::make_tuple(k.next[0], k.next[1], k.z));
        else if (k.kind == ActBlock::LINEAR) carries.append(py::make_tuple(k.next[0], k.next[1]));
        else carries.append(py::make_tuple(k.next[0]));
    }
    return py::make_tuple(blocks.size(), y, carries);
}

}  // namespace

PYBIND11_MODULE(_native, m)
{
    m.def("bind", &bind);
    m.def("any_hook", [](py::handle module, bool deep) { return any_hook(module.ptr(), deep); });
    m.def("stack_act", &stack_act);
    // the other calls touch no Python object: they run without the interpreter's lock
    auto def = [&](const char *name, auto f) { m.def(name, f, py::call_guard<py::gil_scoped_release>()); };
    def("chunk_size", &chunk_size);
    // checks, allocation, launch (memorax_amd/kernels.py)
    auto opt = [](const Tensor &t) { return some(t); };
    def("linear_scan_fwd", [=](const Tensor &a, const Tensor &b, const Tensor &done, const OptTensor &h0, const OptTensor &P0, bool want_P) {
        auto r = scan_fwd(a, b, done, h0, P0, want_P);
        return std::make_tuple(r.h, r.h_last, opt(r.P_last));
    });
    def("linear_scan_bwd", [](const Tensor &a, const Tensor &h, const Tensor &done, const OptTensor &h0, const Tensor &g,
                                const OptTensor &g_last, bool sum_da) {
        auto r = scan_bwd(a, h, done, h0, g, g_last, sum_da);
        return std::make_tuple(r.da, r.db, r.dh0);
    });
    def("linear_scan_last", &scan_last);
    def("mingru_scan_fwd", [=](const Tensor &z, const Tensor &x, const Tensor &done, const OptTensor &h0, const OptTensor &P0, bool want_P) {
        auto r = mingru_fwd(z, x, done, h0, P0, want_P);
        return std::make_tuple(r.h, r.h_last, opt(r.P_last));
    });
    def("mingru_scan_bwd", [](const Tensor &z, const Tensor &x, const Tensor &h, const Tensor &done, const OptTensor &h0, const Tensor &g,
                                const OptTensor &g_last) {
        auto r = mingru_bwd(z, x, h, done, h0, g, g_last);
        return std::make_tuple(r.da, r.db, r.dh0);
    });
    def("mlstm_gates_fwd", [](const Tensor &li, const Tensor &lf, const Tensor &done, const OptTensor &m0, double g_floor) {
        auto r = mlstm_gates_fwd(li, lf, done, m0, g_floor);
        return std::make_tuple(r[0], r[1], r[2]);
    });
    def("mlstm_gates_bwd", [=](const Tensor &li, const Tensor &lf, const Tensor &done, const OptTensor &m0, const Tensor &mm, const OptTensor &dm,
                                 const OptTensor &dg, const OptTensor &dw, double g_floor, bool want_dm0) {
        auto r = mlstm_gates_bwd(li, lf, done, m0, mm, dm, dg, dw, g_floor, want_dm0);
        return std::make_tuple(r[0], r[1], opt(r[2]));
    });
    def("norm_fwd", &norm_fwd);
    def("norm_bwd", [=](const Tensor &x, const OptTensor &scale, const Tensor &dy, double eps, bool want, const OptTensor &dx_add, bool center) {
        auto r = norm_bwd(x, scale, dy, eps, want, dx_add, center);
        return std::make_tuple(r.dx, opt(r.dscale), opt(r.dbias));
    });
    def("silu_gate_fwd", &silu_gate_fwd);
    def("silu_gate_bwd", [](const Tensor &h, const Tensor &g, const Tensor &dy) {
        auto r = silu_gate_bwd(h, g, dy);
        return std::make_tuple(r[0], r[1]);
    });
    def("linear_attn_fwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const OptTensor &S0, int fmap,
                                 bool save_chk, std::optional<bool> chunk_parallel) {
        auto r = linear_attn_fwd(q, k, v, done, S0, fmap, save_chk, chunk_parallel);
        return std::make_tuple(r.o, r.S_last, opt(r.S_chk), r.parallel);
    });
    def("linear_attn_bwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const Tensor &S_chk,
                                 const OptTensor &S_last, const Tensor &dout, const OptTensor &dS_last, int fmap, bool want_dS0) {
        auto r = linear_attn_bwd(q, k, v, done, S_chk, S_last, dout, dS_last, fmap, want_dS0);
        return std::make_tuple(r.dq, r.dk, r.dv, opt(r.dS0));
    });
    def("linear_attn_norm_fwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const OptTensor &S0,
                                      const OptTensor &z0, int fmap, double eps, bool save_chk, bool want_ss) {
        auto r = linear_attn_norm_fwd(q, k, v, done, S0, z0, fmap, eps, save_chk, want_ss);
        return std::make_tuple(r.o, r.den, r.S_last, r.z_last, opt(r.S_chk), opt(r.z_chk), opt(r.ss));
    });
    def("linear_attn_norm_bwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const Tensor &S_chk,
                                      const Tensor &z_chk, const Tensor &S_last, const Tensor &o, const Tensor &den, const Tensor &dout,
                                      const OptTensor &dS_last, const OptTensor &dz_last, int fmap, double eps, bool want_d0,
                                      const OptTensor &d_ss) {
        auto r = linear_attn_norm_bwd(q, k, v, done, S_chk, z_chk, S_last, o, den, dout, dS_last, dz_last, fmap, eps, want_d0, d_ss);
        return std::make_tuple(r.dq, r.dk, r.dv, opt(r.dS0), opt(r.dz0));
    });
    def("gated_linear_attn_fwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done,
                                       const OptTensor &S0, int fmap, bool save_chk) {
        auto r = gated_linear_attn_fwd(q, k, v, g, done, S0, fmap, save_chk);
        return std::make_tuple(r.o, r.S_last, opt(r.S_chk));
    });
    def("gated_linear_attn_bwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done,
                                       const Tensor &S_chk, const Tensor &dout, const OptTensor &dS_last, int fmap, bool want_dS0,
                                       const OptTensor &S_last) {
        auto r = gated_linear_attn_bwd(q, k, v, g, done, S_chk, dout, dS_last, fmap, want_dS0, S_last);
        return std::make_tuple(r.dq, r.dk, r.dv, r.extra, opt(r.dS0));
    });
    def("delta_rule_fwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done, const OptTensor &S0,
                                bool save_chk, const std::optional<std::array<OptTensor, 4>> &out, bool prologue, std::optional<bool> tm_scratch,
                                int factors, int resets) {
        auto r = delta_rule_fwd(q, k, v, beta, done, S0, save_chk, out, prologue, tm_scratch, factors, resets);
        return std::make_tuple(r.o, r.S_last, opt(r.S_chk), opt(r.Tm_chk));
    });
    def("delta_rule_bwd", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done, const Tensor &S_chk,
                                const Tensor &Tm_chk, const Tensor &dout, const OptTensor &dS_last, bool want_dS0,
                                const std::optional<std::array<OptTensor, 5>> &out, bool prologue, int resets) {
        auto r = delta_rule_bwd(q, k, v, beta, done, S_chk, Tm_chk, dout, dS_last, want_dS0, out, prologue, resets);
        return std::make_tuple(r.dq, r.dk, r.dv, r.extra, opt(r.dS0));
    });
    def("delta_rule_fwd_noalloc", [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done,
                                       const OptTensor &S0, const OptTensor &o, const OptTensor &S_last) {
        auto r = delta_rule_fwd_noalloc(q, k, v, beta, done, S0, o, S_last);
        return std::make_tuple(r[0], r[1]);
    });
    def("linear_attn_step", [=](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &done, const OptTensor &S, const OptTensor &z,
                                  int fmap, bool normalise, double eps, bool inplace) {
        auto r = linear_attn_step(q, k, v, done, S, z, fmap, normalise, eps, inplace);
        return std::make_tuple(r.o, r.S, opt(r.z));
    });
    def("gated_linear_attn_step", [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &done, const OptTensor &S,
                                       int fmap, bool inplace) {
        auto r = gated_linear_attn_step(q, k, v, g, done, S, fmap, inplace);
        return std::make_tuple(r.o, r.S);
    });
    def("delta_rule_step", [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &beta, const Tensor &done, const OptTensor &S,
                                bool inplace) {
        auto r = delta_rule_step(q, k, v, beta, done, S, inplace, false);
        return std::make_tuple(r.o, r.S);
    });
    def("row_dense", [](const Tensor &x, int norm, const OptTensor &scale, const OptTensor &nbias, double eps, bool round_norm,
                        const std::vector<Tensor> &weights, const std::vector<OptTensor> &biases, ScalarType product, ScalarType out_dtype,
                        const OptTensor &residual) {
        return row_dense(x, norm, scale, nbias, eps, round_norm, weights, biases, product, out_dtype, residual);
    });
    def("rows_pay", &rows_pay);
    def("gated_scan", &gated_scan);
    def("row_layers_suit", &row_layers_suit);
    def("lru_act", &lru_act);
    def("mlstm_act", &mlstm_act);
    def("mingru_step", &mingru_step);
    def("gated_act", &gated_act);
    def("state_act", &state_act);
    // differentiable operators (memorax_amd/functional.py)
    def("linear_scan", &linear_scan);
    def("mingru_scan", &mingru_scan);
    def("linear_attention", &linear_attention);
    def("normalised_linear_attention", &normalised_linear_attention);
    def("gated_linear_attention", &gated_linear_attention);
    def("delta_rule", &delta_rule);
    def("mlstm_gates", &mlstm_gates);
    def("place_inputs", &place_inputs);
    def("mlstm_gate_rows", &mlstm_gate_rows);
    def("mlstm_keys", &mlstm_keys);
    def("mlstm_read", &mlstm_read);
    def("silu_gate", &silu_gate);
    def("residual_add", &residual_add);
    def("norm", &norm);
    def("dense_group", &dense_group);
    def("dense_onto", &dense_onto);
    def("head_maps", &head_maps);
    def("dense_grads", &dense_grads);
    def("dense_routes", +[](ScalarType dt, int64_t rows, int64_t K, int64_t widest, int64_t outputs, int64_t layers) {
        const DenseRoutes r = dense_routes(dt, rows, K, widest, outputs, layers);
        return std::make_tuple(r.forward, r.params, r.input);
    });
    def("weight_gradient", &weight_gradient);
    def("weight_gradient_slices", &weight_gradient_slices);
    def("lru_layer", &lru_layer);
    def("causal_conv_silu", &causal_conv_silu);
    def("mamba_mix", &mamba_mix);
}
