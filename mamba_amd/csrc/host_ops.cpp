// The host side of the Python layer's calls, native: argument checks, output
// and scratch allocation, argument blocks and the call into libmamba_ss.so.
//
// A scan step's two calls fill about 130 fields of the C ABI's argument
// blocks; from Python, through ctypes, they and the checks ahead of them took
// 251 us per forward + backward of a 2 x 64 x 256 scan whose kernels run for
// 45 us (now 130, most of it torch's autograd engine); a block's decode step
// took 95 us (now 42), RMSNorm forward + backward at 32768 x 768 155 to 164 (92;
// figures bound by the host vary by a quarter between runs there).  The functions
// here take the tensors, the raw stream handle and flags, and raise the same
// exceptions with the same messages.  They hold no state.  The GIL is released
// around the calls into the library.
#include <torch/extension.h>

#include <optional>
#include <string>
#include <vector>

#include "../../include/mamba_ss.h"

namespace py = pybind11;
using at::Tensor;
using OptT = std::optional<Tensor>;

namespace {

[[noreturn]] void value_error(const std::string& msg) { throw py::value_error(msg); }

std::string shape_str(at::IntArrayRef s) {            // as Python prints a tuple
    std::string r = "(";
    for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
    return r + (s.size() == 1 ? ",)" : ")");
}
std::string dtype_str(at::ScalarType t) { return std::string(py::str(py::cast(t))); }

// what: the module's prefix of its messages
#define REQUIRE(what, cond, msg)                                                   \
    do {                                                                           \
        if (!(cond)) value_error(std::string(what) + ": " + (msg));                \
    } while (0)

void check(int rc, const char* what) {
    if (rc == SS_OK) return;
    const std::string msg = std::string(what) + ": " + ss_last_error();
    if (rc == SS_ERR_INVALID || rc == SS_ERR_UNSUPPORTED) value_error(msg);
    throw std::runtime_error(msg);
}

template <typename F>
void launch(const at::Device& dev, const char* what, F&& f) {
    int rc;
    {
        py::gil_scoped_release nogil;
        const c10::OptionalDeviceGuard guard(dev);
        rc = f();
    }
    check(rc, what);                 // (the message is this thread's)
}

bool itype_of(at::ScalarType t, int32_t* out) {
    switch (t) {
        case at::kFloat: *out = SS_F32; return true;
        case at::kBFloat16: *out = SS_BF16; return true;
        case at::kHalf: *out = SS_F16; return true;
        default: return false;
    }
}
bool unit(const Tensor& t) { return t.size(-1) <= 1 || t.stride(-1) == 1; }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const OptT& t) { return t ? t->data_ptr() : nullptr; }
template <typename T> T* fptr(const OptT& t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }
Tensor f32_like(at::IntArrayRef shape, const Tensor& like) {
    return at::empty(shape, like.options().dtype(at::kFloat).memory_format(c10::nullopt));
}
Tensor bytes_on(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

// ------------------------------------------------------------------ scan --
constexpr const char* kScan = "selective_scan";

int64_t chunks(int64_t seqlen) { return (seqlen + ss_chunk_size() - 1) / ss_chunk_size(); }

void check_seq(const char* name, const Tensor& t, at::IntArrayRef shape, at::ScalarType dtype, const at::Device& dev) {
    REQUIRE(kScan, t.device() == dev, std::string(name) + " is on " + t.device().str() + ", expected " + dev.str());
    REQUIRE(kScan, t.sizes() == shape,
            std::string(name) + " has shape " + shape_str(t.sizes()) + ", expected " + shape_str(shape));
    REQUIRE(kScan, t.scalar_type() == dtype,
            std::string(name) + " has dtype " + dtype_str(t.scalar_type()) + ", expected " + dtype_str(dtype));
    REQUIRE(kScan, unit(t), std::string(name) + " must have unit stride along seqlen");
}

void fill_fwd(ss_fwd_args& a, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C,
              const OptT& D, const OptT& bias, bool softplus, const OptT& z, const OptT& out, const OptT& x,
              const OptT& y) {
    REQUIRE(kScan, u.dim() == 3, "u must be (batch, dim, seqlen), got shape " + shape_str(u.sizes()));
    const at::Device dev = u.device();
    REQUIRE(kScan, dev.is_cuda(), "tensors must be on a ROCm GPU device (no CPU path)");
    int32_t itype = 0;
    REQUIRE(kScan, itype_of(u.scalar_type(), &itype), "unsupported dtype " + dtype_str(u.scalar_type()));
    const at::ScalarType dt = u.scalar_type();
    const int64_t batch = u.size(0), dim = u.size(1), seqlen = u.size(2);
    check_seq("delta", delta, u.sizes(), dt, dev);
    REQUIRE(kScan, A.dim() == 2 && A.size(0) == dim, "A must be (dim, dstate), got " + shape_str(A.sizes()));
    REQUIRE(kScan, A.scalar_type() == at::kFloat && A.device() == dev, "A must be fp32 on the same device");
    const int64_t dstate = A.size(1);
    const bool vb = B.dim() >= 3, vc = C.dim() >= 3;
    const int64_t groups = vb ? B.size(1) : vc ? C.size(1) : 1;
    for (int i = 0; i < 2; ++i) {
        const Tensor& M = i ? C : B;
        const std::string name = i ? "C" : "B";
        REQUIRE(kScan, M.device() == dev, name + " is on " + M.device().str() + ", expected " + dev.str());
        if (i ? vc : vb) {
            REQUIRE(kScan, M.dim() == 4 && M.size(0) == batch && M.size(1) == groups && M.size(2) == dstate &&
                               M.size(3) == seqlen,
                    name + " must be (batch, n_groups, dstate, seqlen), got " + shape_str(M.sizes()));
            REQUIRE(kScan, M.scalar_type() == dt,
                    name + " has dtype " + dtype_str(M.scalar_type()) + ", expected " + dtype_str(dt));
            REQUIRE(kScan, seqlen <= 1 || M.stride(3) == 1, name + " must have unit stride along seqlen");
        } else {
            REQUIRE(kScan, M.dim() == 2 && M.size(0) == dim && M.size(1) == dstate,
                    "constant " + name + " must be (dim, dstate), got " + shape_str(M.sizes()));
            REQUIRE(kScan, M.scalar_type() == at::kFloat, "constant " + name + " must be fp32");
        }
    }
    for (int i = 0; i < 2; ++i) {
        const OptT& v = i ? bias : D;
        if (v)
            REQUIRE(kScan, v->dim() == 1 && v->size(0) == dim && v->scalar_type() == at::kFloat && v->device() == dev &&
                               v->is_contiguous(),
                    std::string(i ? "delta_bias" : "D") + " must be a contiguous fp32 (" + std::to_string(dim) +
                        ",) tensor");
    }
    if (z) check_seq("z", *z, u.sizes(), dt, dev);
    a = ss_fwd_args{};
    a.batch = batch; a.dim = dim; a.seqlen = seqlen; a.dstate = dstate; a.n_groups = groups;
    a.itype = itype;
    a.is_var_B = vb; a.is_var_C = vc;
    a.has_D = D.has_value(); a.has_delta_bias = bias.has_value(); a.has_z = z.has_value();
    a.delta_softplus = softplus;
    a.n_chunks = chunks(seqlen);
    a.u_batch_stride = u.stride(0); a.u_dim_stride = u.stride(1);
    a.delta_batch_stride = delta.stride(0); a.delta_dim_stride = delta.stride(1);
    if (z) a.z_batch_stride = z->stride(0), a.z_dim_stride = z->stride(1);
    if (out) a.out_batch_stride = out->stride(0), a.out_dim_stride = out->stride(1);
    if (y) a.y_batch_stride = y->stride(0), a.y_dim_stride = y->stride(1);
    a.A_dim_stride = A.stride(0); a.A_dstate_stride = A.stride(1);
    if (vb) a.B_batch_stride = B.stride(0), a.B_group_stride = B.stride(1), a.B_dstate_stride = B.stride(2);
    else a.B_group_stride = B.stride(0), a.B_dstate_stride = B.stride(1);
    if (vc) a.C_batch_stride = C.stride(0), a.C_group_stride = C.stride(1), a.C_dstate_stride = C.stride(2);
    else a.C_group_stride = C.stride(0), a.C_dstate_stride = C.stride(1);
    a.u = ptr(u); a.delta = ptr(delta); a.A = static_cast<float*>(ptr(A)); a.B = ptr(B); a.C = ptr(C);
    a.D = fptr<float>(D); a.delta_bias = fptr<float>(bias); a.z = ptr(z);
    a.out = ptr(out); a.x = fptr<float>(x); a.y = ptr(y);
}

bool same_shape(const Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }

// As forward_into's checks: the outputs, then everything fill_fwd looks at.
void fill_fwd_into(ss_fwd_args& a, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B,
                   const Tensor& C, const OptT& D, const OptT& bias, bool softplus, const OptT& out, const OptT& x,
                   const OptT& z, const OptT& y, const OptT& last) {
    REQUIRE(kScan, out.has_value(), "out is required");
    check_seq("out", *out, u.sizes(), delta.scalar_type(), u.device());
    REQUIRE(kScan, u.dim() == 3, "u must be (batch, dim, seqlen), got shape " + shape_str(u.sizes()));
    const int64_t batch = u.size(0), dim = u.size(1), seqlen = u.size(2), n = A.dim() == 2 ? A.size(1) : -1;
    if (x)
        REQUIRE(kScan, x->scalar_type() == at::kFloat && x->is_contiguous() && x->device() == u.device() &&
                           same_shape(*x, {batch, chunks(seqlen), dim, n}),
                "x must be a contiguous fp32 (batch, n_chunks, dim, dstate) tensor");
    if (y) check_seq("y", *y, u.sizes(), delta.scalar_type(), u.device());
    if (last)
        REQUIRE(kScan, last->scalar_type() == at::kFloat && last->is_contiguous() && last->device() == u.device() &&
                           same_shape(*last, {batch, dim, n}),
                "last_state must be a contiguous fp32 (batch, dim, dstate) tensor");
    fill_fwd(a, u, delta, A, B, C, D, bias, softplus, z, out, x, y);
    a.last_state = fptr<float>(last);
}

void scan_fwd(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C, const OptT& D,
              const OptT& bias, bool softplus, const OptT& out, const OptT& x, const OptT& z, const OptT& y,
              const OptT& last, bool auto_ws, OptT ws, int64_t stream) {
    ss_fwd_args a;
    fill_fwd_into(a, u, delta, A, B, C, D, bias, softplus, out, x, z, y, last);
    if (auto_ws) {
        const int64_t n = ss_fwd_workspace_bytes(&a);
        if (n < 0) check(SS_ERR_INVALID, "selective_scan.forward");
        if (n > 0) ws = bytes_on(n, u);
    }
    if (ws) {
        REQUIRE(kScan, ws->is_cuda() && ws->is_contiguous(), "workspace must be a contiguous GPU tensor");
        a.workspace = ptr(*ws);
        a.workspace_bytes = ws->numel() * ws->element_size();
    }
    // (a workspace made here is freed to the stream's caching allocator, which
    // keeps it valid for the work queued on the stream)
    launch(u.device(), "selective_scan.forward", [&] { return ss_fwd(&a, reinterpret_cast<void*>(stream)); });
}

Tensor seq_unit(const Tensor& t) { return unit(t) ? t : t.contiguous(); }
Tensor f32c(const Tensor& t) { return t.to(at::kFloat).contiguous(); }

// SelectiveScanZFn's forward: (out, last_state, saved tensors, B squeezed, C squeezed).
py::tuple scan_z_fwd(const Tensor& u_, const Tensor& delta_, const Tensor& A_, const Tensor& B_, const Tensor& C_,
                     const OptT& D_, const OptT& z_, const OptT& bias_, bool softplus, bool need_bwd, bool want_last,
                     int64_t stream) {
    const Tensor u = seq_unit(u_), delta = seq_unit(delta_);
    const OptT z = z_ ? OptT(seq_unit(*z_)) : OptT();
    const bool sqB = B_.dim() == 3, sqC = C_.dim() == 3;
    Tensor B = sqB ? B_.unsqueeze(1) : B_, C = sqC ? C_.unsqueeze(1) : C_;
    B = B.dim() < 3 ? f32c(B) : seq_unit(B);
    C = C.dim() < 3 ? f32c(C) : seq_unit(C);
    const Tensor A = A_.to(at::kFloat);
    const OptT D = D_ ? OptT(f32c(*D_)) : OptT(), bias = bias_ ? OptT(f32c(*bias_)) : OptT();
    REQUIRE(kScan, u.dim() == 3, "u must be (batch, dim, seqlen), got shape " + shape_str(u.sizes()));
    REQUIRE(kScan, A.dim() == 2, "A must be (dim, dstate), got " + shape_str(A.sizes()));
    const int64_t batch = u.size(0), dim = u.size(1), seqlen = u.size(2), n = A.size(1);
    const Tensor out = at::empty_like(delta, delta.options(), at::MemoryFormat::Contiguous);
    // the checkpoints x and the pre-gate output y exist for the backward:
    // without a gradient to compute they are neither allocated nor written
    OptT x, y, last;
    if (need_bwd) x = f32_like({batch, chunks(seqlen), dim, n}, u);
    if (need_bwd && z) y = at::empty_like(out);
    if (want_last) {
        last = f32_like({batch, dim, n}, u);
        if (seqlen == 0) last->zero_();
    }
    scan_fwd(u, delta, A, B, C, D, bias, softplus, out, x, z, y, last, true, OptT(), stream);
    return py::make_tuple(out, last, py::make_tuple(u, delta, A, B, C, D, bias, z, x, y), sqB, sqC);
}

void fill_bwd(ss_bwd_args& b, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C,
              const OptT& D, const OptT& bias, const Tensor& dout, const OptT& x, bool softplus, const Tensor& du,
              const Tensor& ddelta, const OptT& dA, const OptT& dB, const OptT& dC, const OptT& dD, const OptT& dbias,
              const OptT& z, const OptT& y, const OptT& dz) {
    REQUIRE(kScan, x.has_value(), "x (the forward's checkpoints) is required");
    REQUIRE(kScan, !z || (y && dz), "y from the forward and dz are required with z");
    REQUIRE(kScan, u.dim() == 3, "u must be (batch, dim, seqlen), got shape " + shape_str(u.sizes()));
    const int64_t batch = u.size(0), dim = u.size(1), seqlen = u.size(2), n = A.dim() == 2 ? A.size(1) : -1;
    const at::Device dev = u.device();
    REQUIRE(kScan, x->scalar_type() == at::kFloat && same_shape(*x, {batch, chunks(seqlen), dim, n}) &&
                       x->is_contiguous() && x->device() == dev,
            "x does not come from forward");
    const at::ScalarType ddt = delta.scalar_type();
    check_seq("dout", dout, u.sizes(), ddt, dev);
    check_seq("du", du, u.sizes(), u.scalar_type(), dev);
    check_seq("ddelta", ddelta, u.sizes(), ddt, dev);
    if (y) check_seq("y", *y, u.sizes(), ddt, dev);
    if (dz) check_seq("dz", *dz, u.sizes(), ddt, dev);
    const struct { const char* name; const OptT& g; const Tensor* ref; } gs[] = {
        {"dA", dA, &A}, {"dB", dB, &B}, {"dC", dC, &C}, {"dD", dD, D ? &*D : nullptr},
        {"ddelta_bias", dbias, bias ? &*bias : nullptr}};
    for (const auto& e : gs)
        if (e.ref)
            REQUIRE(kScan, e.g && e.g->scalar_type() == at::kFloat && e.g->is_contiguous() &&
                               e.g->sizes() == e.ref->sizes() && e.g->device() == dev,
                    std::string(e.name) + " must be a contiguous fp32 tensor of shape " + shape_str(e.ref->sizes()));
    b = ss_bwd_args{};
    fill_fwd(b.f, u, delta, A, B, C, D, bias, softplus, z, OptT(), x, y);
    b.dout_batch_stride = dout.stride(0); b.dout_dim_stride = dout.stride(1);
    b.du_batch_stride = du.stride(0); b.du_dim_stride = du.stride(1);
    b.ddelta_batch_stride = ddelta.stride(0); b.ddelta_dim_stride = ddelta.stride(1);
    if (dz) b.dz_batch_stride = dz->stride(0), b.dz_dim_stride = dz->stride(1);
    b.dout = ptr(dout); b.du = ptr(du); b.ddelta = ptr(ddelta); b.dz = ptr(dz);
    b.dA = fptr<float>(dA); b.dB = fptr<float>(dB); b.dC = fptr<float>(dC); b.dD = fptr<float>(dD);
    b.ddelta_bias = fptr<float>(dbias);
}

// The backward of a filled block; auto_ws allocates the scratch it asks for.
void run_bwd(ss_bwd_args& b, const Tensor& u, bool auto_ws, OptT ws, bool zero, int64_t stream) {
    if (auto_ws) {
        const int64_t n = ss_bwd_workspace_bytes(&b);
        if (n < 0) check(SS_ERR_INVALID, "selective_scan.backward");
        if (n > 0) ws = bytes_on(n, u);
    }
    if (ws) {
        REQUIRE(kScan, ws->device() == u.device() && ws->is_contiguous(),
                "workspace must be a contiguous tensor on the inputs' device");
        b.workspace = ptr(*ws);
        b.workspace_bytes = ws->numel() * ws->element_size();
    }
    b.zero_grads = zero;
    launch(u.device(), "selective_scan.backward", [&] { return ss_bwd(&b, reinterpret_cast<void*>(stream)); });
}

void scan_bwd(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C, const OptT& D,
              const OptT& bias, const Tensor& dout, const OptT& x, bool softplus, const Tensor& du,
              const Tensor& ddelta, const OptT& dA, const OptT& dB, const OptT& dC, const OptT& dD, const OptT& dbias,
              const OptT& z, const OptT& y, const OptT& dz, bool auto_ws, OptT ws, bool zero, bool deterministic,
              int64_t stream) {
    ss_bwd_args b;
    fill_bwd(b, u, delta, A, B, C, D, bias, dout, x, softplus, du, ddelta, dA, dB, dC, dD, dbias, z, y, dz);
    b.deterministic = deterministic;
    run_bwd(b, u, auto_ws, std::move(ws), zero, stream);
}

// backward(): gradients allocated here, cleared by the library.
py::tuple scan_bwd_new(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C,
                       const OptT& D, const OptT& bias, const Tensor& dout, const OptT& x, bool softplus,
                       const OptT& z, const OptT& y, bool deterministic, int64_t stream) {
    const auto like = [](const Tensor& t) { return at::empty_like(t, t.options(), at::MemoryFormat::Contiguous); };
    const Tensor du = like(u), ddelta = like(delta);
    const Tensor dA = f32_like(A.sizes(), A), dB = f32_like(B.sizes(), B), dC = f32_like(C.sizes(), C);
    const OptT dD = D ? OptT(f32_like(D->sizes(), *D)) : OptT();
    const OptT dbias = bias ? OptT(f32_like(bias->sizes(), *bias)) : OptT(), dz = z ? OptT(like(*z)) : OptT();
    scan_bwd(u, delta, A, B, C, D, bias, dout, x, softplus, du, ddelta, dA, dB, dC, dD, dbias, z, y, dz, true, OptT(),
             true, deterministic, stream);
    return py::make_tuple(du, ddelta, dA, dB, dC, dD, dbias, dz);
}

// ------------------------------------------------------------------ conv --
Tensor weight2d(const Tensor& w_, int64_t dim) {
    const Tensor w = w_.dim() == 3 ? w_.reshape({w_.size(0), w_.size(-1)}) : w_;
    REQUIRE(kScan, w.dim() == 2 && w.size(0) == dim, "weight must be (dim, width), got " + shape_str(w_.sizes()));
    return w;
}
// The weight as (dim, width) and the bias as the library reads them: in the
// rows' type where both are, else in fp32.
std::pair<Tensor, OptT> conv_params(const Tensor& weight, const OptT& bias, int64_t dim, const at::Device& dev,
                                    at::ScalarType rows = at::kFloat) {
    const bool io = weight.scalar_type() == rows && (!bias || bias->scalar_type() == rows);
    const at::ScalarType ty = io ? rows : at::kFloat;
    const Tensor w = weight2d(weight, dim).to(dev, ty);
    OptT b;
    if (bias) {
        b = bias->to(dev, ty).contiguous();
        REQUIRE(kScan, same_shape(*b, {dim}),
                "bias must be (" + std::to_string(dim) + ",), got " + shape_str(bias->sizes()));
    }
    return {w, b};
}
int32_t dtype_code(const Tensor& t) {
    int32_t c = SS_F32;
    itype_of(t.scalar_type(), &c);
    return c;
}
void fill_conv(ss_conv1d_args& a, const Tensor& x, const Tensor& w, const OptT& b, bool silu, const OptT& out) {
    REQUIRE(kScan, x.dim() == 3, "x must be (batch, dim, seqlen), got " + shape_str(x.sizes()));
    REQUIRE(kScan, x.is_cuda(), "tensors must be on a ROCm GPU device (no CPU path)");
    a = ss_conv1d_args{};
    REQUIRE(kScan, itype_of(x.scalar_type(), &a.itype), "unsupported dtype " + dtype_str(x.scalar_type()));
    REQUIRE(kScan, unit(x), "x must have unit stride along seqlen");
    a.batch = x.size(0); a.dim = x.size(1); a.seqlen = x.size(2); a.width = w.size(1);
    a.has_bias = b.has_value(); a.silu = silu;
    a.x_batch_stride = x.stride(0); a.x_dim_stride = x.stride(1);
    if (out) a.out_batch_stride = out->stride(0), a.out_dim_stride = out->stride(1);
    a.w_dim_stride = w.stride(0); a.w_width_stride = w.stride(1);
    // (weight and bias of the type passed beside the block)
    a.x = ptr(x); a.weight = static_cast<float*>(ptr(w)); a.bias = fptr<float>(b); a.out = ptr(out);
}
Tensor conv_fwd(const Tensor& x, const Tensor& weight, const OptT& bias, bool silu, OptT out, int64_t stream) {
    REQUIRE(kScan, x.dim() == 3, "x must be (batch, dim, seqlen), got " + shape_str(x.sizes()));
    const auto [w, b] = conv_params(weight, bias, x.size(1), x.device(), x.scalar_type());
    const int32_t wd = dtype_code(w);
    if (!out) out = at::empty(x.sizes(), x.options());
    REQUIRE(kScan, out->sizes() == x.sizes() && out->scalar_type() == x.scalar_type() && unit(*out),
            "out must match x in shape and dtype, with unit stride along seqlen");
    ss_conv1d_args a;
    fill_conv(a, x, w, b, silu, out);
    launch(x.device(), "causal_conv1d_fwd", [&] { return ss_conv1d_fwd_typed(&a, wd, reinterpret_cast<void*>(stream)); });
    return *out;
}
// (dx, dweight (dim, width), dbias): in fp32, summed by atomics or, when
// deterministic, in a fixed order; with `typed`, of the weight's and bias's
// own types where the library writes them (fixed order, one launch for both).
py::tuple conv_bwd(const Tensor& x, const Tensor& weight, const OptT& bias, const Tensor& dout_, bool silu, OptT dx,
                   bool deterministic, bool typed, int64_t stream) {
    REQUIRE(kScan, x.dim() == 3, "x must be (batch, dim, seqlen), got " + shape_str(x.sizes()));
    const auto [w, b] = typed ? conv_params(weight, bias, x.size(1), x.device(), x.scalar_type())
                              : conv_params(weight, bias, x.size(1), x.device());
    const int32_t wd = dtype_code(w);
    REQUIRE(kScan, dout_.sizes() == x.sizes() && dout_.scalar_type() == x.scalar_type(),
            "dout must match x in shape and dtype");
    const Tensor dout = seq_unit(dout_);
    if (!dx) dx = at::empty(x.sizes(), x.options());
    const bool zero = !typed || x.numel() == 0;
    const Tensor dw = at::empty(w.sizes(), w.options());
    const OptT db = b ? OptT(at::empty(b->sizes(), b->options())) : OptT();
    if (zero) {
        dw.zero_();
        if (db) db->zero_();
    }
    ss_conv1d_bwd_args g{};
    fill_conv(g.f, x, w, b, silu, OptT());
    g.dout_batch_stride = dout.stride(0); g.dout_dim_stride = dout.stride(1);
    g.dx_batch_stride = dx->stride(0); g.dx_dim_stride = dx->stride(1);
    g.dout = ptr(dout); g.dx = ptr(*dx); g.dweight = static_cast<float*>(ptr(dw)); g.dbias = fptr<float>(db);
    OptT ws;
    if (deterministic || typed) {
        const int64_t n = ss_conv1d_bwd_workspace_bytes(&g);
        REQUIRE(kScan, n >= 0, "invalid conv1d sizes");
        ws = f32_like({std::max<int64_t>(n / 4, 1)}, x);
        g.workspace = static_cast<float*>(ptr(*ws));
        g.workspace_bytes = ws->numel() * 4;
    }
    launch(x.device(), "causal_conv1d_bwd", [&] {
        void* st = reinterpret_cast<void*>(stream);
        return typed ? ss_conv1d_bwd_typed(&g, wd, st) : ss_conv1d_bwd(&g, st);
    });
    return py::make_tuple(*dx, dw, db);
}

// --------------------------------------------------------------- RMSNorm --
constexpr const char* kNorm = "rms_norm";

// (rows, dim) view with unit column stride (a copy only when no such view exists)
Tensor norm_rows(const Tensor& t_, int64_t dim) {
    const Tensor t = dim > 1 && t_.stride(-1) != 1 ? t_.contiguous() : t_;
    const Tensor v = t.dim() == 2 && dim > 0 && t.size(1) == dim ? t : t.reshape({-1, dim});
    return dim > 1 && v.stride(1) != 1 ? v.contiguous() : v;
}
Tensor norm_weight(const Tensor& w, const Tensor& x) {
    REQUIRE(kNorm, w.dim() == 1 && w.size(0) == x.size(-1),
            "weight must be (" + std::to_string(x.size(-1)) + ",), got " + shape_str(w.sizes()));
    REQUIRE(kNorm, w.device() == x.device(), "weight is on " + w.device().str() + ", x on " + x.device().str());
    return (w.scalar_type() == x.scalar_type() || w.scalar_type() == at::kFloat ? w : w.to(at::kFloat)).contiguous();
}
py::tuple norm_fwd(const Tensor& x, const Tensor& weight, const OptT& residual, double eps, bool want_rstd, bool want_s,
                   int64_t stream) {
    REQUIRE(kNorm, x.is_cuda(), "tensors must be on a ROCm GPU device (no CPU path)");
    ss_rmsnorm_args a{};
    REQUIRE(kNorm, itype_of(x.scalar_type(), &a.dtype), "unsupported dtype " + dtype_str(x.scalar_type()));
    REQUIRE(kNorm, x.dim() >= 1, "x must have at least one dimension");
    const int64_t dim = x.size(-1);
    const Tensor w = norm_weight(weight, x), x2 = norm_rows(x, dim);
    itype_of(w.scalar_type(), &a.w_dtype);
    OptT r2, rout, rstd;
    if (residual) {
        REQUIRE(kNorm, residual->sizes() == x.sizes() && residual->scalar_type() == x.scalar_type() &&
                           residual->device() == x.device(),
                "residual must match x in shape, dtype and device");
        r2 = norm_rows(*residual, dim);
    }
    const Tensor out = at::empty(x2.sizes(), x.options());
    if (r2 && want_s) rout = at::empty_like(out);
    if (want_rstd) rstd = f32_like({x2.size(0)}, x);
    a.rows = x2.size(0); a.dim = dim;
    a.eps = float(eps);
    a.x_row_stride = x2.stride(0); a.out_row_stride = out.stride(0);
    if (r2) {
        a.residual_row_stride = r2->stride(0);
        if (rout) a.residual_out_row_stride = rout->stride(0);
    }
    a.x = ptr(x2); a.residual = ptr(r2); a.weight = ptr(w);
    a.out = ptr(out); a.residual_out = ptr(rout); a.rstd = fptr<float>(rstd);
    launch(x.device(), "rms_norm forward", [&] { return ss_rmsnorm_fwd(&a, reinterpret_cast<void*>(stream)); });
    return py::make_tuple(out, rout, rstd);
}
py::tuple norm_bwd(const Tensor& s, const Tensor& weight, const Tensor& rstd, const Tensor& dout,
                   const OptT& dresidual_out, int64_t stream) {
    const int64_t dim = s.size(-1);
    const Tensor w = norm_weight(weight, s), s2 = norm_rows(s, dim), dy = norm_rows(dout.to(s.scalar_type()), dim);
    const OptT dr = dresidual_out ? OptT(norm_rows(dresidual_out->to(s.scalar_type()), dim)) : OptT();
    const int64_t rows = s2.size(0);
    REQUIRE(kNorm, dy.sizes() == s2.sizes() && (!dr || dr->sizes() == s2.sizes()), "dout must match s");
    REQUIRE(kNorm, rstd.scalar_type() == at::kFloat && same_shape(rstd, {rows}) && rstd.is_contiguous(),
            "rstd must be fp32 (rows,) contiguous");
    const Tensor dx = at::empty(s2.sizes(), s.options()), dw = at::empty({dim}, w.options());
    const int64_t n = ss_rmsnorm_bwd_workspace_bytes(rows, dim);
    const Tensor ws = bytes_on(std::max<int64_t>(n, 1), s);
    ss_rmsnorm_bwd_args g{};
    g.rows = rows; g.dim = dim;
    REQUIRE(kNorm, itype_of(s.scalar_type(), &g.dtype) && itype_of(w.scalar_type(), &g.w_dtype),
            "unsupported dtype " + dtype_str(s.scalar_type()));
    g.s_row_stride = s2.stride(0); g.dout_row_stride = dy.stride(0); g.dx_row_stride = dx.stride(0);
    if (dr) g.dresidual_out_row_stride = dr->stride(0);
    g.s = ptr(s2); g.weight = ptr(w); g.rstd = static_cast<float*>(ptr(rstd)); g.dout = ptr(dy); g.dresidual_out = ptr(dr);
    g.dx = ptr(dx); g.dweight = ptr(dw); g.workspace = ptr(ws); g.workspace_bytes = n;
    launch(s.device(), "rms_norm backward", [&] { return ss_rmsnorm_bwd(&g, reinterpret_cast<void*>(stream)); });
    return py::make_tuple(dx, dw);
}

// ---------------------------------------------------------------- decode --
bool mult(const Tensor& t, int64_t stride0, size_t align) {
    return t.stride(0) % stride0 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % align == 0;
}
// the shapes ss_decode_linear takes (others run on torch's library GEMM)
bool linear_fits(const Tensor& x, const Tensor& weight, const OptT& bias, int64_t max_rows) {
    return x.is_cuda() && x.dim() == 2 && (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf) &&
           weight.scalar_type() == x.scalar_type() && weight.dim() == 2 && weight.size(1) == x.size(1) &&
           x.size(1) % 16 == 0 && 0 < x.size(0) && x.size(0) <= max_rows && x.stride(1) == 1 &&
           weight.stride(1) == 1 && mult(x, 4, 8) && mult(weight, 4, 8) &&
           (!bias || ((bias->scalar_type() == x.scalar_type() || bias->scalar_type() == at::kFloat) &&
                      bias->is_contiguous()));
}
bool linear_norm_fits(const Tensor& x, const OptT& residual, const Tensor& nw) {
    const auto rows16 = [](const Tensor& t) { return t.stride(1) == 1 && mult(t, 8, 16); };
    return x.size(1) <= 1024 && rows16(x) &&
           (!residual || (residual->sizes() == x.sizes() && residual->scalar_type() == x.scalar_type() &&
                          rows16(*residual))) &&
           nw.dim() == 1 && nw.size(0) == x.size(1) &&
           (nw.scalar_type() == x.scalar_type() || nw.scalar_type() == at::kFloat) && nw.is_contiguous() &&
           reinterpret_cast<uintptr_t>(nw.data_ptr()) % 16 == 0;
}
// Workspace bytes of the K split for a product of these sizes.
int64_t linear_ws_bytes(int64_t batch, int64_t n_out, int64_t k_in) {
    ss_decode_linear_args a{};
    a.batch = batch; a.n_out = n_out; a.k_in = k_in;
    return ss_decode_linear_workspace_bytes(&a);
}
// The fused launch for fitting tensors: (y, s or None).
py::tuple linear(const Tensor& x, const Tensor& weight, const OptT& bias, bool has_conv, const OptT& conv_state,
                 const OptT& conv_w, const OptT& conv_b, bool silu, bool has_norm, const OptT& residual,
                 const OptT& nw, double eps, const OptT& ws, int64_t stream) {
    const int64_t batch = x.size(0), k_in = x.size(1), n_out = weight.size(0);
    const Tensor y = at::empty({batch, n_out}, x.options());
    ss_decode_linear_args a{};
    a.batch = batch; a.n_out = n_out; a.k_in = k_in;
    itype_of(x.scalar_type(), &a.dtype);
    a.bias_dtype = a.dtype;
    if (bias) itype_of(bias->scalar_type(), &a.bias_dtype);
    a.x_row_stride = x.stride(0); a.w_row_stride = weight.stride(0); a.y_row_stride = y.stride(0);
    a.x = ptr(x); a.weight = ptr(weight); a.bias = ptr(bias); a.y = ptr(y);
    ss_conv1d_update_args c{};
    Tensor w;
    OptT cb;
    if (has_conv) {
        REQUIRE(kScan, conv_state && conv_w, "conv_state and the conv weight are required");
        const int64_t dim = conv_state->size(1);
        std::tie(w, cb) = conv_params(*conv_w, conv_b, dim, x.device());
        REQUIRE(kScan, conv_state->dim() == 3 && same_shape(*conv_state, {batch, dim, w.size(1)}) &&
                           conv_state->scalar_type() == x.scalar_type() && conv_state->device() == x.device() &&
                           dim <= n_out,
                "conv_state must be (" + std::to_string(batch) + ", dim <= " + std::to_string(n_out) +
                    ", width) of x's dtype, got " + shape_str(conv_state->sizes()));
        c.batch = batch; c.dim = dim; c.width = w.size(1);
        c.itype = a.dtype; c.has_bias = cb.has_value(); c.silu = silu;
        c.state_batch_stride = conv_state->stride(0);
        c.state_dim_stride = conv_state->stride(1);
        c.state_width_stride = conv_state->stride(2);
        c.w_dim_stride = w.stride(0); c.w_width_stride = w.stride(1);
        c.conv_state = ptr(*conv_state); c.weight = static_cast<float*>(ptr(w)); c.bias = fptr<float>(cb);
        a.conv = &c;
    }
    ss_rmsnorm_args n{};
    OptT s;
    if (has_norm) {
        s = residual ? at::empty_like(x) : x;
        n.rows = batch; n.dim = k_in;
        n.dtype = a.dtype;
        itype_of(nw->scalar_type(), &n.w_dtype);
        n.eps = float(eps);
        n.x_row_stride = x.stride(0);
        if (residual) {
            n.residual_row_stride = residual->stride(0);
            n.residual_out_row_stride = s->stride(0);
            n.residual = ptr(*residual);
            n.residual_out = ptr(*s);
        }
        n.x = ptr(x); n.weight = ptr(*nw);
        a.norm = &n;
        a.x = nullptr;
        a.x_row_stride = 0;
    }
    if (ws && ss_decode_linear_workspace_bytes(&a) > 0) {
        a.workspace = ptr(*ws);
        a.workspace_bytes = ws->numel();
    }
    launch(x.device(), "decode_linear", [&] { return ss_decode_linear(&a, reinterpret_cast<void*>(stream)); });
    return py::make_tuple(y, s);
}

constexpr const char* kState = "selective_state_update";

Tensor state_update(const Tensor& state, const Tensor& x, const OptT& dt, const OptT& dt_low, const OptT& dt_w,
                    const Tensor& A, const Tensor& B_, const Tensor& C_, const OptT& D, const OptT& z,
                    const OptT& dt_bias, bool softplus, OptT out, int64_t stream) {
    REQUIRE(kState, x.dim() == 2 && x.is_cuda(), "x must be (batch, dim) on a ROCm GPU device (no CPU path)");
    ss_state_update_args a{};
    REQUIRE(kState, itype_of(x.scalar_type(), &a.itype), "unsupported dtype " + dtype_str(x.scalar_type()));
    const int64_t batch = x.size(0), dim = x.size(1);
    const at::Device dev = x.device();
    const at::ScalarType ty = x.scalar_type();
    const auto num = [](int64_t v) { return std::to_string(v); };
    REQUIRE(kState, state.dim() == 3 && state.size(0) == batch && state.size(1) == dim &&
                        state.scalar_type() == at::kFloat && state.device() == dev,
            "state must be fp32 (" + num(batch) + ", " + num(dim) + ", dstate)");
    const int64_t n = state.size(2);
    if (dt_low) {
        REQUIRE(kState, dt_low->dim() == 2 && dt_low->size(0) == batch && dt_low->scalar_type() == ty &&
                            dt_low->device() == dev,
                "dt_low must be (batch, rank) in x's dtype");
        REQUIRE(kState, dt_w.has_value(), "dt_weight is required with dt_low");
        REQUIRE(kState, same_shape(*dt_w, {dim, dt_low->size(1)}) && dt_w->scalar_type() == ty && dt_w->device() == dev,
                "dt_weight must be (dim, rank) in x's dtype");
    } else {
        REQUIRE(kState, dt.has_value(), "dt is required");
        REQUIRE(kState, dt->sizes() == x.sizes() && dt->scalar_type() == ty, "dt must match x in shape and dtype");
    }
    REQUIRE(kState, same_shape(A, {dim, n}), "A must be (" + num(dim) + ", " + num(n) + ")");
    const Tensor A32 = A.to(dev, at::kFloat);
    const Tensor B = B_.dim() == 2 ? B_.unsqueeze(1) : B_, C = C_.dim() == 2 ? C_.unsqueeze(1) : C_;
    REQUIRE(kState, B.dim() == 3 && B.size(0) == batch && B.size(2) == n && B.scalar_type() == ty,
            "B must be (batch, [n_groups,] dstate) in x's dtype");
    REQUIRE(kState, C.sizes() == B.sizes() && C.scalar_type() == ty, "C must match B");
    REQUIRE(kState, B.size(1) > 0 && dim % B.size(1) == 0,
            "dim " + num(dim) + " is not a multiple of n_groups " + num(B.size(1)));
    const OptT D32 = D ? OptT(D->to(dev, at::kFloat).contiguous()) : OptT();
    const OptT b32 = dt_bias ? OptT(dt_bias->to(dev, at::kFloat).contiguous()) : OptT();
    REQUIRE(kState, !D32 || same_shape(*D32, {dim}), "D must be (" + num(dim) + ",)");
    REQUIRE(kState, !b32 || same_shape(*b32, {dim}), "dt_bias must be (" + num(dim) + ",)");
    REQUIRE(kState, !z || (z->sizes() == x.sizes() && z->scalar_type() == ty), "z must match x");
    if (!out) out = at::empty({batch, dim}, x.options());
    a.batch = batch; a.dim = dim; a.dstate = n; a.n_groups = B.size(1);
    a.has_D = D32.has_value(); a.has_z = z.has_value(); a.has_delta_bias = b32.has_value();
    a.delta_softplus = softplus;
    a.state_batch_stride = state.stride(0); a.state_dim_stride = state.stride(1); a.state_dstate_stride = state.stride(2);
    a.x_batch_stride = x.stride(0); a.x_dim_stride = x.stride(1);
    if (dt_low) {
        a.delta_rank = dt_low->size(1);
        a.delta_low_batch_stride = dt_low->stride(0); a.delta_low_rank_stride = dt_low->stride(1);
        a.delta_weight_dim_stride = dt_w->stride(0); a.delta_weight_rank_stride = dt_w->stride(1);
        a.delta_low = ptr(*dt_low); a.delta_weight = ptr(*dt_w);
    } else {
        a.delta_batch_stride = dt->stride(0); a.delta_dim_stride = dt->stride(1);
        a.delta = ptr(*dt);
    }
    if (z) a.z_batch_stride = z->stride(0), a.z_dim_stride = z->stride(1);
    a.out_batch_stride = out->stride(0); a.out_dim_stride = out->stride(1);
    a.A_dim_stride = A32.stride(0); a.A_dstate_stride = A32.stride(1);
    a.B_batch_stride = B.stride(0); a.B_group_stride = B.stride(1); a.B_dstate_stride = B.stride(2);
    a.C_batch_stride = C.stride(0); a.C_group_stride = C.stride(1); a.C_dstate_stride = C.stride(2);
    a.state = static_cast<float*>(ptr(state)); a.x = ptr(x); a.A = static_cast<float*>(ptr(A32));
    a.B = ptr(B); a.C = ptr(C); a.D = fptr<float>(D32); a.z = ptr(z); a.delta_bias = fptr<float>(b32); a.out = ptr(*out);
    launch(dev, "selective_state_update", [&] { return ss_state_update(&a, reinterpret_cast<void*>(stream)); });
    return *out;
}

}  // namespace

PYBIND11_MODULE(mamba_host, m) {
    // argument blocks at an address (ctypes structures of the prepared launches and queries)
    m.def("fill_fwd_into", [](uintptr_t at, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B,
                              const Tensor& C, const OptT& D, const OptT& bias, bool softplus, const OptT& out,
                              const OptT& x, const OptT& z, const OptT& y, const OptT& last) {
        fill_fwd_into(*reinterpret_cast<ss_fwd_args*>(at), u, delta, A, B, C, D, bias, softplus, out, x, z, y, last);
    });
    m.def("fill_bwd", [](uintptr_t at, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B,
                         const Tensor& C, const OptT& D, const OptT& bias, const Tensor& dout, const OptT& x,
                         bool softplus, const Tensor& du, const Tensor& ddelta, const OptT& dA, const OptT& dB,
                         const OptT& dC, const OptT& dD, const OptT& dbias, const OptT& z, const OptT& y,
                         const OptT& dz) {
        fill_bwd(*reinterpret_cast<ss_bwd_args*>(at), u, delta, A, B, C, D, bias, dout, x, softplus, du, ddelta, dA,
                 dB, dC, dD, dbias, z, y, dz);
    });
    m.def("scan_fwd", &scan_fwd);
    m.def("scan_z_fwd", &scan_z_fwd);
    m.def("scan_bwd", &scan_bwd);
    m.def("scan_bwd_new", &scan_bwd_new);
    m.def("conv_fwd", &conv_fwd);
    m.def("conv_bwd", &conv_bwd);
    m.def("norm_fwd", &norm_fwd);
    m.def("norm_bwd", &norm_bwd);
    m.def("linear_fits", &linear_fits);
    m.def("linear_norm_fits", &linear_norm_fits);
    m.def("linear_ws_bytes", &linear_ws_bytes);
    m.def("linear", &linear);
    m.def("state_update", &state_update);
    m.def("abi", [] { return py::make_tuple(SS_ABI_VERSION, sizeof(ss_fwd_args), sizeof(ss_bwd_args)); });
}
