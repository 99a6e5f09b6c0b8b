// Python entry points of the operator on the host: argument checks, output and scratch allocation,
// and the calls of libdwoconv1d_hip.so on the tensors' device and current stream.
//
// What bounds a call on small tensors is this path (the stage convolutions of ConvNeXt-T at batch
// 64 take 216 us of GPU time in 12 kernels).  Kept in Python, with one ctypes call, one device query,
// one stream object and up to four tensor constructions per kernel, forward and backward of one
// layer took 90 to 170 us of host time, hence native code, without the GIL.  For ordinary tensors the
// autograd function is native as well (Convolution below): as a Python one its backward pass took the GIL on the
// engine's device thread while the caller waited for it, and the stage convolutions of ConvNeXt-T, forward and backward,
// took 190 or 380 us of wall time from process to process for the same 186 us of kernels.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/extension.h>

#include <stdexcept>
#include <string>
#include <tuple>

#include "dwoconv1d_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// the entry points of the library that the Python side has loaded
struct Library {
    decltype(&::dwo_status_string) status_string;
    decltype(&::dwo_taps_bytes) taps_bytes;
    decltype(&::dwo_fprop) fprop;
    decltype(&::dwo_dgrad) dgrad;
    decltype(&::dwo_wgrad_scratch_bytes) wgrad_scratch_bytes;
    decltype(&::dwo_wgrad) wgrad;
    decltype(&::dwo_layernorm_nhwc) layernorm_nhwc;
    decltype(&::dwo_nchw_layernorm_nhwc) nchw_layernorm_nhwc;
    decltype(&::dwo_nhwc_scale_add_nchw) nhwc_scale_add_nchw;
    decltype(&::dwo_pointwise_wgrad_scratch_bytes) pointwise_wgrad_scratch_bytes;
    decltype(&::dwo_pointwise_wgrad) pointwise_wgrad;
    decltype(&::dwo_block_scratch_bytes) block_scratch_bytes;
    decltype(&::dwo_ln_rows) ln_rows;
    decltype(&::dwo_ln_rows_backward) ln_rows_backward;
    decltype(&::dwo_ln_tile) ln_tile;
    decltype(&::dwo_ln_tile_backward) ln_tile_backward;
    decltype(&::dwo_block_tail) block_tail;
    decltype(&::dwo_block_tail_backward) block_tail_backward;
    decltype(&::dwo_linear_wgrad_scratch_bytes) linear_wgrad_scratch_bytes;
    decltype(&::dwo_linear_wgrad) linear_wgrad;
    decltype(&::dwo_ln_patch) ln_patch;
    decltype(&::dwo_ln_patch_backward) ln_patch_backward;
    decltype(&::dwo_pointwise_forward) pointwise_forward;
    decltype(&::dwo_block_mlp) block_mlp;
    decltype(&::dwo_linear_rows) linear_rows;
    decltype(&::dwo_linear_planes) linear_planes;
    decltype(&::dwo_linear_norm_planes) linear_norm_planes;
} lib;

[[noreturn]] void fail(const std::string &msg) { throw std::runtime_error(msg); }

void bind_library(const std::string &path) {
    void *h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (h == nullptr) fail(dlerror());
    auto find = [h](auto &fn, const char *name) {
        fn = reinterpret_cast<std::decay_t<decltype(fn)>>(dlsym(h, name));
        if (fn == nullptr) fail(std::string("missing symbol ") + name);
    };
    find(lib.status_string, "dwo_status_string");
    find(lib.taps_bytes, "dwo_taps_bytes");
    find(lib.fprop, "dwo_fprop");
    find(lib.dgrad, "dwo_dgrad");
    find(lib.wgrad_scratch_bytes, "dwo_wgrad_scratch_bytes");
    find(lib.wgrad, "dwo_wgrad");
    find(lib.layernorm_nhwc, "dwo_layernorm_nhwc");
    find(lib.nchw_layernorm_nhwc, "dwo_nchw_layernorm_nhwc");
    find(lib.nhwc_scale_add_nchw, "dwo_nhwc_scale_add_nchw");
    find(lib.pointwise_wgrad_scratch_bytes, "dwo_pointwise_wgrad_scratch_bytes");
    find(lib.pointwise_wgrad, "dwo_pointwise_wgrad");
    find(lib.block_scratch_bytes, "dwo_block_scratch_bytes");
    find(lib.ln_rows, "dwo_ln_rows");
    find(lib.ln_rows_backward, "dwo_ln_rows_backward");
    find(lib.ln_tile, "dwo_ln_tile");
    find(lib.ln_tile_backward, "dwo_ln_tile_backward");
    find(lib.block_tail, "dwo_block_tail");
    find(lib.block_tail_backward, "dwo_block_tail_backward");
    find(lib.linear_wgrad_scratch_bytes, "dwo_linear_wgrad_scratch_bytes");
    find(lib.linear_wgrad, "dwo_linear_wgrad");
    find(lib.ln_patch, "dwo_ln_patch");
    find(lib.ln_patch_backward, "dwo_ln_patch_backward");
    find(lib.pointwise_forward, "dwo_pointwise_forward");
    find(lib.block_mlp, "dwo_block_mlp");
    find(lib.linear_rows, "dwo_linear_rows");
    find(lib.linear_planes, "dwo_linear_planes");
    find(lib.linear_norm_planes, "dwo_linear_norm_planes");
}

void check(int status, const char *what) {
    if (status != 0)
        fail(std::string(what) + " failed: " + lib.status_string(status) + " (status " +
             std::to_string(status) + ")");
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return DWO_F32;
        case at::kBFloat16: return DWO_BF16;
        case at::kHalf: return DWO_F16;
        default: return -1;
    }
}

int dtype_code(const Tensor &t) { return dtype_code(t.scalar_type()); }

// models/dwoconv1d/kernels/kernels.cu:11-13,17-18
void check_activation(const Tensor &t, const char *name) {
    if (!t.is_cuda()) fail(std::string(name) + " must be a CUDA tensor");
    if (!t.is_contiguous()) fail(std::string(name) + " must be contiguous");
    if (dtype_code(t) < 0)
        {
            py::gil_scoped_acquire gil;
            fail(std::string(name) + " has unsupported dtype " +
                 py::cast<std::string>(py::str(py::cast(t).attr("dtype"))));
        }
    if (t.dim() != 4) fail(std::string(name) + " must be a 4-d tensor");
}

void check_taps(const Tensor &taps, int64_t C, int64_t K) {
    const int64_t want = (int64_t)lib.taps_bytes((int)C, (int)K);
    if (taps.scalar_type() != at::kByte || taps.numel() != want)
        fail("tap table does not match C=" + std::to_string(C) + ", K=" + std::to_string(K) + " (" +
             std::to_string(taps.numel()) + " bytes, expected " + std::to_string(want) + ")");
}

// extents of the input side; sizes beyond int32 saturate, which the library refuses
struct Dims {
    int64_t n, c, h, w;
    Dims(const Tensor &t, bool nhwc)
        : n(t.size(0)), c(t.size(nhwc ? 3 : 1)), h(t.size(nhwc ? 1 : 2)), w(t.size(nhwc ? 2 : 3)) {}
};
int as_int(int64_t v) { return v > 0x7fffffff ? 0x7fffffff : (int)v; }
int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

std::array<int64_t, 4> shape_of(int64_t n, int64_t c, int64_t h, int64_t w, bool nhwc) {
    if (nhwc) return {n, h, w, c};
    return {n, c, h, w};
}

void check_stride(int64_t stride) {
    if (stride != 1 && stride != 2 && stride != 4) fail(lib.status_string(DWO_ERR_BAD_STRIDE));
}

// the weights as [C, K] fp32 rows
Tensor rows_f32(const Tensor &w, int64_t C) {
    if (w.scalar_type() == at::kFloat && w.is_contiguous() && C > 0 && w.numel() % C == 0 && w.numel() > 0)
        return w;
    return w.detach().reshape({C, -1}).to(at::kFloat).contiguous();
}

const void *ptr(const Tensor &t) { return t.const_data_ptr(); }
const float *fptr(const OptTensor &t) {
    return t.has_value() ? reinterpret_cast<const float *>(t->const_data_ptr()) : nullptr;
}

// the tensor's device made current, and the current stream there
struct Place {
    c10::OptionalDeviceGuard guard;
    void *stream;
    explicit Place(const Tensor &t) : guard(t.device()) {
        stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    }
};

Tensor fprop(const Tensor &x, const Tensor &w, const Tensor &taps, int64_t stride, const OptTensor &bias,
             int64_t layout) {
    const bool nhwc = layout & DWO_NHWC;
    check_activation(x, "x");
    check_stride(stride);
    const Dims d(x, nhwc);
    const Tensor w2 = rows_f32(w, d.c);
    const int64_t K = w2.numel() / std::max<int64_t>(d.c, 1);
    check_taps(taps, d.c, K);
    const Place at(x);
    Tensor y = at::empty(shape_of(d.n, d.c, up(d.h, stride), up(d.w, stride), nhwc), x.options());
    check(lib.fprop(ptr(x), (const float *)ptr(w2), fptr(bias), ptr(taps), y.data_ptr(), as_int(d.n),
                    as_int(d.c), as_int(d.h), as_int(d.w), as_int(K), as_int(stride), dtype_code(x), (int)layout,
                    at.stream),
          "dwo_fprop");
    return y;
}

Tensor dgrad(const Tensor &dy, const Tensor &w, const Tensor &taps, int64_t H, int64_t W, int64_t stride,
             int64_t layout) {
    const bool nhwc = layout & DWO_NHWC;
    check_activation(dy, "dy");
    check_stride(stride);
    const Dims d(dy, nhwc);
    if (d.h != up(H, stride) || d.w != up(W, stride)) fail("dy extent does not match the input extent and stride");
    const Tensor w2 = rows_f32(w, d.c);
    const int64_t K = w2.numel() / std::max<int64_t>(d.c, 1);
    check_taps(taps, d.c, K);
    const Place at(dy);
    Tensor dx = at::empty(shape_of(d.n, d.c, H, W, nhwc), dy.options());
    check(lib.dgrad(ptr(dy), (const float *)ptr(w2), ptr(taps), dx.data_ptr(), as_int(d.n), as_int(d.c),
                    as_int(H), as_int(W), as_int(K), as_int(stride), dtype_code(dy), (int)layout, at.stream),
          "dwo_dgrad");
    return dx;
}

std::tuple<Tensor, OptTensor> wgrad(const Tensor &dy, const Tensor &x, const Tensor &taps, int64_t K,
                                    int64_t stride, int64_t layout, bool with_bias) {
    const bool nhwc = layout & DWO_NHWC;
    check_activation(dy, "dy");
    check_activation(x, "x");
    check_stride(stride);
    if (dy.scalar_type() != x.scalar_type()) fail("dy and x must have the same dtype");
    const Dims d(x, nhwc);
    const auto want = shape_of(d.n, d.c, up(d.h, stride), up(d.w, stride), nhwc);
    if (dy.sizes() != at::IntArrayRef(want)) fail("dy extent does not match the input extent and stride");
    check_taps(taps, d.c, K);
    const Place at(x);
    const int n = as_int(d.n), c = as_int(d.c), h = as_int(d.h), wd = as_int(d.w), k = as_int(K),
              s = as_int(stride), dt = dtype_code(x);
    const size_t nbytes = lib.wgrad_scratch_bytes(n, c, h, wd, k, s, dt, (int)layout);
    const Tensor scratch = at::empty({(int64_t)std::max<size_t>(nbytes, 16)}, x.options().dtype(at::kByte));
    const auto f32 = x.options().dtype(at::kFloat);
    Tensor dw = at::empty({d.c, 1, 1, K}, f32);
    OptTensor db;
    if (with_bias) db = at::empty({d.c}, f32);
    check(lib.wgrad(ptr(dy), ptr(x), ptr(taps), (float *)dw.data_ptr(), db.has_value() ? (float *)db->data_ptr() : nullptr,
                    scratch.data_ptr(), nbytes, n, c, h, wd, k, s, dt, (int)layout, at.stream),
          "dwo_wgrad");
    return {dw, db};
}

// the same for callers that hold the GIL
Tensor fprop_entry(const Tensor &x, const Tensor &w, const Tensor &taps, int64_t stride, const OptTensor &bias,
                   int64_t layout) {
    py::gil_scoped_release nogil;
    return fprop(x, w, taps, stride, bias, layout);
}
Tensor dgrad_entry(const Tensor &dy, const Tensor &w, const Tensor &taps, int64_t H, int64_t W, int64_t stride,
                   int64_t layout) {
    py::gil_scoped_release nogil;
    return dgrad(dy, w, taps, H, W, stride, layout);
}
std::tuple<Tensor, OptTensor> wgrad_entry(const Tensor &dy, const Tensor &x, const Tensor &taps, int64_t K,
                                          int64_t stride, int64_t layout, bool with_bias) {
    py::gil_scoped_release nogil;
    return wgrad(dy, x, taps, K, stride, layout, with_bias);
}

// The operator as a node of autograd (the contract of models/dwoconv1d/dwoconv1d.py:18-69): gradients of x, w and bias, none
// of theta, which is an input all the same: data-parallel wrappers wait for every parameter that takes gradients and
// is not part of the graph.  w32 and bias32 are fp32 copies where the parameters are not dense fp32 themselves; resid is added to the weights.
struct Convolution : torch::autograd::Function<Convolution> {
    using Context = torch::autograd::AutogradContext;
    using List = torch::autograd::variable_list;

    static Tensor forward(Context *ctx, const Tensor &x_, const Tensor &w, const OptTensor &bias, const OptTensor &w32,
                          const OptTensor &bias32, const OptTensor &resid, const Tensor &taps, const Tensor & /*theta*/,
                          int64_t stride, int64_t layout) {
        ctx->set_materialize_grads(false);
        const Tensor x = x_.contiguous();
        Tensor weights = w32.has_value() ? *w32 : w;
        if (resid.has_value()) weights = weights + resid->to(weights.options());
        ctx->save_for_backward({x, weights, taps});
        const bool has_bias = bias.has_value();
        ctx->saved_data["p"] = std::vector<int64_t>{
            stride, layout, w.size(-1), (int64_t)w.scalar_type(), has_bias ? (int64_t)bias->scalar_type() : -1};
        return fprop(x, weights, taps, stride, bias32.has_value() ? bias32 : bias, layout);
    }

    static List backward(Context *ctx, const List &grads) {
        List out(10);
        if (!grads[0].defined()) return out;
        const List saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &weights = saved[1], &taps = saved[2];
        const std::vector<int64_t> p = ctx->saved_data["p"].toIntVector();
        const int64_t stride = p[0], layout = p[1], K = p[2];
        const auto w_type = (at::ScalarType)p[3];
        const bool nhwc = layout & DWO_NHWC, has_bias = p[4] >= 0, need_db = has_bias && ctx->needs_input_grad(2);
        Tensor dy = grads[0].contiguous();
        if (dy.scalar_type() != x.scalar_type()) dy = dy.to(x.scalar_type());
        if (ctx->needs_input_grad(0))
            out[0] = dgrad(dy, weights, taps, x.size(nhwc ? 1 : 2), x.size(nhwc ? 2 : 3), stride, layout);
        if (ctx->needs_input_grad(1)) {
            auto [dw, db] = wgrad(dy, x, taps, K, stride, layout, need_db);
            out[1] = dw.scalar_type() == w_type ? dw : dw.to(w_type);
            if (need_db) out[2] = db->to((at::ScalarType)p[4]);
        } else if (need_db) {
            out[2] = dy.sum(nhwc ? at::IntArrayRef{0, 1, 2} : at::IntArrayRef{0, 2, 3}, false, at::kFloat)
                         .to((at::ScalarType)p[4]);
        }
        return out;
    }
};

Tensor convolution(const Tensor &x, const Tensor &w, const OptTensor &bias, const OptTensor &w32,
                   const OptTensor &bias32, const OptTensor &resid, const Tensor &taps, const Tensor &theta,
                   int64_t stride, int64_t layout) {
    py::gil_scoped_release nogil;
    return Convolution::apply(x, w, bias, w32, bias32, resid, taps, theta, stride, layout);
}

void check_glue(const Tensor &t, const char *name) {
    if (!t.is_cuda() || dtype_code(t) < 0)
        fail(std::string(name) + " must be a CUDA tensor of type float32, bfloat16 or float16");
}

// gamma, beta or a layer scale, which the kernels read as C dense floats
void check_channels(const Tensor &x, const Tensor &p, int64_t C, const char *name) {
    if (p.device() != x.device() || p.scalar_type() != at::kFloat || !p.is_contiguous() || p.numel() != C)
        fail(std::string(name) + " must be " + std::to_string(C) + " contiguous float32 values on x's device");
}
void check_norm(const Tensor &x, const Tensor &g, const Tensor &b, int64_t C) {
    check_channels(x, g, C, "weight");
    check_channels(x, b, C, "bias");
}

Tensor layernorm_nhwc(const Tensor &x_, const Tensor &g, const Tensor &b, double eps, bool gelu) {
    check_glue(x_, "x");
    if (x_.dim() < 1) fail("x must have a dimension of channels");
    check_norm(x_, g, b, x_.size(-1));
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = x_.contiguous();
    const int64_t C = x.size(-1);
    Tensor out = at::empty_like(x);
    check(lib.layernorm_nhwc(ptr(x), (const float *)ptr(g), (const float *)ptr(b), out.data_ptr(),
                             (size_t)(x.numel() / std::max<int64_t>(C, 1)), as_int(C), (float)eps, gelu,
                             dtype_code(x), at.stream),
          "dwo_layernorm_nhwc");
    return out;
}

Tensor nchw_layernorm_nhwc(const Tensor &x_, const Tensor &g, const Tensor &b, double eps) {
    check_glue(x_, "x");
    if (x_.dim() != 4) throw py::value_error("x must be a 4-d tensor");
    check_norm(x_, g, b, x_.size(1));
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = x_.contiguous();
    const Dims d(x, false);
    Tensor out = at::empty({d.n, d.h, d.w, d.c}, x.options());
    check(lib.nchw_layernorm_nhwc(ptr(x), (const float *)ptr(g), (const float *)ptr(b), out.data_ptr(),
                                  as_int(d.n), as_int(d.c), as_int(d.h), as_int(d.w), (float)eps, dtype_code(x),
                                  at.stream),
          "dwo_nchw_layernorm_nhwc");
    return out;
}

Tensor nhwc_scale_add_nchw(const Tensor &y_, const OptTensor &scale, const OptTensor &residual) {
    check_glue(y_, "y");
    if (y_.dim() != 4) throw py::value_error("y must be a 4-d tensor");
    if (scale.has_value()) check_channels(y_, *scale, y_.size(3), "scale");
    py::gil_scoped_release nogil;
    const Place at(y_);
    const Tensor y = y_.contiguous();
    const Dims d(y, true);
    Tensor res;
    if (residual.has_value()) {
        const std::array<int64_t, 4> want = {d.n, d.c, d.h, d.w};
        if (residual->sizes() != at::IntArrayRef(want) || residual->scalar_type() != y.scalar_type())
            fail("residual must be [N,C,H,W] of the same type as y");
        res = residual->contiguous();
    }
    Tensor out = at::empty({d.n, d.c, d.h, d.w}, y.options());
    check(lib.nhwc_scale_add_nchw(ptr(y), fptr(scale), res.defined() ? ptr(res) : nullptr, out.data_ptr(),
                                  as_int(d.n), as_int(d.c), as_int(d.h), as_int(d.w), dtype_code(y), at.stream),
          "dwo_nhwc_scale_add_nchw");
    return out;
}

// dy [.., C] and x [.., Cin] of one type, contiguous
std::tuple<Tensor, OptTensor> pointwise_wgrad(const Tensor &dy, const Tensor &x, bool with_bias) {
    check_glue(dy, "dy");
    if (!dy.is_contiguous() || !x.is_contiguous() || x.device() != dy.device() ||
        dy.scalar_type() != x.scalar_type())
        fail("dy and x must be contiguous, on one device and of one type");
    if (dy.dim() < 1 || x.dim() != dy.dim() || x.sizes().slice(0, x.dim() - 1) != dy.sizes().slice(0, dy.dim() - 1))
        fail("dy and x must have the same pixels");
    const int64_t C = dy.size(-1), Cin = x.size(-1);
    py::gil_scoped_release nogil;
    const Place at(dy);
    const size_t nbytes = lib.pointwise_wgrad_scratch_bytes(as_int(Cin), as_int(C));
    const Tensor scratch = at::empty({(int64_t)std::max<size_t>(nbytes, 16)}, dy.options().dtype(at::kByte));
    const auto f32 = dy.options().dtype(at::kFloat);
    Tensor dw = at::empty({C, Cin}, f32);
    OptTensor db;
    if (with_bias) db = at::empty({C}, f32);
    check(lib.pointwise_wgrad(ptr(dy), ptr(x), (float *)dw.data_ptr(),
                              db.has_value() ? (float *)db->data_ptr() : nullptr, scratch.data_ptr(), nbytes,
                              (size_t)(dy.numel() / std::max<int64_t>(C, 1)), as_int(Cin), as_int(C),
                              dtype_code(dy), at.stream),
          "dwo_pointwise_wgrad");
    return {dw, db};
}

// dense and 16-byte aligned, as the block's kernels read and write (a gradient may be a piece of another buffer)
Tensor dense(const Tensor &t) {
    Tensor d = t.contiguous();
    if (reinterpret_cast<uintptr_t>(d.const_data_ptr()) % 16 != 0) d = d.clone();
    return d;
}
void check_pair(const Tensor &a, const Tensor &b) {
    if (a.device() != b.device()) fail("tensors on different devices");
}
Tensor bytes(const Tensor &like, size_t n) {
    return at::empty({(int64_t)std::max<size_t>(n, 16)}, like.options().dtype(at::kByte));
}

// dy [.., N] and x [.., K] of one 16-bit type -> dw [N, K], db [N] of grad_dtype
std::tuple<Tensor, OptTensor> linear_wgrad(const Tensor &dy_, const Tensor &x_, bool with_bias,
                                           at::ScalarType grad_dtype) {
    check_glue(dy_, "dy");
    check_glue(x_, "x");
    check_pair(dy_, x_);
    if (dy_.scalar_type() != x_.scalar_type()) fail("dy and x must have the same dtype");
    if (dy_.dim() < 1 || x_.dim() != dy_.dim() ||
        x_.sizes().slice(0, x_.dim() - 1) != dy_.sizes().slice(0, dy_.dim() - 1))
        fail("dy and x must have the same rows");
    py::gil_scoped_release nogil;
    const Place at(dy_);
    const Tensor dy = dense(dy_), x = dense(x_);
    const int64_t N = dy.size(-1), K = x.size(-1), rows = dy.numel() / std::max<int64_t>(N, 1);
    const size_t nbytes = lib.linear_wgrad_scratch_bytes((size_t)rows, as_int(N), as_int(K));
    const Tensor scratch = bytes(dy, nbytes);
    const auto opt = dy.options().dtype(grad_dtype);
    Tensor dw = at::empty({N, K}, opt);
    OptTensor db;
    if (with_bias) db = at::empty({N}, opt);
    check(lib.linear_wgrad(ptr(dy), ptr(x), dw.data_ptr(), db.has_value() ? db->data_ptr() : nullptr,
                           scratch.data_ptr(), nbytes, (size_t)rows, as_int(N), as_int(K), dtype_code(dy),
                           dtype_code(grad_dtype), at.stream),
          "dwo_linear_wgrad");
    return {dw, db};
}

const void *optr(const OptTensor &t) { return t.has_value() ? t->const_data_ptr() : nullptr; }
void check_layer(const Tensor &x, const Tensor &w) {
    check_glue(x, "x");
    check_pair(x, w);
    if (w.dim() != 2 || w.size(1) != x.size(-1) || w.scalar_type() != x.scalar_type())
        fail("w must be [N, K] of the same type as x");
}
// a bias or layer scale of n values of x's type, dense (a parameter may be a view with a stride)
OptTensor dense_values(const Tensor &x, const OptTensor &t, int64_t n, const char *name) {
    if (!t.has_value()) return t;
    check_pair(x, *t);
    if (t->numel() != n || t->scalar_type() != x.scalar_type())
        fail(std::string(name) + " must be " + std::to_string(n) + " values of the same type as x");
    return t->contiguous();
}

// x [.., Cin] -> [.., C]: x w^T + b, all of one type
Tensor pointwise_forward(const Tensor &x_, const Tensor &w_, const OptTensor &b_) {
    check_layer(x_, w_);
    py::gil_scoped_release nogil;
    const Place at(x_);
    const OptTensor b = dense_values(x_, b_, w_.size(0), "bias");
    const Tensor x = x_.contiguous(), w = w_.contiguous();
    auto shape = x.sizes().vec();
    shape.back() = w.size(0);
    Tensor y = at::empty(shape, x.options());
    check(lib.pointwise_forward(ptr(x), ptr(w), optr(b), y.data_ptr(), (size_t)(x.numel() / std::max<int64_t>(w.size(1), 1)),
                                as_int(w.size(1)), as_int(w.size(0)), dtype_code(x), at.stream),
          "dwo_pointwise_forward");
    return y;
}

// LayerNorm (+ GELU) over the last dimension; (out, stats)
std::tuple<Tensor, OptTensor> ln_rows(const Tensor &x_, const Tensor &g, const Tensor &b, double eps, int64_t gelu,
                                      at::ScalarType out_dtype, bool with_stats) {
    check_glue(x_, "x");
    if (x_.dim() < 1) fail("x must have a dimension of channels");
    check_norm(x_, g, b, x_.size(-1));
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = dense(x_);
    const int64_t C = x.size(-1), rows = x.numel() / std::max<int64_t>(C, 1);
    Tensor out = at::empty(x.sizes(), x.options().dtype(out_dtype));
    OptTensor stats;
    if (with_stats) stats = at::empty({rows, 2}, x.options().dtype(at::kFloat));
    check(lib.ln_rows(ptr(x), (const float *)ptr(g), (const float *)ptr(b), out.data_ptr(),
                      stats.has_value() ? (float *)stats->data_ptr() : nullptr, (size_t)rows, as_int(C), (float)eps, (int)gelu, dtype_code(x), dtype_code(out_dtype), at.stream),
          "dwo_ln_rows");
    return {out, stats};
}

std::tuple<Tensor, Tensor, Tensor> ln_rows_backward(const Tensor &dout_, const Tensor &x_, const Tensor &stats,
                                                    const Tensor &g, const Tensor &b, int64_t gelu,
                                                    at::ScalarType grad_dtype) {
    check_glue(dout_, "dout");
    check_glue(x_, "x");
    check_pair(dout_, x_);
    if (dout_.sizes() != x_.sizes()) fail("dout and x must have the same shape");
    check_norm(x_, g, b, x_.size(-1));
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = dense(x_), dout = dense(dout_);
    const int64_t C = x.size(-1), rows = x.numel() / std::max<int64_t>(C, 1);
    const size_t nbytes = lib.block_scratch_bytes(as_int(C));
    const Tensor scratch = bytes(x, nbytes);
    Tensor dx = at::empty(x.sizes(), x.options());
    Tensor dg = at::empty({C}, x.options().dtype(grad_dtype)), db = at::empty({C}, dg.options());
    check(lib.ln_rows_backward(ptr(dout), ptr(x), (const float *)ptr(stats), (const float *)ptr(g),
                               (const float *)ptr(b), dx.data_ptr(), dg.data_ptr(), db.data_ptr(), scratch.data_ptr(),
                               nbytes, (size_t)rows, as_int(C), (int)gelu, dtype_code(x), dtype_code(dout),
                               dtype_code(grad_dtype), at.stream),
          "dwo_ln_rows_backward");
    return {dx, dg, db};
}

// [N,C,H,W] -> LayerNorm over C -> [N,H,W,C], or with `patches` [N,H/2,W/2,4C]; (out, stats)
std::tuple<Tensor, OptTensor> ln_tile(const Tensor &x_, const Tensor &g, const Tensor &b, double eps, bool patches,
                                      at::ScalarType out_dtype, bool with_stats) {
    check_glue(x_, "x");
    if (x_.dim() != 4) throw py::value_error("x must be a 4-d tensor");
    check_norm(x_, g, b, x_.size(1));
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = dense(x_);
    const Dims d(x, false);
    const std::array<int64_t, 4> shape = patches ? std::array<int64_t, 4>{d.n, d.h / 2, d.w / 2, 4 * d.c}
                                                 : std::array<int64_t, 4>{d.n, d.h, d.w, d.c};
    Tensor out = at::empty(shape, x.options().dtype(out_dtype));
    OptTensor stats;
    if (with_stats) stats = at::empty({out.numel() / std::max<int64_t>(d.c, 1), 2}, x.options().dtype(at::kFloat));
    check((patches ? lib.ln_patch : lib.ln_tile)(ptr(x), (const float *)ptr(g), (const float *)ptr(b), out.data_ptr(),
                                                 stats.has_value() ? (float *)stats->data_ptr() : nullptr, as_int(d.n),
                                                 as_int(d.c), as_int(d.h), as_int(d.w), (float)eps, dtype_code(x),
                                                 dtype_code(out_dtype), at.stream),
          patches ? "dwo_ln_patch" : "dwo_ln_tile");
    return {out, stats};
}

std::tuple<Tensor, Tensor, Tensor> ln_tile_backward(const Tensor &dout_, const Tensor &x_, const Tensor &stats,
                                                    const Tensor &g, bool patches, at::ScalarType grad_dtype) {
    check_glue(dout_, "dout");
    check_glue(x_, "x");
    check_pair(dout_, x_);
    const Dims d(x_, false);
    check_channels(x_, g, d.c, "weight");
    const std::array<int64_t, 4> want = patches ? std::array<int64_t, 4>{d.n, d.h / 2, d.w / 2, 4 * d.c}
                                                : std::array<int64_t, 4>{d.n, d.h, d.w, d.c};
    if (dout_.sizes() != at::IntArrayRef(want)) fail("dout does not match x");
    py::gil_scoped_release nogil;
    const Place at(x_);
    const Tensor x = dense(x_), dout = dense(dout_);
    const size_t nbytes = lib.block_scratch_bytes(as_int(d.c));
    const Tensor scratch = bytes(x, nbytes);
    // (an odd last row or column is in no patch)
    Tensor dx = patches && (d.h % 2 != 0 || d.w % 2 != 0) ? at::zeros(x.sizes(), x.options()) : at::empty(x.sizes(), x.options());
    Tensor dg = at::empty({d.c}, x.options().dtype(grad_dtype)), db = at::empty({d.c}, dg.options());
    check((patches ? lib.ln_patch_backward : lib.ln_tile_backward)(
              ptr(dout), ptr(x), (const float *)ptr(stats), (const float *)ptr(g), dx.data_ptr(), dg.data_ptr(),
              db.data_ptr(), scratch.data_ptr(), nbytes, as_int(d.n), as_int(d.c), as_int(d.h), as_int(d.w),
              dtype_code(x), dtype_code(dout), dtype_code(grad_dtype), at.stream),
          patches ? "dwo_ln_patch_backward" : "dwo_ln_tile_backward");
    return {dx, dg, db};
}

// res + scale * y as planes of out_dtype: y [N,H,W,C], res [N,C,H,W]
Tensor block_tail(const Tensor &y_, const OptTensor &scale, const OptTensor &res_, at::ScalarType out_dtype,
                  bool rounded) {
    check_glue(y_, "y");
    if (y_.dim() != 4) throw py::value_error("y must be a 4-d tensor");
    const Dims d(y_, true);
    if (scale.has_value()) check_channels(y_, *scale, d.c, "scale");
    const std::array<int64_t, 4> shape = {d.n, d.c, d.h, d.w};
    if (res_.has_value()) {
        check_glue(*res_, "res");
        check_pair(y_, *res_);
        if (res_->sizes() != at::IntArrayRef(shape)) fail("res must be [N,C,H,W]");
    }
    py::gil_scoped_release nogil;
    const Place at(y_);
    const Tensor y = dense(y_);
    Tensor res, out = at::empty(shape, y.options().dtype(out_dtype));
    if (res_.has_value()) res = dense(*res_);
    check(lib.block_tail(ptr(y), fptr(scale), res.defined() ? ptr(res) : nullptr, out.data_ptr(), as_int(d.n),
                         as_int(d.c), as_int(d.h), as_int(d.w), rounded, dtype_code(y),
                         res.defined() ? dtype_code(res) : dtype_code(out_dtype), dtype_code(out_dtype), at.stream),
          "dwo_block_tail");
    return out;
}

// dout [N,C,H,W] -> (dy [N,H,W,C] of y_dtype, dscale); without y only dy
std::tuple<Tensor, OptTensor> block_tail_backward(const Tensor &dout_, const OptTensor &y_, const OptTensor &scale,
                                                  at::ScalarType y_dtype, at::ScalarType grad_dtype) {
    check_glue(dout_, "dout");
    if (dout_.dim() != 4) throw py::value_error("dout must be a 4-d tensor");
    const Dims d(dout_, false);
    if (scale.has_value()) check_channels(dout_, *scale, d.c, "scale");
    const std::array<int64_t, 4> shape = {d.n, d.h, d.w, d.c};
    if (y_.has_value()) {
        check_glue(*y_, "y");
        check_pair(dout_, *y_);
        if (y_->sizes() != at::IntArrayRef(shape) || y_->scalar_type() != y_dtype) fail("y does not match dout");
    }
    py::gil_scoped_release nogil;
    const Place at(dout_);
    const Tensor dout = dense(dout_);
    Tensor y, scratch, dy = at::empty(shape, dout.options().dtype(y_dtype));
    OptTensor ds;
    size_t nbytes = 0;
    if (y_.has_value()) {
        y = dense(*y_);
        nbytes = lib.block_scratch_bytes(as_int(d.c));
        scratch = bytes(y, nbytes);
        ds = at::empty({d.c}, y.options().dtype(grad_dtype));
    }
    check(lib.block_tail_backward(ptr(dout), y.defined() ? ptr(y) : nullptr, fptr(scale), dy.data_ptr(),
                                  ds.has_value() ? ds->data_ptr() : nullptr,
                                  scratch.defined() ? scratch.data_ptr() : nullptr, nbytes, as_int(d.n), as_int(d.c),
                                  as_int(d.h), as_int(d.w), dtype_code(y_dtype), dtype_code(dout),
                                  dtype_code(grad_dtype), at.stream),
          "dwo_block_tail_backward");
    return {dy, ds};
}

// act(x w^T + b) over the last dimension
Tensor linear_rows(const Tensor &x_, const Tensor &w_, const OptTensor &b_, bool gelu) {
    check_layer(x_, w_);
    py::gil_scoped_release nogil;
    const Place at(x_);
    const OptTensor b = dense_values(x_, b_, w_.size(0), "bias");
    const Tensor x = dense(x_), w = dense(w_);
    const int64_t N = w.size(0), K = w.size(1);
    auto shape = x.sizes().vec();
    shape.back() = N;
    Tensor out = at::empty(shape, x.options());
    check(lib.linear_rows(ptr(x), ptr(w), optr(b), out.data_ptr(), (size_t)(x.numel() / std::max<int64_t>(K, 1)),
                          as_int(N), as_int(K), gelu, dtype_code(x), at.stream),
          "dwo_linear_rows");
    return out;
}

// x [N,H,W,K] -> [N,C,H,W]: res + scale * (x w^T + b)
Tensor linear_planes(const Tensor &x_, const Tensor &w_, const OptTensor &b_, const OptTensor &scale_,
                     const OptTensor &res_) {
    check_layer(x_, w_);
    if (x_.dim() != 4) throw py::value_error("x must be a 4-d tensor");
    const int64_t C = w_.size(0), K = w_.size(1);
    const Dims d(x_, true);
    py::gil_scoped_release nogil;
    const Place at(x_);
    const OptTensor b = dense_values(x_, b_, C, "bias"), scale = dense_values(x_, scale_, C, "scale");
    const Tensor x = dense(x_), w = dense(w_);
    Tensor out = at::empty({d.n, C, d.h, d.w}, x.options()), res;
    if (res_.has_value()) {
        check_pair(x_, *res_);
        if (res_->sizes() != out.sizes() || res_->scalar_type() != x.scalar_type())
            fail("residual must be [N,C,H,W] of the same type as x");
        res = dense(*res_);
    }
    check(lib.linear_planes(ptr(x), ptr(w), optr(b), optr(scale), res.defined() ? ptr(res) : nullptr, out.data_ptr(),
                            as_int(d.n), as_int(d.h * d.w), as_int(C), as_int(K), dtype_code(x), at.stream),
          "dwo_linear_planes");
    return out;
}

// x [N,H,W,K] -> [N,C,H,W]: LayerNorm over C (fp32 g and beta) of z w^T + b with z = GELU(LayerNorm over K of x)
Tensor linear_norm_planes(const Tensor &x_, const Tensor &g_in, const Tensor &beta_in, double eps_in, const Tensor &w_,
                          const OptTensor &b_, const Tensor &g, const Tensor &beta, double eps) {
    check_layer(x_, w_);
    if (x_.dim() != 4) throw py::value_error("x must be a 4-d tensor");
    const int64_t C = w_.size(0), K = w_.size(1);
    check_norm(x_, g, beta, C);
    check_norm(x_, g_in, beta_in, K);
    const Dims d(x_, true);
    py::gil_scoped_release nogil;
    const Place at(x_);
    const OptTensor b = dense_values(x_, b_, C, "bias");
    const Tensor x = dense(x_), w = dense(w_);
    Tensor out = at::empty({d.n, C, d.h, d.w}, x.options());
    check(lib.linear_norm_planes(ptr(x), (const float *)ptr(g_in), (const float *)ptr(beta_in), (float)eps_in, ptr(w), optr(b), (const float *)ptr(g),
                                 (const float *)ptr(beta), (float)eps, out.data_ptr(), as_int(d.n), as_int(d.h * d.w),
                                 as_int(C), as_int(K), dtype_code(x), at.stream),
          "dwo_linear_norm_planes");
    return out;
}

// x [N,H,W,C], res [N,C,H,W] -> res + scale * (w2 gelu(w1 x + b1) + b2), planes
Tensor block_mlp(const Tensor &x_, const Tensor &w1_, const Tensor &b1_, const Tensor &w2_, const Tensor &b2_,
                 const OptTensor &scale_, const Tensor &res_) {
    check_layer(x_, w1_);
    if (x_.dim() != 4) throw py::value_error("x must be a 4-d tensor");
    const int64_t C = x_.size(3);
    if (w1_.size(0) != 4 * C || w2_.dim() != 2 || w2_.size(0) != C || w2_.size(1) != 4 * C ||
        w2_.scalar_type() != x_.scalar_type())
        fail("w1 must be [4C, C] and w2 [C, 4C], of the same type as x");
    const Dims d(x_, true);
    const std::array<int64_t, 4> shape = {d.n, d.c, d.h, d.w};
    if (res_.sizes() != at::IntArrayRef(shape) || res_.scalar_type() != x_.scalar_type())
        fail("residual must be [N,C,H,W] of the same type as x");
    check_pair(x_, w2_), check_pair(x_, res_);
    py::gil_scoped_release nogil;
    const Place at(x_);
    const OptTensor b1 = dense_values(x_, b1_, 4 * C, "first bias"), b2 = dense_values(x_, b2_, C, "second bias"),
                    scale = dense_values(x_, scale_, C, "scale");
    const Tensor x = dense(x_), w1 = dense(w1_), w2 = dense(w2_), c1 = dense(*b1), res = dense(res_);
    Tensor out = at::empty(shape, x.options());
    check(lib.block_mlp(ptr(x), ptr(w1), ptr(c1), ptr(w2), optr(b2), optr(scale), ptr(res), out.data_ptr(), as_int(d.n),
                        as_int(d.h * d.w), as_int(C), dtype_code(x), at.stream),
          "dwo_block_mlp");
    return out;
}

// [N,C,H,W] -> operator (NCHW, stride 1; fp32 weights and bias) -> LayerNorm over C -> [N,H,W,C], without gradients (`pieces`: by
// ln_tile)
Tensor conv_norm(const Tensor &x, const Tensor &w, const OptTensor &bias, const Tensor &taps, const Tensor &g,
                 const Tensor &b, double eps, bool pieces) {
    const Tensor y = fprop_entry(x, w, taps, 1, bias, DWO_NCHW);
    return pieces ? std::get<0>(ln_tile(y, g, b, eps, false, y.scalar_type(), false)) : nchw_layernorm_nhwc(y, g, b, eps);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    m.def("bind", &bind_library);
    m.def("convolution", &convolution);
    m.def("fprop", &fprop_entry);
    m.def("dgrad", &dgrad_entry);
    m.def("wgrad", &wgrad_entry);
    m.def("pointwise_wgrad", &pointwise_wgrad);
    m.def("layernorm_nhwc", &layernorm_nhwc);
    m.def("nchw_layernorm_nhwc", &nchw_layernorm_nhwc);
    m.def("nhwc_scale_add_nchw", &nhwc_scale_add_nchw);
    m.def("linear_wgrad", &linear_wgrad);
    m.def("pointwise_forward", &pointwise_forward);
    m.def("block_mlp", &block_mlp);
    m.def("conv_norm", &conv_norm);
    m.def("linear_rows", &linear_rows);
    m.def("linear_planes", &linear_planes);
    m.def("linear_norm_planes", &linear_norm_planes);
    m.def("ln_rows", &ln_rows);
    m.def("ln_rows_backward", &ln_rows_backward);
    m.def("ln_tile", &ln_tile);
    m.def("ln_tile_backward", &ln_tile_backward);
    m.def("block_tail", &block_tail);
    m.def("block_tail_backward", &block_tail_backward);
}
