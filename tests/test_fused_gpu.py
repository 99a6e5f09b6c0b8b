"""The forward-only glue kernels against the PyTorch passes they replace
(models/convnext.py:306-318 and :176-190): LayerNorm over channels with and without the layout
change, exact GELU, layer scale + transpose + residual.  Tolerances: fp32 1e-5, 16-bit 1e-2
(tensor-level, as for the operator)."""
import pytest
import torch
import torch.nn.functional as F

from parity_util import TOL, rel_err

from oriented1d_amd import fused

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _close(got, ref, dtype, what):
    e_max, e_l2 = rel_err(got.float().cpu().numpy(), ref.double().cpu().numpy())
    assert e_max <= TOL[dtype] and e_l2 <= TOL[dtype], (what, e_max, e_l2)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("N,C,H,W", [(2, 96, 56, 56), (3, 192, 28, 28), (2, 384, 14, 14),
                                     (2, 768, 7, 7), (1, 1024, 7, 7), (2, 64, 9, 13), (1, 6, 3, 5)])
def test_nchw_layernorm_nhwc(N, C, H, W, dtype):
    torch.manual_seed(C + H)
    x = (torch.randn(N, C, H, W, device="cuda") * 2 + 0.5).to(dtype)
    g = torch.randn(C, device="cuda") * 0.5 + 1
    b = torch.randn(C, device="cuda") * 0.1
    got = fused.nchw_layernorm_nhwc(x, g, b, 1e-6)
    ref = F.layer_norm(x.double().permute(0, 2, 3, 1), (C,), g.double(), b.double(), 1e-6)
    assert got.shape == (N, H, W, C) and got.dtype == dtype and got.is_contiguous()
    _close(got, ref, dtype, "nchw_layernorm_nhwc")


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("shape", [(2, 112, 112, 64), (3, 14, 14, 384), (5, 7, 7, 1536), (7, 2048),
                                   (1, 3, 5, 2)])
def test_layernorm_nhwc(shape, gelu, dtype):
    torch.manual_seed(shape[-1])
    C = shape[-1]
    x = (torch.randn(*shape, device="cuda") * 3 - 0.25).to(dtype)
    g = torch.randn(C, device="cuda") * 0.5 + 1
    b = torch.randn(C, device="cuda") * 0.1
    got = fused.layernorm_nhwc(x, g, b, 1e-6, gelu=gelu)
    ref = F.layer_norm(x.double(), (C,), g.double(), b.double(), 1e-6)
    if gelu:
        ref = F.gelu(ref)
    assert got.shape == x.shape and got.dtype == dtype
    _close(got, ref, dtype, "layernorm_nhwc")


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("with_scale,with_res", [(True, True), (False, False), (True, False)])
@pytest.mark.parametrize("N,C,H,W", [(2, 96, 56, 56), (2, 768, 7, 7), (3, 64, 9, 13), (1, 1536, 2, 3)])
def test_nhwc_scale_add_nchw(N, C, H, W, with_scale, with_res, dtype):
    torch.manual_seed(C + W)
    y = torch.randn(N, H, W, C, device="cuda").to(dtype)
    s = torch.randn(C, device="cuda") if with_scale else None
    r = torch.randn(N, C, H, W, device="cuda").to(dtype) if with_res else None
    got = fused.nhwc_scale_add_nchw(y, s, r)
    ref = y.double()
    if with_scale:
        ref = ref * s.double()
    ref = ref.permute(0, 3, 1, 2)
    if with_res:
        ref = ref + r.double()
    assert got.shape == (N, C, H, W) and got.is_contiguous()
    _close(got, ref, dtype, "nhwc_scale_add_nchw")


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("Cin,C,H,W,K,stride", [(3, 64, 64, 48, 31, 2), (3, 24, 37, 29, 15, 2),
                                               (4, 8, 20, 20, 7, 1), (1, 16, 33, 70, 31, 4),
                                               (3, 64, 224, 224, 31, 2)])  # the stem's own shape
def test_pointwise_then_oriented_conv(oracle, Cin, C, H, W, K, stride, dtype):
    """dwo_pointwise_fprop_nhwc against the two separate layers: nn.Linear Cin -> C rounded to
    the activation type (what the reference's pw1 hands to dw1, models/convnext.py:177-178),
    then the oracle's fprop with bias."""
    import numpy as np
    from parity_util import grouped_theta, rounded
    from oriented1d_amd.dwoconv1d import DepthwiseOrientedConv1d

    torch.manual_seed(Cin * 100 + C)
    lin = torch.nn.Linear(Cin, C).cuda()
    conv = DepthwiseOrientedConv1d(C, C, K, groups=C, stride=stride, padding=K // 2, bias=True,
                                   angle=grouped_theta(C).tolist(), nhwc=True).cuda()
    torch.nn.init.normal_(conv.bias, std=0.3)
    x = torch.randn(2, H, W, Cin, device="cuda").to(dtype)
    with torch.no_grad():
        got = fused.pointwise_dwconv_nhwc(x, lin, conv)
    mid = x.double().cpu().numpy() @ lin.weight.detach().double().cpu().numpy().T \
        + lin.bias.detach().double().cpu().numpy()
    mid = rounded(mid.astype(np.float32), dtype)  # the separate layer's output in the tensor's type
    ref = oracle.fprop(np.ascontiguousarray(mid.transpose(0, 3, 1, 2)),
                       conv.weight.detach().cpu().numpy(), conv.theta.detach().cpu().numpy(), stride)
    ref = ref + conv.bias.detach().double().cpu().numpy().reshape(1, -1, 1, 1)
    P, Q = -(-H // stride), -(-W // stride)
    assert got.shape == (2, P, Q, C) and got.dtype == dtype
    _close(got.permute(0, 3, 1, 2), torch.from_numpy(ref), dtype, "pointwise_fprop")


def test_argument_errors():
    x = torch.randn(2, 7, 4, 4, device="cuda")  # odd channel count
    with pytest.raises(RuntimeError):
        fused.nchw_layernorm_nhwc(x, torch.ones(7), torch.zeros(7), 1e-6)
    assert not fused.usable(x, 7, tiled=True)
    assert not fused.usable(torch.randn(2, 8, 4, 4), 8, tiled=True)  # CPU tensor
    w = torch.randn(2, 8, 4, 4, device="cuda", requires_grad=True)
    assert not fused.usable(w, 8, tiled=True)
    with torch.no_grad():
        assert fused.usable(w, 8, tiled=True)


def _composed(m, x, monkeypatch):
    """m(x) with PyTorch's passes around the operator: gradient recording switches the inference kernels off, and what is not
    ordinary execution the training kernels."""
    with monkeypatch.context() as patch:
        patch.setattr(fused, "ordinary", lambda *tensors: False)
        return m(x.detach().requires_grad_(True)).detach()


@pytest.mark.parametrize("variant", ["1d", "1dpp"])
def test_block_and_stem_fused_equal_unfused(variant, monkeypatch):
    """Block-level parity: the harness in no-grad eval mode (fused glue) against the same
    modules as PyTorch composes them."""
    from oriented1d_amd.convnext1d import ConvNeXt1D

    torch.manual_seed(3)
    m = ConvNeXt1D(depths=(1, 1, 1, 1), dims=(16, 32, 64, 128), variant=variant, stem_dim1=24,
                   num_classes=10, layer_scale_init_value=1.0).cuda().eval()
    for name, p in m.named_parameters():
        if name.endswith("bias") or "norm" in name:
            torch.nn.init.normal_(p, mean=0.3, std=0.2)
    x = torch.randn(2, 3, 64, 64, device="cuda")
    with torch.no_grad():
        y_fused = m(x)
    y_plain = _composed(m, x, monkeypatch)
    _close(y_fused, y_plain, torch.float32, "network")


def test_bf16_network_fused_equal_unfused_and_parameter_copies_refresh(monkeypatch):
    """The 16-bit network (parameters cast with .bfloat16(): the library works from cached fp32
    copies of them) with and without the glue kernels, and the copies follow in-place updates."""
    from oriented1d_amd.convnext1d import ConvNeXt1D

    torch.manual_seed(4)
    m = ConvNeXt1D(depths=(1, 1, 1, 1), dims=(16, 32, 64, 128), variant="1d", stem_dim1=24,
                   num_classes=10, layer_scale_init_value=1.0).cuda().bfloat16().eval()
    x = torch.randn(2, 3, 64, 64, device="cuda").bfloat16()
    with torch.no_grad():
        y_fused = m(x)
    y_plain = _composed(m, x, monkeypatch)
    _close(y_fused, y_plain, torch.bfloat16, "bf16 network")
    with torch.no_grad():
        m.stages[0][0].dwconv.weight.mul_(3.0)   # in-place update: the cached copy must refresh
        y_fused2 = m(x)
    y_plain2 = _composed(m, x, monkeypatch)
    _close(y_fused2, y_plain2, torch.bfloat16, "bf16 network after update")
    assert not torch.equal(y_fused, y_fused2)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape,cin", [((1, 1, 1, 8), 1), ((2, 9, 13, 64), 3), ((1, 40, 50, 24), 2),
                                       ((2, 224, 224, 64), 3), ((1, 7, 5, 1024), 4)])
def test_pointwise_linear_gradients(shape, cin, dtype):
    """dw and db of a layer with few inputs; sums of P terms in fp32 in another order: the bound is
    the rounding of the largest partial sums, sqrt(P) * 2^-24 relative to the sums' own spread
    sqrt(P), far below 1e-5; 16-bit results are rounded once."""
    torch.manual_seed(cin)
    C = shape[-1]
    x = torch.randn(*shape[:-1], cin, device="cuda").to(dtype)
    lin = torch.nn.Linear(cin, C).cuda().to(dtype)
    dy = torch.randn(*shape, device="cuda").to(dtype)
    y = fused.pointwise_linear(x, lin)
    assert torch.equal(y, lin(x)) and type(y.grad_fn).__name__ == "_PointwiseLinearBackward"
    dw, db = torch.autograd.grad(y, (lin.weight, lin.bias), dy)
    rows, xs = dy.double().reshape(-1, C), x.double().reshape(-1, cin)
    _close(dw, rows.t() @ xs, dtype, "dw")
    _close(db, rows.sum(0), dtype, "db")
    # gradients of gradients, input gradients and a view of another buffer: as nn.Linear has them
    xg, buf = x.clone().requires_grad_(), torch.cat([dy.reshape(-1)[:1], dy.reshape(-1)])
    odd = buf[1:].view(shape)
    for layer in (fused.pointwise_linear, lambda a, m: m(a)):
        g = torch.autograd.grad(layer(xg, lin), (xg, lin.weight, lin.bias), odd, create_graph=True)
        gg = torch.autograd.grad(g[1].double().sum(), xg)[0]
        if layer is fused.pointwise_linear:
            first = g + (gg,)
    for a, b in zip(first, g + (gg,)):
        _close(a.detach(), b.detach(), dtype, "second order")


def test_pointwise_linear_second_order_under_autocast():
    """d(sum of dw) / dx under autocast: dw is linear in x, so it is the upstream gradient's channel sum."""
    torch.manual_seed(0)
    x = torch.randn(2, 5, 7, 3, device="cuda", requires_grad=True)
    lin = torch.nn.Linear(3, 64).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = fused.pointwise_linear(x, lin)
    dy = torch.randn(y.shape, device="cuda").to(torch.bfloat16).requires_grad_()
    dw = torch.autograd.grad(y, lin.weight, dy, create_graph=True)[0]
    gx = torch.autograd.grad(dw.sum(), x)[0]
    _close(gx, dy.detach().double().sum(-1, keepdim=True).expand(x.shape), torch.bfloat16, "autocast second order")


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("C,H,W,K", [(64, 1, 1, 7), (64, 33, 66, 31), (64, 65, 131, 15), (128, 18, 5, 13),
                                     (64, 97, 70, 27), (64, 2, 200, 31)])
def test_projected_stem_tile_edges(C, H, W, K, dtype):
    """The projecting kernel at the edges of its tiles, and where the claim of common orientations does
    not hold (mixed angles behind it), against the two separate layers."""
    from parity_util import canonical_theta, grouped_theta
    from oriented1d_amd.dwoconv1d import DepthwiseOrientedConv1d

    torch.manual_seed(H)
    lin = torch.nn.Linear(3, C).cuda()
    x = torch.randn(2, H, W, 3, device="cuda").to(dtype)
    for theta, claimed in ((grouped_theta(C), False), (canonical_theta(C), True)):
        conv = DepthwiseOrientedConv1d(C, C, K, groups=C, stride=2, padding=K // 2, bias=True, angle=theta.tolist(),
                                       nhwc=True, arbitrary_size=True).cuda()
        torch.nn.init.normal_(conv.bias, std=0.3)
        if claimed:
            look = conv._taps.lookup
            conv._taps.lookup = lambda *a: (look(*a)[0], {2: 3, 4: 3})
        with torch.no_grad():
            got = fused.pointwise_dwconv_nhwc(x, lin, conv)
            if claimed:
                conv._taps.lookup = look
            mid = torch.nn.functional.linear(x.double(), lin.weight.double(), lin.bias.double()).to(dtype)
            _close(got, conv(mid), dtype, "projected")


@pytest.mark.parametrize("N,C,H,W,K", [(40, 64, 66, 131, 31), (30, 64, 97, 70, 15), (1700, 64, 5, 13, 7), (1200, 64, 2, 59, 27),
                                       (3, 128, 260, 201, 31), (40000, 64, 1, 1, 13)])
def test_projected_stem_as_products(N, C, H, W, K):
    """The stem's matrix products at the edges of their tiles against the two layers in 64 and 32 bits: nothing but the
    result is rounded to bf16 (2^-9 of a value, 1e-2 is the operator's bound)."""
    from oriented1d_amd.convnext1d import channel_angles
    from oriented1d_amd.dwoconv1d import DepthwiseOrientedConv1d

    torch.manual_seed(H)
    lin = torch.nn.Linear(3, C).cuda()
    x = torch.randn(N, H, W, 3, device="cuda").to(torch.bfloat16)
    conv = DepthwiseOrientedConv1d(C, C, K, groups=C, stride=2, padding=K // 2, bias=True, angle=channel_angles(C),
                                   nhwc=True, arbitrary_size=True).cuda()
    torch.nn.init.normal_(conv.bias, std=0.3)
    with torch.no_grad():
        def layers(rounded):
            mid = torch.nn.functional.linear(x.double(), lin.weight.double(), lin.bias.double())
            return conv(mid.to(torch.bfloat16 if rounded else torch.float32))
        _close(fused.pointwise_dwconv_nhwc(x, lin, conv), layers(False), torch.bfloat16, "products")
        # a claim of common orientations that does not hold, infinities and NaN: tap by tap
        look = conv._taps.lookup
        mixed = DepthwiseOrientedConv1d(C, C, K, groups=C, stride=2, padding=K // 2, bias=True, nhwc=True,
                                        angle=[c % 8 * 0.39 for c in range(C)], arbitrary_size=True).cuda()
        conv._taps.lookup = lambda *a: (mixed._taps.lookup(mixed.theta, *a[1:])[0], {2: 3, 4: 3})
        got = fused.pointwise_dwconv_nhwc(x, lin, conv)
        conv._taps.lookup = look
        mixed.weight.copy_(conv.weight), mixed.bias.copy_(conv.bias)
        mid = torch.nn.functional.linear(x.double(), lin.weight.double(), lin.bias.double()).to(torch.bfloat16)
        _close(got, mixed(mid), torch.bfloat16, "mixed orientations")
        x[0, 0, 0, 0], x[-1, -1, -1, 2] = float("inf"), float("nan")
        got, ref = fused.pointwise_dwconv_nhwc(x, lin, conv), layers(True)
        # (the grouped kernels add up the weights of taps that meet on a pixel, inf (w1 + w2) for inf w1 + inf w2: an
        # infinity there may be NaN here)
        assert torch.equal(got.isfinite(), ref.isfinite())


@pytest.mark.parametrize("dtype", DTYPES[1:], ids=["bf16", "f16"])
def test_pointwise_linear_leaves_the_autocast_cache_alone(dtype):
    """Two passes of one autocast region, the second on an input that is differentiated itself (it stays
    with PyTorch, which takes the region's cached low-precision parameters): both give the parameters
    their gradients, as nn.Linear does, in either order."""
    torch.manual_seed(1)
    lin = torch.nn.Linear(3, 64).cuda()
    x, xg = torch.randn(2, 2, 9, 11, 3, device="cuda").unbind(0)
    xg = xg.clone().requires_grad_()
    dy = torch.randn(2, 9, 11, 64, device="cuda").to(dtype)
    for inputs in ((x, xg), (xg, x)):
        grads = []
        for layer in (fused.pointwise_linear, lambda a, m: m(a)):
            with torch.autocast("cuda", dtype=dtype):
                ys = [layer(a, lin) for a in inputs]
            grads.append([torch.autograd.grad(y, (lin.weight, lin.bias), dy, allow_unused=True) for y in ys])
        for got, want in zip(*grads):
            for a, b in zip(got, want):
                assert a is not None
                _close(a, b, dtype, "autocast cache")


def test_pointwise_linear_with_parameters_updated_before_backward():
    """Images take no gradient, so backward needs no weights: an update between the passes (two losses,
    stepped one after the other) is allowed, as with nn.Linear."""
    torch.manual_seed(2)
    lin = torch.nn.Linear(3, 64).cuda()
    x, dy = torch.randn(2, 5, 7, 3, device="cuda"), torch.randn(2, 5, 7, 64, device="cuda")
    for context in (torch.autocast("cuda", enabled=False), torch.autocast("cuda", dtype=torch.bfloat16)):
        with context:
            y = fused.pointwise_linear(x, lin)
        assert type(y.grad_fn).__name__ == "_PointwiseLinearBackward"
        with torch.no_grad():
            lin.weight.mul_(0.5)
            lin.bias.add_(1.0)
        dw, db = torch.autograd.grad(y, (lin.weight, lin.bias), dy.to(y.dtype))
        _close(dw, dy.double().reshape(-1, 64).t() @ x.double().reshape(-1, 3), y.dtype, "dw")
        _close(db, dy.double().reshape(-1, 64).sum(0), y.dtype, "db")


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("use", ["forward_mode", "func_grad", "vmap", "trace", "compile", "subclass", "fx"])
def test_pointwise_linear_inside_transforms(use):
    """What nn.Linear takes part in and an autograd function with a native backward cannot: forward-mode
    derivatives, torch.func transforms, tracing (of the backward pass too), compilation and tensor subclasses."""
    from oriented1d_amd.convnext1d import PointwiseLinear

    torch.manual_seed(3)
    lin = PointwiseLinear(3, 64).cuda()
    plain = torch.nn.Linear(3, 64).cuda()
    plain.load_state_dict(lin.state_dict())
    x, t = torch.randn(2, 4, 5, 6, 3, device="cuda").unbind(0)

    def results(layer):
        if use == "forward_mode":
            import torch.autograd.forward_ad as fw
            with fw.dual_level():
                dual = fw.unpack_dual(layer(fw.make_dual(x, t)))
                return [dual.primal.detach(), dual.tangent.detach()]
        if use == "func_grad":
            p = {k: v.detach() for k, v in layer.named_parameters()}
            return list(torch.func.grad(lambda q: torch.func.functional_call(layer, q, x).square().sum())(p).values())
        if use == "vmap":
            return [torch.vmap(layer)(x).detach()]
        if use == "trace":
            traced = torch.jit.trace(layer, x)
            assert "PythonOp" not in str(traced.graph)
            return [traced(t).detach()]
        if use == "compile":
            return [torch.compile(layer, backend="eager", fullgraph=True)(x).detach()]
        if use == "fx":
            from torch.fx.experimental.proxy_tensor import make_fx
            dy = torch.randn(4, 5, 6, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(4))
            graph = make_fx(lambda a: torch.autograd.grad(layer(a), (layer.weight, layer.bias), dy))(x)
            return list(graph(t))
        y = layer(x.as_subclass(_Sub))
        assert type(y) is _Sub and type(y.grad_fn).__name__ != "_PointwiseLinearBackward"
        return [y.detach().as_subclass(torch.Tensor)]

    for a, b in zip(results(lin), results(plain)):
        _close(a, b, torch.float32, use)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape,N", [((1, 1, 1, 8), 8), ((1, 3, 5, 72), 96), ((2, 8, 8, 64), 64), ((1, 13, 5, 136), 328),
                                     ((2, 33, 32, 96), 384), ((3, 7, 7, 1536), 200), ((40, 20, 28, 96), 128),
                                     ((64, 14, 14, 200), 264), ((128, 7, 7, 384), 768)])
def test_linear_rows_and_planes(shape, N, dtype):
    """Both tile sizes of the product kernels, rows and columns that fill no tile, planes of 8 k, 4 k and odd pixels;
    the GELU against the exact one."""
    torch.manual_seed(N)
    B, H, W, K = shape
    x = torch.randn(*shape, device="cuda").to(dtype)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).to(dtype)
    b, s = torch.randn(N, device="cuda").to(dtype), torch.randn(N, device="cuda").to(dtype)
    res = torch.randn(B, N, H, W, device="cuda").to(dtype)
    host = fused._lib.host(0)
    y = F.linear(x.double(), w.double(), b.double())
    _close(host.linear_rows(x, w, b, True), F.gelu(y), dtype, "rows, gelu")
    _close(host.linear_rows(x, w, None, False), y - b.double(), dtype, "rows")
    _close(host.linear_planes(x, w, b, s, res), res.double() + (s.double() * y).permute(0, 3, 1, 2), dtype, "planes")
    _close(host.linear_planes(x, w, b, None, None), y.permute(0, 3, 1, 2), dtype, "planes alone")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape,N", [((1, 1, 1, 1032), 8), ((2, 1, 1, 64), 16), ((1, 7, 7, 3072), 768), ((1, 14, 14, 264), 384),
                                     ((1, 16, 16, 328), 512), ((1, 1, 257, 72), 512), ((2, 16, 16, 760), 512),
                                     ((1, 1, 513, 760), 512), ((8, 8, 8, 1024), 1024), ((2, 2, 127, 1016), 1024),
                                     ((1, 1, 513, 1024), 1024), ((98, 8, 4, 256), 24), ((5, 4, 5, 2056), 136),
                                     ((1, 1, 265, 1272), 1024), ((1, 1, 265, 1280), 1024)])
def test_product_kernels_of_few_tiles(shape, N, dtype):
    """Both sides of the lines between narrow, wide and 64 x 64 tiles (256 and 512 workgroups, rows of 1280), tails of the summed
    index, tiles that no XCD's share divides; rows, even and odd planes."""
    torch.manual_seed(N)
    B, H, W, K = shape
    x = torch.randn(*shape, device="cuda").to(dtype)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).to(dtype)
    b, s = torch.randn(N, device="cuda").to(dtype), torch.randn(N, device="cuda").to(dtype)
    res = torch.randn(B, N, H, W, device="cuda").to(dtype)
    host = fused._lib.host(0)
    y = F.linear(x.double(), w.double(), b.double())
    _close(host.linear_rows(x, w, b, True), F.gelu(y), dtype, "rows, gelu")
    _close(host.linear_planes(x, w, b, s, res), res.double() + (s.double() * y).permute(0, 3, 1, 2), dtype, "planes")


def test_product_kernels_keep_refusals():
    host = fused._lib.host(0)
    x = torch.zeros(1, 2, 2, 16, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(8, 16, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        host.linear_rows(x, w.half(), None, True)
    with pytest.raises(RuntimeError):
        host.linear_rows(x, w[:, :8], None, True)
    with pytest.raises(RuntimeError):
        host.linear_rows(x.float(), w.float(), None, True)
    with pytest.raises(RuntimeError):
        host.linear_planes(x, w, None, None, torch.zeros(1, 8, 2, 3, device="cuda", dtype=torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("C", [96, 128, 192, 384])
@pytest.mark.parametrize("N,H,W,scaled", [(1, 1, 1, True), (3, 13, 7, True), (2, 8, 24, False), (5, 14, 14, True), (9, 4, 32, True)])
def test_block_mlp(N, H, W, scaled, C, dtype):
    """Both layers in one kernel: rows that fill no workgroup, waves without pixels, planes of 8 k, 4 k and odd pixels (a wave's run
    then crosses images)."""
    torch.manual_seed(C + H)
    x = torch.randn(N, H, W, C, device="cuda").to(dtype)
    w1, b1 = (torch.randn(4 * C, C, device="cuda") * C ** -0.5).to(dtype), torch.randn(4 * C, device="cuda").to(dtype)
    w2, b2 = (torch.randn(C, 4 * C, device="cuda") * C ** -0.5).to(dtype), torch.randn(C, device="cuda").to(dtype)
    s = torch.randn(C, device="cuda").to(dtype) if scaled else None
    res = torch.randn(N, C, H, W, device="cuda").to(dtype)
    got = fused._lib.host(0).block_mlp(x, w1, b1, w2, b2, s, res)
    y = F.linear(F.gelu(F.linear(x.double(), w1.double(), b1.double())), w2.double(), b2.double())
    y = y if s is None else y * s.double()
    _close(got, res.double() + y.permute(0, 3, 1, 2), dtype, "block_mlp")
    with pytest.raises(RuntimeError):
        fused._lib.host(0).block_mlp(x, w1[:, :8], b1, w2, b2, s, res)
    with pytest.raises(RuntimeError):
        fused._lib.host(0).block_mlp(x, w1, b1, w2, b2, s, res.float())


def test_parameters_of_another_length_are_refused():
    """The kernels read as many values as x has channels: what is shorter, on the host or not fp32 is refused before a launch."""
    from oriented1d_amd import _lib
    from oriented1d_amd.convnext1d import ChannelsFirstLayerNorm
    host, dt = _lib.host(0), torch.bfloat16
    x, rows = torch.randn(2, 16, 4, 4, device="cuda").to(dt), torch.randn(5, 16, device="cuda").to(dt)
    good, stats = torch.ones(16, device="cuda"), torch.zeros(32, 2, device="cuda")
    nhwc, patches = x.permute(0, 2, 3, 1).contiguous(), torch.randn(2, 2, 2, 64, device="cuda").to(dt)
    for bad in (torch.ones(8, device="cuda"), torch.ones(16), torch.ones(16, device="cuda", dtype=dt),
                torch.ones(16, 2, device="cuda")[:, 0]):
        for call in (lambda: host.layernorm_nhwc(rows, bad, good, 1e-6, False),
                     lambda: host.layernorm_nhwc(rows, good, bad, 1e-6, True),
                     lambda: host.nchw_layernorm_nhwc(x, bad, good, 1e-6),
                     lambda: host.nhwc_scale_add_nchw(nhwc, bad, None),
                     lambda: host.ln_rows(rows, good, bad, 1e-6, 0, dt, True),
                     lambda: host.ln_rows_backward(rows, rows, stats, bad, good, 0, torch.float32),
                     lambda: host.ln_tile(x, bad, good, 1e-6, False, dt, True),
                     lambda: host.ln_tile_backward(nhwc, x, stats, bad, False, torch.float32),
                     lambda: host.ln_tile_backward(patches, x, stats, bad, True, torch.float32),
                     lambda: host.block_tail(nhwc, bad, x, dt, False),
                     lambda: host.block_tail_backward(x, nhwc, bad, dt, torch.float32)):
            with pytest.raises(RuntimeError, match="contiguous float32 values"):
                call()
    # a norm of half the channels in front of a downsampling layer: as F.layer_norm refuses it
    norm, conv = ChannelsFirstLayerNorm(8).cuda().to(dt), torch.nn.Conv2d(16, 24, 2, 2).cuda().to(dt)
    assert fused.downsample(x, norm, conv) is None
    with pytest.raises(RuntimeError):
        norm(x)
    with torch.no_grad():
        assert fused.downsample(x, norm, conv) is None
        with pytest.raises(RuntimeError):
            norm(x)


@pytest.mark.parametrize("which", ["first bias", "second bias", "layer scale", "stem bias"])
@pytest.mark.parametrize("rows", [4, 112])
def test_parameters_that_are_not_dense(which, rows):
    """Biases and layer scales that are views with a stride, in a block at inference (two kernels, one kernel) and in the stem's
    first layer in training: the values of dense ones."""
    from oriented1d_amd.convnext1d import Block
    torch.manual_seed(rows)
    dt = torch.bfloat16
    block = Block(96, (7,), False, layer_scale_init_value=1.0, arbitrary_size=True).cuda().to(dt).eval()
    stem = torch.nn.Linear(3, 64).cuda().to(dt)
    owner, name = {"first bias": (block.pwconv1, "bias"), "second bias": (block.pwconv2, "bias"),
                   "layer scale": (block, "gamma"), "stem bias": (stem, "bias")}[which]
    n = getattr(owner, name).numel()
    x = torch.randn(1, 96, rows, 112, device="cuda").to(dt)
    px = torch.randn(1, rows, 112, 3, device="cuda").to(dt)

    def outputs():
        with torch.no_grad():
            y = block(x)
        return y, fused.pointwise_linear(px, stem).detach()
    wide = torch.randn(n, 3, device="cuda").to(dt)
    setattr(owner, name, torch.nn.Parameter(wide[:, 1]))
    assert not getattr(owner, name).is_contiguous()
    got = outputs()
    setattr(owner, name, torch.nn.Parameter(wide[:, 1].contiguous()))
    for a, b in zip(got, outputs()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_gelu_of_a_product_far_out(dtype):
    """Beyond the range of its polynomial: u or 0 as far as the type reaches, and what u * (1 + erf) gives for infinities and NaN."""
    from oriented1d_amd import _lib
    far = [8.5, 20.0, 300.0, torch.finfo(dtype).max]
    u = torch.tensor(far + [-v for v in far[1:]] + [float("inf"), -float("inf"), float("nan"), 0.0, -0.0], device="cuda").to(dtype)
    x, w = torch.zeros(u.numel(), 8, device="cuda", dtype=dtype), torch.zeros(8, 8, device="cuda", dtype=dtype)
    x[:, 0], w[:, 0] = u, 1.0
    ref = (0.5 * u.double() * (1 + torch.special.erf(u.double() * 0.5 ** 0.5))).to(dtype)
    got = _lib.host(0).linear_rows(x, w, None, True)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)[:, None].expand(-1, 8))
    assert torch.equal(got.nan_to_num(1.5), ref.nan_to_num(1.5)[:, None].expand(-1, 8))


@pytest.mark.parametrize("dtype,unit", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)], ids=["bf16", "f16"])
def test_gelu_of_the_negative_tail(dtype, unit):
    """GELU value by value, as far as results are normal numbers.  Behind LayerNorm: the rounding of the result (``unit`` of it)
    and 2 % for what GELU takes, whose fp32 rounding the tail magnifies (relative slope about u^2 <= 16).  In a product
    kernel no more than separate layers, whose u is rounded first: units of the result, and u^2 of them."""
    from oriented1d_amd import _lib
    torch.manual_seed(0)
    x = torch.randn(20000, 64, device="cuda").to(dtype)
    w, b = torch.full((64,), 2.0, device="cuda"), torch.full((64,), -1.0, device="cuda")
    host = _lib.host(0)
    u1 = (-4 + 8 * torch.rand(4096, 8, device="cuda")).to(dtype)  # a product of one term: u is what the kernel holds
    for u, y, bound in (
            (F.layer_norm(x.double(), (64,), w.double(), b.double(), 1e-6), host.ln_rows(x, w, b, 1e-6, 1, dtype, False)[0],
             lambda u: 1.02 * unit),
            (u1.double(), host.linear_rows(u1, torch.eye(8, device="cuda").to(dtype), None, True),
             lambda u: (1 + u * u) * unit)):
        ref = u * torch.special.erfc(-u * 0.5 ** 0.5) / 2
        # (normal results; around zero the sum of LayerNorm's scale and shift cancels)
        some = (u.abs() >= 0.25) & (u.abs() <= 4) & (ref.abs() >= 2.0 ** -14)
        assert (u[some] < -3).sum() > 100
        assert (((y.double() - ref).abs() / ref.abs()) <= bound(u))[some].all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("C,images,H,W,want", [
    (96, 1, 128, 96, "one"), (96, 1, 128, 95, "two"), (128, 5, 29, 113, "one"), (128, 1, 128, 128, "two"),
    (192, 7, 64, 64, "one"), (192, 1, 169, 169, "two"), (384, 6, 11, 331, "one"), (384, 5, 17, 257, "two"),
    (384, 1, 256, 128, "one"), (384, 1, 331, 99, "two"), (384, 10, 17, 257, "two"), (384, 23, 38, 50, "one"),
    (512, 2, 32, 32, "two"), (512, 1, 32, 64, "two"), (520, 1, 32, 64, "two"), (520, 1, 32, 65, "rows"), (64, 1, 9, 7, "two")])
@pytest.mark.parametrize("scaled", [True, False])
def test_block_dispatch_at_inference(C, images, H, W, want, scaled, dtype, monkeypatch):
    """A block at inference on both sides of each line between its routes (one kernel for both layers, two product kernels,
    the first one and the library's product), against the composition in fp64 behind the block's own convolution; the entry points
    that were called are those that the rule names."""
    from oriented1d_amd import _lib
    from oriented1d_amd.convnext1d import Block
    if dtype == torch.float16 and not scaled:
        pytest.skip("one type without a layer scale")
    torch.manual_seed(C + W)
    block = Block(C, (7,), False, layer_scale_init_value=1.0 if scaled else 0.0, arbitrary_size=True).cuda().to(dtype).eval()
    with torch.no_grad():
        for p in block.parameters():
            if p.dim() == 1:
                p.add_((torch.randn_like(p) * 0.3))
        block.dwconv.theta.zero_()
    x = torch.randn(images, C, H, W, device="cuda").to(dtype)
    called, real = [], _lib.host(0)

    class Host:
        def __getattr__(self, name):
            called.append(name)
            return getattr(real, name)
    monkeypatch.setattr(_lib, "host", lambda device: Host())
    with torch.no_grad():
        got = block(x)
    monkeypatch.undo()
    assert (block.gamma is not None) == scaled
    assert [n for n in called if n in ("block_mlp", "linear_rows", "linear_planes", "nhwc_scale_add_nchw")] == {
        "one": ["block_mlp"], "two": ["linear_rows", "linear_planes"], "rows": ["linear_rows", "nhwc_scale_add_nchw"]}[want]
    with torch.no_grad():
        y = block.dwconv(x).permute(0, 2, 3, 1)
        d = [t if t is None else t.double() for t in (block.norm.weight, block.norm.bias, block.pwconv1.weight, block.pwconv1.bias,
                                                      block.pwconv2.weight, block.pwconv2.bias, block.gamma)]
        for n in range(images):  # (an image at a time: the hidden tensor in fp64)
            h = F.gelu(F.linear(F.layer_norm(y[n].double(), (C,), d[0], d[1], 1e-6), d[2], d[3]))
            h = F.linear(h, d[4], d[5])
            ref = x[n].double() + (h if d[6] is None else d[6] * h).permute(2, 0, 1)
            _close(got[n], ref, dtype, "block")


@pytest.mark.parametrize("C,plus_plus,hw,N,dtype,gamma,wrapped", [
    (96, False, 9, 3, torch.bfloat16, 0.1, False), (96, True, 12, 2, torch.float16, 0.1, True),
    (384, False, 14, 128, torch.bfloat16, 0.0, False),  # (both layers as one kernel, no layer scale)
    (768, True, 7, 50, torch.bfloat16, 0.1, False)])    # (second layer by the library)
def test_inference_block_checked_once(C, plus_plus, hw, N, dtype, gamma, wrapped, monkeypatch):
    """A block at inference whose layers are checked once gives the bits of its layers one by one, and leaves blocks with hooks,
    in autocast or of another type to them."""
    from oriented1d_amd import fused
    from oriented1d_amd.convnext1d import Block
    torch.manual_seed(C + hw)
    block = Block(C, (15, 31) if plus_plus else (31,), plus_plus, layer_scale_init_value=gamma, arbitrary_size=True,
                  wrapped=wrapped).cuda().to(dtype).eval()
    x = torch.randn(N, C, hw, hw, device="cuda").to(dtype)
    taken = []
    whole = fused.infer_block
    monkeypatch.setattr(fused, "infer_block", lambda *a: taken.append(whole(*a)) or taken[-1])
    with torch.no_grad():
        got = block(x.transpose(2, 3).contiguous().transpose(2, 3))  # (not dense)
        assert taken[-1] is not None
        monkeypatch.setattr(fused, "infer_block", lambda *a: None)
        assert torch.equal(got, block(x))
        monkeypatch.setattr(fused, "infer_block", lambda *a: taken.append(whole(*a)) or taken[-1])
        seen = []
        handle = block.pwconv2.register_forward_hook(lambda *_: seen.append(1))
        block(x)
        handle.remove()
        assert taken[-1] is None and seen
        with torch.autocast("cuda", dtype=dtype):
            block(x)
        assert taken[-1] is None
        block.float()(x.float())
        assert taken[-1] is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("N,H,W,C,bias", [(1, 1, 1, 96, True), (3, 33, 31, 96, True), (2, 6, 10, 128, False), (5, 8, 12, 128, True),
                                          (70, 56, 56, 96, True)])  # (pixels by eight, four and one; waves that take several tiles)
def test_stem_tail_as_one_kernel(N, H, W, C, bias, dtype):
    """LayerNorm + GELU + pointwise layer + LayerNorm as planes against the same layers in fp64, the value between them rounded as a
    layer's output; tolerance: twice the type's rounding in the norm, its largest step relative to the largest value."""
    import torch.nn.functional as F
    from oriented1d_amd import fused
    torch.manual_seed(H * W)
    before, norm, linear = torch.nn.LayerNorm(64, eps=1e-6), torch.nn.LayerNorm(C, eps=1e-6), fused.Linear(64, C, bias=bias)
    with torch.no_grad():
        for m in (before, norm):
            m.weight.add_(torch.randn(m.weight.shape) * 0.3), m.bias.add_(torch.randn(m.bias.shape) * 0.3)
        before, norm, linear = (m.cuda().to(dtype) for m in (before, norm, linear))
        x = (torch.randn(N, H, W, 64, device="cuda") * 3 + 1).to(dtype)
        got = fused.norm_planes(x, before, linear, norm)
        z = F.gelu(F.layer_norm(x.double(), (64,), before.weight.double(), before.bias.double(), 1e-6)).to(dtype).double()
        y = F.linear(z, linear.weight.double(), None if not bias else linear.bias.double())
        ref = F.layer_norm(y, (C,), norm.weight.double(), norm.bias.double(), 1e-6).permute(0, 3, 1, 2)
        assert got.shape == ref.shape and got.is_contiguous() and got.dtype == dtype
        ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        assert (got.double() - ref).norm() <= ulp * ref.norm() and (got.double() - ref).abs().max() <= 2 * ulp * ref.abs().max()
        handle = linear.register_forward_hook(lambda *_: None)
        assert fused.norm_planes(x, before, linear, norm) is None
        handle.remove()
        assert fused.norm_planes(x.float(), before.float(), linear.float(), norm.float()) is None
    assert fused.norm_planes(x, before.to(dtype), linear.to(dtype), norm.to(dtype)) is None  # (gradients are on)


@pytest.mark.parametrize("plus_plus,wrapped", [(False, True), (False, False), (True, True)])
def test_inference_block_leaves_what_watches_it_to_its_layers(plus_plus, wrapped, monkeypatch):
    """Hooks on any layer, the operator or its wrapper, dispatch modes, dual tensors, subclasses and recorded gradients see the
    layers one by one, with the same values but for roundings between them."""
    import torch.autograd.forward_ad as fwd
    import torch.nn.modules.module as modules
    from torch.utils._python_dispatch import TorchDispatchMode
    from oriented1d_amd.convnext1d import Block
    torch.manual_seed(5)
    block = Block(64, (15, 31) if plus_plus else (31,), plus_plus, layer_scale_init_value=0.1, arbitrary_size=True,
                  wrapped=wrapped).cuda().bfloat16().eval()
    x, taken, whole = torch.randn(2, 64, 9, 11, device="cuda").bfloat16(), [], fused.infer_block
    monkeypatch.setattr(fused, "infer_block", lambda *a: taken.append(whole(*a)) or taken[-1])

    def refused(run):
        del taken[:]
        y = run()
        assert taken and all(t is None for t in taken)
        return y

    class Watch(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Watch.ops += 1
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    with torch.no_grad():
        ref = block(x)
        assert taken[-1] is not None
        for name, layer in block.named_modules():
            if type(layer).__name__ in ("Linear", "ConvWrapper", "DepthwiseOrientedConv1d"):
                seen = []
                for register in (layer.register_forward_hook, layer.register_forward_pre_hook):
                    handle = register(lambda *_: seen.append(1))
                    _close(refused(lambda: block(x)), ref, x.dtype, name)
                    assert seen, name
                    handle.remove()
        handle = modules.register_module_forward_hook(lambda *_: None)
        _close(refused(lambda: block(x)), ref, x.dtype, "global hook")
        handle.remove()
        with Watch():
            _close(refused(lambda: block(x)), ref, x.dtype, "dispatch mode")
        assert Watch.ops > 0
        with fwd.dual_level(), pytest.raises(NotImplementedError, match="jvp"):  # (no layer drops a tangent silently)
            block(fwd.make_dual(x, torch.ones_like(x)))
        _close(refused(lambda: block(x.as_subclass(Sub))).as_subclass(torch.Tensor), ref, x.dtype, "subclass")
        assert torch.equal(block(x), ref) and taken[-1] is not None
    assert refused(lambda: block(x.clone().requires_grad_())).requires_grad


@pytest.mark.parametrize("plus_plus,which", [(False, "dwconv"), (True, "dwconv1"), (True, "dwconv2")])
@pytest.mark.parametrize("arbitrary_size", [True, False])
def test_inference_block_with_functions_of_the_caller(plus_plus, which, arbitrary_size, monkeypatch):
    """A block whose operator holds five functions that are no ``KernelTuple`` runs layer by layer, through them."""
    from oriented1d_amd.convnext1d import Block
    torch.manual_seed(3)
    block = Block(64, (15, 31) if plus_plus else (31,), plus_plus, layer_scale_init_value=0.1,
                  arbitrary_size=arbitrary_size).cuda().bfloat16().eval()
    conv, name, calls = getattr(block, which), "module_fp32_large" if arbitrary_size else "module_fp32", []
    own = tuple(getattr(conv, name))
    setattr(conv, name, (lambda *a: calls.append(1) or own[0](*a),) + own[1:])
    taken, whole = [], fused.infer_block
    monkeypatch.setattr(fused, "infer_block", lambda *a: taken.append(whole(*a)) or taken[-1])
    x = torch.randn(2, 64, 9, 11, device="cuda").bfloat16()
    with torch.no_grad():
        got = block(x)
        assert taken == [None] and calls == [1]
        monkeypatch.setattr(fused, "infer_block", lambda *a: None)
        assert torch.equal(got, block(x))
