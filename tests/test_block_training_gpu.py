"""The training passes of the block and the stem (LayerNorm in both layouts, GELU, layer scale + residual, the
pointwise layers' parameter gradients) against the same compositions in fp64 PyTorch.

Tolerances: tensors and sums of fp32 are good to 1e-5 as the operator's; what is rounded to a 16-bit type on the way out
carries that type's rounding, 2^-9 (bf16) or 2^-12 (fp16) of the value at most, and 1e-2 is the operator's own bound for them.
Parameter gradients are fp32 sums of exact products of the inputs: 1e-5 whatever the inputs' type, except where
they are asked for in 16 bits."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from parity_util import TOL, rel_err

from oriented1d_amd import fused

pytestmark = pytest.mark.gpu
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
TYPES = [(F32, F32), (F32, BF16), (F32, F16), (BF16, BF16), (BF16, F32), (F16, F16), (F16, F32)]


def close(got, ref, tol, what):
    e = rel_err(got.detach().float().cpu().numpy(), ref.detach().double().cpu().numpy())
    assert max(e) <= tol, (what, e)


def run_norm(x, w, b, dout, native, reference, tol_out, tol_dx):
    leaves = [t.detach().clone().requires_grad_(True) for t in (x, w, b)]
    out = native(*leaves)
    got = torch.autograd.grad(out, leaves, dout)
    ref_leaves = [t.detach().double().requires_grad_(True) for t in (x, w, b)]
    ref = reference(*ref_leaves)
    want = torch.autograd.grad(ref, ref_leaves, dout.double())
    close(out, ref, tol_out, "out")
    close(got[0], want[0], tol_dx, "dx")
    close(got[1], want[1], 1e-5, "dw")
    close(got[2], want[2], 1e-5, "db")


@pytest.mark.parametrize("types", TYPES, ids=str)
@pytest.mark.parametrize("N,C,H,W", [(2, 96, 9, 8), (1, 8, 1, 1), (3, 64, 5, 13), (2, 72, 16, 16), (1, 128, 33, 2),
                                     (2, 256, 7, 7), (2, 520, 3, 4), (1, 1024, 7, 7), (40, 96, 56, 56),
                                     (33, 64, 1, 3), (7, 264, 3, 5), (9, 512, 2, 2), (260, 128, 7, 12)])
def test_tile_norm(N, C, H, W, types):
    if N == 40 and types != (F32, BF16):
        pytest.skip("one type at the size where workgroups take several tiles")
    tin, tout = types
    torch.manual_seed(C + H)
    x = (torch.randn(N, C, H, W, device="cuda") * 2 + 0.5).to(tin)
    w, b = torch.randn(C, device="cuda") * 0.5 + 1, torch.randn(C, device="cuda") * 0.1
    dout = torch.randn(N, H, W, C, device="cuda").to(tout)
    run_norm(x, w, b, dout, lambda x, w, b: fused._TileNorm.apply(x, w, b, 1e-6, tout),
             lambda x, w, b: F.layer_norm(x.permute(0, 2, 3, 1), (C,), w, b, 1e-6), TOL[tout], TOL[tin])


@pytest.mark.parametrize("types", TYPES, ids=str)
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("shape", [(2, 11, 5, 64), (1, 8), (37, 72), (9, 9, 128), (130, 256), (33, 520), (5, 1024),
                                   (9000, 64)])
def test_row_norm(shape, gelu, types):
    tin, tout = types
    C = shape[-1]
    torch.manual_seed(C)
    x = (torch.randn(*shape, device="cuda") * 2 - 0.25).to(tin)
    w, b = torch.randn(C, device="cuda") * 0.5 + 1, torch.randn(C, device="cuda") * 0.1
    dout = torch.randn(*shape, device="cuda").to(tout)

    def reference(x, w, b):
        y = F.layer_norm(x, (C,), w, b, 1e-6)
        return F.gelu(y) if gelu else y
    run_norm(x, w, b, dout, lambda x, w, b: fused._RowNorm.apply(x, w, b, 1e-6, int(gelu), tout), reference,
             TOL[tout], TOL[tin])


@pytest.mark.parametrize("ty,tr", [(F32, F32), (BF16, F32), (F16, F32), (BF16, BF16), (F16, F16)], ids=str)
@pytest.mark.parametrize("N,C,H,W", [(2, 96, 9, 8), (1, 8, 1, 1), (3, 64, 5, 13), (2, 136, 16, 16), (2, 768, 7, 7),
                                     (70, 64, 56, 56)])
def test_block_tail(N, C, H, W, ty, tr):
    torch.manual_seed(C + W)
    y = torch.randn(N, H, W, C, device="cuda").to(ty).requires_grad_(True)
    g = (torch.randn(C, device="cuda") * 0.5).requires_grad_(True)
    x = torch.randn(N, C, H, W, device="cuda").to(tr).requires_grad_(True)
    dout = torch.randn(N, C, H, W, device="cuda").to(tr)
    out = fused._BlockTail.apply(y, g, x, tr, False)
    got = torch.autograd.grad(out, (y, g, x), dout)
    leaves = [t.detach().double().requires_grad_(True) for t in (y, g, x)]
    ref = leaves[2] + (leaves[1] * leaves[0]).permute(0, 3, 1, 2)
    want = torch.autograd.grad(ref, leaves, dout.double())
    close(out, ref, TOL[tr], "out")
    close(got[0], want[0], TOL[ty], "dy")
    close(got[1], want[1], 1e-5, "dgamma")
    assert torch.equal(got[2], dout)


def test_block_tail_of_a_16_bit_stream_and_planes_alone():
    torch.manual_seed(5)
    y = torch.randn(2, 5, 9, 72, device="cuda").to(BF16).requires_grad_(True)
    g = torch.randn(72, device="cuda", requires_grad=True)
    x = torch.randn(2, 72, 5, 9, device="cuda").to(BF16).requires_grad_(True)
    out = fused.block_tail(y, g, x)  # (16-bit stream, fp32 layer scale: the sum is fp32)
    assert out.dtype == F32 and (x + (g * y).permute(0, 3, 1, 2)).dtype == F32
    dout = torch.randn_like(out)
    got = torch.autograd.grad(out, (y, g, x), dout)
    leaves = [t.detach().double().requires_grad_(True) for t in (y, g, x)]
    ref = leaves[2] + (leaves[1] * leaves[0]).permute(0, 3, 1, 2)
    want = torch.autograd.grad(ref, leaves, dout.double())
    close(out, ref, 1e-5, "out")
    for a, b, tol in zip(got, want, (TOL[BF16], 1e-5, TOL[BF16])):
        close(a, b, tol, "gradient")
    z = fused.planes(y)
    assert type(z.grad_fn).__name__ == "_BlockTailBackward" and torch.equal(z, y.permute(0, 3, 1, 2))
    d = torch.randn_like(z)
    assert torch.equal(torch.autograd.grad(z, y, d)[0], d.permute(0, 2, 3, 1))


@pytest.mark.parametrize("types", [(F32, F32), (F32, BF16), (BF16, BF16), (F16, F16)], ids=str)
@pytest.mark.parametrize("N,C,H,W", [(1, 8, 2, 2), (2, 96, 8, 12), (3, 64, 5, 13), (2, 72, 17, 6), (1, 256, 33, 64),
                                     (2, 520, 6, 4), (1, 1024, 3, 9), (30, 96, 56, 56)])
def test_patch_norm(N, C, H, W, types):
    tin, tout = types
    torch.manual_seed(C + H)
    x = (torch.randn(N, C, H, W, device="cuda") * 2 + 0.5).to(tin)
    w, b = torch.randn(C, device="cuda") * 0.5 + 1, torch.randn(C, device="cuda") * 0.1
    dout = torch.randn(N, H // 2, W // 2, 4 * C, device="cuda").to(tout)
    run_norm(x, w, b, dout, lambda x, w, b: fused._TileNorm.apply(x, w, b, 1e-6, tout, True),
             lambda x, w, b: fused._patches(F.layer_norm(x.permute(0, 2, 3, 1), (C,), w, b, 1e-6)), TOL[tout], TOL[tin])


@pytest.mark.parametrize("mode", ["autocast", "bf16", "infer"])
@pytest.mark.parametrize("N,C,D,H,W", [(2, 64, 128, 12, 12), (1, 96, 192, 7, 9), (3, 32, 40, 14, 6), (1, 768, 1024, 4, 4)])
def test_downsample_against_the_convolution(N, C, D, H, W, mode):
    from oriented1d_amd.convnext1d import ChannelsFirstLayerNorm
    torch.manual_seed(C)
    norm, conv = ChannelsFirstLayerNorm(C).cuda(), nn.Conv2d(C, D, 2, 2).cuda()
    with torch.no_grad():
        norm.weight.add_(torch.randn_like(norm.weight) * 0.3)
        norm.bias.add_(torch.randn_like(norm.bias) * 0.3)
    x = torch.randn(N, C, H, W, device="cuda")
    if mode != "autocast":
        norm, conv, x = norm.to(BF16), conv.to(BF16), x.to(BF16)
    params = [norm.weight, norm.bias, conv.weight, conv.bias]
    ref_leaves = [t.detach().double().requires_grad_(True) for t in [x] + params]
    rx, rw, rb, rc, rd = ref_leaves
    ref = F.conv2d(F.layer_norm(rx.permute(0, 2, 3, 1), (C,), rw, rb, 1e-6).permute(0, 3, 1, 2), rc, rd, stride=2)
    if mode == "infer":
        with torch.no_grad():
            y = fused.downsample(x, norm, conv)
        close(y, ref, TOL[BF16], "y")
        return
    x.requires_grad_(True)
    with torch.autocast("cuda", dtype=BF16, enabled=mode == "autocast"):
        y = fused.downsample(x, norm, conv)
    assert y.dtype == BF16 and y.is_contiguous()
    dy = torch.randn_like(y)
    got = torch.autograd.grad(y, [x] + params, dy)
    want = torch.autograd.grad(ref, ref_leaves, dy.double())
    close(y, ref, TOL[BF16], "y")
    # (through a 16-bit product of K = 4 C terms and its 16-bit gradient)
    for a, b in zip(got, want):
        assert a.shape == b.shape
        close(a, b, 2 * TOL[BF16], "gradient")


@pytest.mark.parametrize("dtype", [BF16, F16], ids=str)
@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (63, 96, 384), (64, 128, 128), (65, 136, 120), (4096, 64, 72), (777, 768, 192),
                                   (20000, 96, 136), (300, 1024, 264)])
def test_linear_gradients(M, K, N, dtype):
    torch.manual_seed(M + K)
    m = fused.Linear(K, N).cuda()
    x = torch.randn(M, K, device="cuda", requires_grad=True)
    dy = torch.randn(M, N, device="cuda").to(dtype)
    with torch.autocast("cuda", dtype=dtype):
        y = m(x)
    assert type(y.grad_fn).__name__ == "_LinearBackward" and y.dtype == dtype
    dx, dw, db = torch.autograd.grad(y, (x, m.weight, m.bias), dy)
    xq, wq = x.detach().to(dtype).double(), m.weight.detach().to(dtype).double()
    close(dx, dy.double() @ wq, TOL[dtype], "dx")
    assert dw.dtype == F32 and db.dtype == F32
    close(dw, dy.double().t() @ xq, 1e-5, "dw")
    close(db, dy.double().sum(0), 1e-5, "db")


# stages of 32 rows, four in flight: rows around a stage, a step of 64 and the four; outputs around a tile of 128; few tiles, whose
# sums are kept in halves where there are fewer splits; as many tiles as CUs, which write the gradients themselves in either type
# as long as the rows are few (54 or 128 steps)
@pytest.mark.parametrize("grad", [F32, BF16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (31, 128, 128), (33, 136, 120), (65, 256, 264), (127, 8, 1024), (129, 64, 72),
                                   (1023, 128, 256), (1025, 120, 128), (4161, 256, 136), (20011, 128, 96), (97, 1920, 1920),
                                   (1300, 1800, 2056), (3456, 1792, 2048), (3457, 1792, 2048), (8192, 3584, 1024),
                                   (8193, 3584, 1024), (16640, 512, 128)])
def test_linear_wgrad_stages_and_splits(M, N, K, grad):
    from oriented1d_amd import _lib
    torch.manual_seed(M + N)
    x, dy = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    for bias in (True, False):
        dw, db = _lib.host(0).linear_wgrad(dy, x, bias, grad)
        tol = 1e-5 if grad == F32 else 2.0 ** -8
        close(dw, dy.double().t() @ x.double(), tol, "dw")
        assert (db is None) == (not bias)
        if bias:
            close(db, dy.double().sum(0), tol, "db")


@pytest.mark.parametrize("rows", [449, 512, 576, 640, 700, 832, 960])
def test_linear_wgrad_of_many_tiles_sums_in_chains_as_short_as_two_splits(rows):
    """256 tiles (one workgroup per tile, whose sums are kept in halves) against 192 of the same columns (two splits of the
    rows): the same error against 64 bits, within what a chain longer by 64 of 320 to 448 rows gives (sqrt(1.04)) and 2 %."""
    from oriented1d_amd import _lib
    torch.manual_seed(rows)
    x, dy = torch.randn(rows, 1024, device="cuda").bfloat16(), torch.randn(rows, 4096, device="cuda").bfloat16()
    ref = dy.double().t() @ x[:, :768].double()
    err = [((dw[:, :768].double() - ref).norm() / ref.norm()).item()
           for dw in (_lib.host(0).linear_wgrad(dy, v, False, F32)[0] for v in (x, x[:, :768].contiguous()))]
    assert 0 < err[0] <= 1.04 * err[1] and err[1] < 2e-7, err


def test_linear_covers_batches_views_and_second_order():
    torch.manual_seed(0)
    m = fused.Linear(64, 128).cuda().bfloat16()
    x = torch.randn(2, 3, 5, 64, device="cuda").to(BF16)
    buf = torch.randn(2 * 3 * 5 * 128 + 1, device="cuda").to(BF16)
    dy = buf[1:].view(2, 3, 5, 128)  # a gradient that is a misaligned piece of another buffer
    y = m(x)
    dw, db = torch.autograd.grad(y, (m.weight, m.bias), dy)
    assert dw.dtype == BF16
    close(dw, dy.double().reshape(-1, 128).t() @ x.double().reshape(-1, 64), TOL[BF16], "dw")
    close(db, dy.double().sum((0, 1, 2)), TOL[BF16], "db")
    m = fused.Linear(64, 64).cuda()
    x = torch.randn(7, 64, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=BF16):
        y = m(x)
    gx, gw = torch.autograd.grad(y.float().square().sum(), (x, m.weight), create_graph=True)
    hx, hw = torch.autograd.grad(gx.square().sum() + gw.square().sum(), (x, m.weight))
    p = nn.Linear(64, 64).cuda()
    p.load_state_dict(m.state_dict())
    z = p(x)
    px, pw = torch.autograd.grad(z.square().sum(), (x, p.weight), create_graph=True)
    rx, rw = torch.autograd.grad(px.square().sum() + pw.square().sum(), (x, p.weight))
    close(hx, rx, 3e-2, "second order x")  # (a chain of four bf16 products)
    close(hw, rw, 3e-2, "second order w")


def test_16_bit_passes_round_where_separate_passes_do():
    """Without autocast every pass of the composition returns a 16-bit tensor: the fused passes round at the same places, so
    that they differ from it only where a sum's last bit decides a rounding."""
    torch.manual_seed(8)
    norm = nn.LayerNorm(64, eps=1e-6).cuda().to(BF16)
    with torch.no_grad():
        norm.weight.add_(torch.randn_like(norm.weight) * 0.3)
    x = torch.randn(4, 20, 20, 64, device="cuda").to(BF16).requires_grad_(True)
    gamma = torch.randn(64, device="cuda").to(BF16)
    planes = torch.randn(4, 64, 20, 20, device="cuda").to(BF16)
    for native, composed in ((lambda: fused.row_norm(x, norm, gelu=True), lambda: F.gelu(norm(x))),
                             (lambda: fused.block_tail(x, gamma, planes),
                              lambda: planes + (gamma * x).permute(0, 3, 1, 2).contiguous())):
        y, z = native(), composed()
        d = torch.randn_like(y)
        for a, b in zip((y, *torch.autograd.grad(y, x, d)), (z, *torch.autograd.grad(z, x, d))):
            assert (a != b).float().mean() < 5e-3


@pytest.mark.parametrize("which", ["tile", "rows", "tail"])
def test_second_order_of_the_passes(which):
    torch.manual_seed(1)
    a = torch.randn(2, 16, 3, 5, device="cuda", dtype=F32, requires_grad=True)
    w = torch.randn(16, device="cuda", requires_grad=True)
    b = torch.randn(16, device="cuda", requires_grad=True)
    nhwc = a.permute(0, 2, 3, 1).contiguous()
    native, reference = {
        "tile": (lambda: fused._TileNorm.apply(a, w, b, 1e-6, F32),
                 lambda: F.layer_norm(a.permute(0, 2, 3, 1), (16,), w, b, 1e-6)),
        "rows": (lambda: fused._RowNorm.apply(nhwc, w, b, 1e-6, 1, F32),
                 lambda: F.gelu(F.layer_norm(nhwc, (16,), w, b, 1e-6))),
        "tail": (lambda: fused._BlockTail.apply(nhwc, w, a, F32, False),
                 lambda: a + (w * nhwc).permute(0, 3, 1, 2))}[which]
    res = []
    for f in (native, reference):
        y = f()
        g = torch.autograd.grad((y ** 3).sum(), (a, w), create_graph=True)
        res.append(torch.autograd.grad(sum((t * t).sum() for t in g), (a, w)))
    for got, ref in zip(*res):
        close(got, ref.double(), 1e-4, which)  # (fp32 on both sides)


@pytest.mark.parametrize("which", ["tile", "patch", "rows", "tail", "planes"])
def test_recorded_backward_of_inputs_that_are_not_dense(which):
    """Gradients and gradients of gradients of views in another order, through the functions that the modules call, against the
    composition (fp32 on both sides, the patches' layer in bf16)."""
    from oriented1d_amd.convnext1d import ChannelsFirstLayerNorm
    torch.manual_seed(2)
    a = torch.randn(2, 6, 4, 16, device="cuda", requires_grad=True)
    w = torch.randn(16, device="cuda", requires_grad=True)
    norm = (nn.LayerNorm(16, eps=1e-6) if which == "rows" else ChannelsFirstLayerNorm(16)).cuda()
    conv = nn.Conv2d(16, 24, 2, 2).cuda()
    planes = a.permute(0, 3, 1, 2)                  # [N,C,H,W], channels last in memory
    rows = a.permute(0, 2, 1, 3)                    # [N,W,H,C]
    assert not planes.is_contiguous() and not rows.is_contiguous()

    def normed(x):
        return F.layer_norm(x, (16,), norm.weight, norm.bias, 1e-6)

    def native():
        if which == "tile":
            return norm(planes)
        if which == "patch":
            with torch.autocast("cuda", dtype=BF16):
                return fused.downsample(planes, norm, conv).float()
        if which == "rows":
            return fused.row_norm(rows, norm, gelu=True)
        return fused.block_tail(rows, w, planes.transpose(2, 3)) if which == "tail" else fused.planes(rows)

    def reference():
        if which == "tile":
            return normed(planes.permute(0, 2, 3, 1)).permute(0, 3, 1, 2)
        if which == "patch":
            return conv(normed(planes.permute(0, 2, 3, 1)).permute(0, 3, 1, 2))
        if which == "rows":
            return F.gelu(normed(rows))
        return planes.transpose(2, 3) + (w * rows).permute(0, 3, 1, 2) if which == "tail" else rows.permute(0, 3, 1, 2)

    params = {"tail": [w], "planes": []}.get(which, [norm.weight, norm.bias])
    res = []
    for f in (native, reference):
        y = f()
        assert y.grad_fn is not None
        first = torch.autograd.grad((y ** 3).sum(), [a] + params, create_graph=True)
        res.append(list(first) + list(torch.autograd.grad(sum((t * t).sum() for t in first), [a] + params)))
    # (fp32 sums in another order; a chain of four 16-bit products behind the patches)
    for got, ref in zip(*res):
        close(got, ref.double(), 5e-2 if which == "patch" else 1e-4, which)


def test_recorded_backward_takes_the_weights_of_the_forward_pass():
    """Parameters that autocast converts may be updated between the passes, as with PyTorch's own layers: their 16-bit copies of the
    forward pass are what every backward pass differentiates."""
    from oriented1d_amd.convnext1d import ChannelsFirstLayerNorm
    torch.manual_seed(6)
    lin, norm, conv = fused.Linear(16, 8).cuda(), ChannelsFirstLayerNorm(16).cuda(), nn.Conv2d(16, 8, 2, 2).cuda()
    for layer, weight, shape in ((lin, lin.weight, (4, 16)), (lambda x: fused.downsample(x, norm, conv), conv.weight, (1, 16, 4, 4))):
        x = torch.randn(*shape, device="cuda", requires_grad=True)

        def run(recorded, factor):
            with torch.autocast("cuda", dtype=BF16):
                y = layer(x)
            with torch.no_grad():
                weight.mul_(factor)
            g, = torch.autograd.grad(y.float().square().sum(), x, create_graph=recorded)
            h = torch.autograd.grad(g.square().sum(), (x, weight)) if recorded else ()
            with torch.no_grad():
                weight.mul_(1.0 / factor)
            return [g, *h]
        (plain,), kept, doubled = run(False, 2.0), run(True, 1.0), run(True, 2.0)
        close(kept[0], plain.double(), 2 * TOL[BF16], "dx")  # (products in 16 bits on both sides)
        for got, ref in zip(doubled, kept):
            assert torch.equal(got, ref)


def test_hooks_and_replaced_forwards_keep_the_module_path():
    from oriented1d_amd.convnext1d import Block
    torch.manual_seed(0)
    blk = Block(32, (31,), False, layer_scale_init_value=0.5).cuda()
    x = torch.randn(2, 32, 12, 12, device="cuda")
    plain = blk(x)
    assert type(plain.grad_fn).__name__ == "_BlockTailBackward"
    seen = []
    handle = blk.norm.register_forward_hook(lambda m, i, o: seen.append(tuple(i[0].shape)))
    hooked = blk(x)
    handle.remove()
    assert seen == [(2, 12, 12, 32)]
    close(hooked, plain.double(), 1e-5, "hooked")
    blk.norm.forward = lambda t: torch.zeros_like(t)
    zeroed = blk(x)
    del blk.norm.forward
    assert not torch.allclose(zeroed, plain)


@pytest.mark.parametrize("mode", ["autocast", "f32"])
@pytest.mark.parametrize("variant", ["1d", "1dpp"])
@pytest.mark.parametrize("hooks", ["checkpoint", "cpu"])
def test_passes_under_saved_tensor_hooks(hooks, variant, mode):
    """Activation checkpointing and activations kept on the host, around a stem, a downsampling layer and a block: the gradients
    without them (the same kernels on the same values; the library's convolution gradients sum in an order of their own)."""
    from torch.autograd.graph import save_on_cpu
    from torch.utils.checkpoint import checkpoint
    from oriented1d_amd.convnext1d import ConvNeXt1D
    torch.manual_seed(9)
    net = ConvNeXt1D(depths=(1, 1, 1, 1), dims=(16, 32, 64, 128), variant=variant, stem_dim1=64, num_classes=8,
                     layer_scale_init_value=0.5, arbitrary_size=True).cuda()
    img = torch.randn(2, 3, 36, 44, device="cuda")

    def part(x):
        return net.stages[1](net._downsample(1, net.stages[0](net._downsample(0, x))))
    grads = []
    for hooked in (False, True):
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=BF16, enabled=mode == "autocast"):
            if not hooked:
                y = part(img)
            elif hooks == "checkpoint":
                y = checkpoint(part, img, use_reentrant=False)
            else:
                with save_on_cpu():
                    y = part(img)
        y.float().square().sum().backward()
        grads.append([p.grad for p in net.parameters() if p.grad is not None])
    assert len(grads[0]) == len(grads[1]) > 20
    for a, b in zip(*grads):
        close(a, b.double(), 1e-5, "gradient")


@pytest.mark.parametrize("variant", ["1d", "1dpp"])
@pytest.mark.parametrize("mode", ["autocast", "bf16", "f32"])
def test_network_gradients_against_the_composition(variant, mode, monkeypatch):
    """A training pass on these kernels and on the PyTorch composition of the same network."""
    from oriented1d_amd.convnext1d import ConvNeXt1D
    torch.manual_seed(3)
    net = ConvNeXt1D(depths=(1, 2, 1, 1), dims=(16, 32, 64, 128), variant=variant, num_classes=16,
                     layer_scale_init_value=0.5, arbitrary_size=True).cuda()
    net = net.to(BF16) if mode == "bf16" else net
    img = torch.randn(3, 3, 72, 56, device="cuda").to(BF16 if mode == "bf16" else F32)
    grads = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(fused, "_recording", lambda *t: False)
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=BF16, enabled=mode == "autocast"):
            y = net(img)
        y.float().square().sum().backward()
        grads.append([y.detach()] + [p.grad for p in net.parameters() if p.grad is not None])
    assert len(grads[0]) == len(grads[1])
    tol = 2e-5 if mode == "f32" else 4e-2  # (16-bit: two sets of roundings through the whole network)
    for a, b in zip(*grads):
        assert a.dtype == b.dtype and a.shape == b.shape
        e = (a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-20)
        assert e <= tol, (tuple(a.shape), float(e))


def test_row_norm_gelu_of_infinities():
    """The cheaper erf of 16-bit outputs gives what u * (1 + erf) gives where LayerNorm's parameters overflow."""
    x = torch.randn(4, 64, device="cuda").to(F16).requires_grad_(True)
    w, b = torch.ones(64, device="cuda"), torch.zeros(64, device="cuda")
    b[:3] = torch.tensor([float("inf"), float("-inf"), float("nan")])
    y = fused._RowNorm.apply(x, w, b, 1e-6, 1, F16)
    z = F.gelu(F.layer_norm(x.float(), (64,), w, b, 1e-6)).to(F16)
    assert torch.equal(torch.isnan(y), torch.isnan(z)) and torch.equal(torch.isinf(y), torch.isinf(z))


@pytest.mark.parametrize("dtype", [F32, BF16], ids=str)
@pytest.mark.parametrize("N,C,H,W,K,stride", [(1, 64, 17, 17, 31, 1), (1, 64, 58, 58, 31, 1), (2, 64, 20, 33, 7, 2),
                                              (3, 128, 21, 45, 15, 2), (1, 256, 62, 62, 7, 1), (2, 64, 130, 70, 27, 2)])
def test_grouped_wgrad_of_few_planes(N, C, H, W, K, stride, dtype):
    """Channels grouped by orientation, fewer planes than workgroup slots: the grouped kernels against the tile kernels (the
    same call without the claim); both sum fp32 products of the same values in fp32."""
    from oriented1d_amd import _lib
    from oriented1d_amd.convnext1d import channel_angles
    from oriented1d_amd.dwoconv1d import build_taps
    torch.manual_seed(H)
    taps = build_taps(torch.tensor(channel_angles(C)), C, K).cuda()
    x = torch.randn(N, H, W, C, device="cuda").to(dtype)
    dy = torch.randn(N, -(-H // stride), -(-W // stride), C, device="cuda").to(dtype)
    host = _lib.host(0)
    got = host.wgrad(dy, x, taps, K, stride, _lib.NHWC + _lib.GROUPED, True)
    ref = host.wgrad(dy, x, taps, K, stride, _lib.NHWC, True)
    for a, b in zip(got, ref):
        close(a, b.double(), 1e-5, "wgrad")
