"""Depth-wise convolution of token rows against the same convolution in float64: filter sizes, grids whose width is not a
multiple of the kernels' strips of 7 or 8 columns (and narrower than the filter), channel counts that end inside a
64-channel block, filters shared between heads, strided rows (a chunk of a joint projection), both gradients.

Bounds: a value is one fp32 sum of at most 49 products rounded once (u = unit roundoff of the type); a filter gradient is
an fp32 sum over B*H*W tokens, whose rounding error stays below 2^-24 * sqrt(terms) * 4 of the sum of magnitudes."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from helpers import UNIT_ROUNDOFF
from flash_bla.ops.depthwise import depthwise_conv_tokens, runs_on_tokens

pytestmark = pytest.mark.gpu

SHAPES = [  # B, H, W, heads, Cw, K
    (2, 9, 7, 1, 64, 3), (1, 5, 8, 2, 32, 5), (3, 4, 15, 3, 24, 5), (2, 1, 1, 1, 8, 3), (1, 2, 2, 2, 8, 7),
    (2, 17, 23, 1, 136, 7), (1, 56, 56, 2, 32, 3), (4, 3, 29, 5, 16, 5),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_convolution_and_gradients(shape, dtype):
    B, H, W, heads, Cw, K = shape
    C, N = heads * Cw, H * W
    torch.manual_seed(B * 1000 + W)
    conv = nn.Conv2d(Cw, Cw, K, padding=K // 2, groups=Cw).cuda().to(dtype)
    joint = torch.randn(B, N, 3 * C, device="cuda").to(dtype).requires_grad_()
    x = joint.chunk(3, dim=-1)[1]
    g = torch.randn(B, N, 2 * C, device="cuda").to(dtype)[..., :C]
    assert runs_on_tokens(x, conv)
    y = depthwise_conv_tokens(x, conv, H, W)
    y.backward(g)

    w64 = conv.weight.detach().double().repeat(heads, 1, 1, 1).requires_grad_()
    b64 = conv.bias.detach().double().repeat(heads).requires_grad_()
    image = x.detach().double().transpose(1, 2).reshape(B, C, H, W)
    rows = image.clone().requires_grad_()
    ref = F.conv2d(rows, w64, b64, padding=K // 2, groups=C)
    ref.backward(g.double().transpose(1, 2).reshape(B, C, H, W))
    u = UNIT_ROUNDOFF[dtype]
    as_rows = lambda t: t.reshape(B, C, N).transpose(1, 2)  # noqa: E731
    magnitude = F.conv2d(image.abs(), w64.detach().abs(), b64.detach().abs(), padding=K // 2, groups=C)
    err = (y.double() - as_rows(ref)).abs()
    assert (err <= u * as_rows(ref).abs() + 2.0 ** -24 * 50 * as_rows(magnitude)).all(), err.max()
    dx = joint.grad.chunk(3, dim=-1)[1].double()
    want = as_rows(rows.grad)
    assert (dx - want).abs().max() <= (u + 2.0 ** -24 * 50) * want.abs().max()
    assert joint.grad.chunk(3, dim=-1)[0].abs().max() == 0
    dw = w64.grad.view(heads, Cw, 1, K, K).sum(0)
    db = b64.grad.view(heads, Cw).sum(0)
    terms = B * N * heads
    slack = 2.0 ** -24 * 4 * terms ** 0.5
    scale = (x.detach().double().square().mean() * g.double().square().mean()).sqrt() * terms
    assert ((conv.weight.grad.double() - dw).abs() <= u * dw.abs() + slack * scale).all()
    assert ((conv.bias.grad.double() - db).abs() <= u * db.abs() + slack * g.double().abs().mean() * terms).all()


def test_what_the_kernels_do_not_take_runs_as_the_torch_convolution():
    for conv, C in ((nn.Conv2d(12, 12, 3, padding=1, groups=12), 12), (nn.Conv2d(16, 16, 9, padding=4, groups=16), 32)):
        conv = conv.cuda()
        x = torch.randn(2, 20, C, device="cuda")[..., :C]
        assert runs_on_tokens(x, conv) == (conv.kernel_size[0] == 3)
        y = depthwise_conv_tokens(x, conv, 4, 5)
        rep = C // conv.weight.shape[0]
        want = F.conv2d(x.double().transpose(1, 2).reshape(2, C, 4, 5), conv.weight.double().repeat(rep, 1, 1, 1),
                        conv.bias.double().repeat(rep), padding=conv.padding, groups=C).reshape(2, C, 20).transpose(1, 2)
        assert (y.double() - want).abs().max() <= 1e-5 * want.abs().max()


def test_hooks_run_and_the_gradient_has_a_gradient():
    torch.manual_seed(0)
    conv = nn.Conv2d(8, 8, 3, padding=1, groups=8).cuda()
    x = torch.randn(2, 12, 16, device="cuda", requires_grad=True)
    g, = torch.autograd.grad(depthwise_conv_tokens(x, conv, 3, 4).square().sum(), x, create_graph=True)
    ours = torch.autograd.grad(g.square().sum(), (x, conv.weight, conv.bias))
    seen = []
    conv.register_forward_hook(lambda *a: seen.append(1))
    assert not runs_on_tokens(x, conv)
    g, = torch.autograd.grad(depthwise_conv_tokens(x, conv, 3, 4).square().sum(), x, create_graph=True)
    want = torch.autograd.grad(g.square().sum(), (x, conv.weight, conv.bias))
    assert seen
    for a, b in zip(ours, want):  # fp32 sums of 9 products, twice: a few 2^-24 of the largest
        assert (a - b).abs().max() <= 2.0 ** -18 * b.abs().max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("where", ["input", "gradient", "filters"])
@pytest.mark.parametrize("H,W,K", [(3, 9, 3), (4, 20, 5), (2, 3, 7), (3, 14, 3), (2, 16, 5), (2, 1, 3)])
def test_infinities_and_nan_meet_what_lies_on_the_grid_alone(H, W, K, where, dtype):
    """What surrounds the grid has no products, not zeros: infinities in the first and last columns (or in the outer taps of
    a filter) and a NaN, whether the last strip of a row ends with the row or behind it, against the products of the
    overlapping parts in float64 (which is what torch's convolutions in 16 and 32 bits give).  Whole numbers small enough to
    be exact in every type."""
    torch.manual_seed(W)
    numbers = lambda *shape: torch.randint(-2, 3, shape, device="cuda").to(dtype)  # noqa: E731
    x, g, w = numbers(2, H, W, 16), numbers(2, H, W, 16), numbers(8, 1, K, K)
    inf, nan = float("inf"), float("nan")
    if where == "filters":
        w[:3, :, :, 0], w[2:4, :, :, -1], w[4, 0, 0, K // 2], w[5, 0, K // 2, 0] = inf, -inf, inf, nan
    else:
        t = x if where == "input" else g
        t[:, :, -1, :6], t[:, :, 0, 4:8], t[:, 0, :, 9], t[1, -1, -1, 10] = inf, -inf, inf, nan
    conv = nn.Conv2d(8, 8, K, padding=K // 2, groups=8, bias=False).cuda().to(dtype)
    conv.weight.data.copy_(w)
    rows = x.reshape(2, H * W, 16).requires_grad_()
    assert runs_on_tokens(rows, conv)
    y = depthwise_conv_tokens(rows, conv, H, W)
    y.backward(g.reshape(2, H * W, 16))

    x64, w64, P = x.double().requires_grad_(), w.double().requires_grad_(), K // 2
    want = torch.zeros_like(x64)
    for ky in range(K):
        for kx in range(K):  # output rows and columns whose neighbour at this tap lies on the grid
            rows_out, columns_out = (slice(max(0, P - k), min(n, n + P - k)) for k, n in ((ky, H), (kx, W)))
            rows_in, columns_in = (slice(max(0, k - P), min(n, n + k - P)) for k, n in ((ky, H), (kx, W)))
            want = want.clone()
            if rows_out.start < rows_out.stop and columns_out.start < columns_out.stop:
                want[:, rows_out, columns_out] += x64[:, rows_in, columns_in] * w64[:, 0, ky, kx].repeat(2)
    want.backward(g.double())
    for name, a, b in (("y", y, want), ("dx", rows.grad, x64.grad), ("dw", conv.weight.grad, w64.grad)):
        b = b.detach().reshape(a.shape).to(dtype)
        torch.testing.assert_close(a.detach(), b, rtol=0, atol=0, equal_nan=True, msg=lambda m: f"{name}: {m}")


@pytest.mark.parametrize("shape", [(2, 9, 7, 1, 64, 3), (4, 28, 28, 8, 32, 5), (2, 17, 23, 1, 136, 7)])
def test_fp32_sums_are_rounded_once(shape):
    """As torch's convolution in fp32: products and sums in 64 bits, one rounding (2^-24 of the value; the sums themselves
    are off by less than 50 x 2^-53 of the magnitudes)."""
    B, H, W, heads, Cw, K = shape
    torch.manual_seed(K)
    conv = nn.Conv2d(Cw, Cw, K, padding=K // 2, groups=Cw).cuda()
    x, g = (torch.randn(B, H * W, heads * Cw, device="cuda") for _ in range(2))
    x.requires_grad_()
    y = depthwise_conv_tokens(x, conv, H, W)
    dx, = torch.autograd.grad(y, x, g)
    rows = x.detach().double().requires_grad_()
    image = rows.transpose(1, 2).reshape(B, heads * Cw, H, W)
    want = F.conv2d(image, conv.weight.double().repeat(heads, 1, 1, 1), conv.bias.double().repeat(heads), padding=K // 2,
                    groups=heads * Cw).reshape(B, heads * Cw, H * W).transpose(1, 2)
    exact_dx, = torch.autograd.grad(want, rows, g.double())
    for a, b in ((y, want), (dx, exact_dx)):
        assert ((a.double() - b).abs() <= 2.0 ** -24 * b.abs() + 2.0 ** -46).all()


def test_fp32_bias_gradient_is_close_to_exact():
    """Sums of the gradient alone in 64 bits: what is left is the chunks' rounding and the result's, 2^-25 each (root mean
    square; 32-bit sums are at 1.1e-7 to 1.5e-7 here)."""
    for B, H, W, heads, Cw, K in ((4, 28, 28, 8, 32, 5), (8, 56, 56, 1, 64, 3), (2, 20, 20, 2, 64, 7)):
        torch.manual_seed(K)
        conv = nn.Conv2d(Cw, Cw, K, padding=K // 2, groups=Cw).cuda()
        x, g = (torch.randn(B, H * W, heads * Cw, device="cuda") for _ in range(2))
        db, = torch.autograd.grad(depthwise_conv_tokens(x, conv, H, W), conv.bias, g)
        want = g.double().sum((0, 1)).view(heads, Cw).sum(0)
        assert (db.double() - want).norm() <= 2 * 2.0 ** -25 * want.norm()
