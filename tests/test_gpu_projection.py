"""Weight and bias gradients of the blocks' projections against float64: results that end inside a 128 x 128 tile, token
counts around a step of 64 and a chunk of 256, strided rows, an expanded gradient.  Bound: products of 16-bit values are
exact in fp32 (fp32 products add their own 2^-24, covered by the same bound), so a gradient is an fp32 sum of `tokens` terms, whose error stays below 2^-24 * sqrt(tokens) * 4 of the root
mean square of its terms times tokens, and one rounding to the type."""
import pytest
import torch
import torch.nn as nn

from helpers import UNIT_ROUNDOFF
from flash_bla.ops import projection
from flash_bla.ops.projection import TokenLinear, runs_on_rows


def _gradients(layer, x, g, x64=None):
    y = layer(x)
    y.backward(g)
    return y, layer.weight.grad, None if layer.bias is None else layer.bias.grad


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,N,M,bias,layout", [
    (1, 8, 8, True, "plain"), (63, 64, 136, True, "plain"), (64, 72, 128, False, "plain"), (257, 128, 120, True, "strided"),
    (511, 256, 264, True, "expanded"), (4096 + 65, 64, 128, True, "strided"), (3000, 640, 640, False, "plain")])
def test_weight_gradient(tokens, N, M, bias, layout, dtype, monkeypatch):
    monkeypatch.setattr(projection, "splits_tokens", lambda *a: True)
    torch.manual_seed(tokens)
    layer = TokenLinear(N, M, bias=bias).cuda().to(dtype)
    wide = torch.randn(1, tokens, 2 * N if layout == "strided" else N, device="cuda").to(dtype).requires_grad_()
    x = wide[..., :N]
    g = torch.randn(1, tokens, 3 * M if layout == "strided" else M, device="cuda").to(dtype)[..., -M:]
    if layout == "expanded":
        g = g[:, :1].expand(1, tokens, M)
    assert runs_on_rows(x, layer.weight, layer.bias)
    y, dw, db = _gradients(layer, x, g)
    x64, g64 = x.detach().double().reshape(tokens, N), g.double().reshape(tokens, M)
    slack = 2.0 ** -24 * 4 * tokens ** 0.5
    u = UNIT_ROUNDOFF[dtype]
    want = g64.t() @ x64
    rms = (g64.square().t() @ x64.square() / tokens).sqrt()
    assert ((dw.double() - want).abs() <= u * want.abs() + slack * rms * tokens ** 0.5 + 2.0 ** -24).all()
    if bias:
        want, rms = g64.sum(0), (g64.square().mean(0)).sqrt()
        # equal terms (the expanded gradient) round alike in every addition, so the errors add up instead of averaging out: at
        # most 2^-24 of the sum of magnitudes for each of the additions one after the other, 32 in a lane (256 tokens, 8 rows
        # at a time), 8 over the rows and 2 over the chunks
        alike = 42 * 2.0 ** -24 * g64.abs().sum(0) if layout == "expanded" else 0.0
        assert ((db.double() - want).abs() <= u * want.abs() + slack * rms * tokens ** 0.5 + 2.0 ** -24 + alike).all()
    assert torch.equal(y, nn.functional.linear(x, layer.weight, layer.bias))
    dx = wide.grad[..., :N]
    assert torch.equal(dx, g @ layer.weight) and (layout != "strided" or wide.grad[..., N:].abs().max() == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,N,M,bias", [
    (8192, 640, 640, False),  # 25 tiles, 19 chunks of 448: two groups of eight on one XCD each, three in plain order
    (40001, 136, 264, True),  # 6 tiles, 79 chunks of 512, the last of 65: nine groups and seven
    (50176, 256, 512, True),  # 8 tiles, 61 chunks of 832: seven groups and five
    (131072, 64, 128, True),  # one tile, 512 chunks of 256: plain order throughout
    (200704, 64, 128, True)])  # one tile, 448 chunks of 448: groups throughout
def test_weight_gradient_of_chunks_that_share_an_xcd(tokens, N, M, bias, dtype, monkeypatch):
    test_weight_gradient(tokens, N, M, bias, "plain", dtype, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,M", [(1024, 128), (50176, 512), (12544, 256), (200704, 128)])
def test_fp32_bias_gradient_is_close_to_exact(tokens, M, monkeypatch):
    """Four rows in 32 bits, the rest of the sum in 64: measured 3.5e-8 to 5.6e-8 (32-bit sums 1.1e-7 to 2.1e-7, torch's
    column sums 0.8e-7 to 2.5e-7)."""
    monkeypatch.setattr(projection, "splits_tokens", lambda *a: True)
    torch.manual_seed(tokens)
    layer = TokenLinear(64, M).cuda()
    x, g = torch.randn(tokens, 64, device="cuda"), torch.randn(tokens, M, device="cuda")
    assert runs_on_rows(x, layer.weight, layer.bias)
    _, _, db = _gradients(layer, x, g)
    want = g.double().sum(0)
    assert (db.double() - want).norm() <= 8e-8 * want.norm()


@pytest.mark.gpu
def test_gradient_of_the_gradient(monkeypatch):
    monkeypatch.setattr(projection, "splits_tokens", lambda *a: True)
    torch.manual_seed(0)
    layer = TokenLinear(16, 8).cuda().half()
    plain = nn.Linear(16, 8).cuda().half()
    plain.load_state_dict(layer.state_dict())
    results = []
    for f in (layer, plain):
        x = torch.linspace(-1, 1, 96, device="cuda").half().reshape(6, 16).requires_grad_()
        dw, = torch.autograd.grad(f(x).square().sum(), f.weight, create_graph=True)
        dw.square().sum().backward()
        results.append((x.grad, f.weight.grad))
    for a, b in zip(*results):
        torch.testing.assert_close(a, b, rtol=2e-2, atol=2e-2 * b.abs().max().item())


def test_other_calls_are_plain_linear():
    layer = TokenLinear(16, 8)
    x = torch.randn(3, 16)
    assert not runs_on_rows(x, layer.weight, layer.bias)
    assert torch.equal(layer(x), nn.functional.linear(x, layer.weight, layer.bias))
    assert isinstance(layer, nn.Linear) and list(layer.state_dict()) == ["weight", "bias"]
