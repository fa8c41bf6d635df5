"""The blocks' attention on their projections' rows (16-bit types, heads of 32 channels): head counts of every workgroup split,
token counts around a wave's 32, tokens of several workgroups, fewer keys than queries, groups of several batches, small
values, a NaN that stays in its batch.

Bounds: as in test_gpu_whole_blocks.py: against float64 no further off than the steps, up to the chance of few roundings (1.25
times, 1.3 u; sums over few values vary more: a hundred output values leave a fifth of the norm to chance)."""
import pytest
import torch

from helpers import UNIT_ROUNDOFF
from flash_bla.layers import MambaLikeLinearAttention, PolaLinearAttention
from test_gpu_whole_blocks import _distance, _exact, _steps, counted  # noqa: F401

pytestmark = pytest.mark.gpu


def _block(kind, heads, H, W, sr, dtype):
    torch.manual_seed(0)
    C = 32 * heads
    if kind == "mlla":
        block = MambaLikeLinearAttention(C, (H, W), heads, qkv_bias=True)
    else:
        block = PolaLinearAttention(C, H * W, num_heads=heads, sr_ratio=sr, qkv_bias=True)
    with torch.no_grad():
        for p in block.parameters():
            if not p.any():
                p.add_(0.1 * torch.randn(p.shape))
    block = block.cuda().to(dtype)
    if kind == "mlla":
        block.rope.float()
    return block, () if kind == "mlla" else (H, W)


#        kind    heads H   W  sr  B   values
CASES = [("mlla", 1, 1, 1, 1, 2, 1.0), ("mlla", 3, 5, 5, 1, 3, 1.0), ("mlla", 4, 6, 6, 1, 2, 1.0), ("mlla", 8, 8, 8, 1, 5, 1.0),
         ("mlla", 2, 9, 9, 1, 1, 2.0 ** -6), ("mlla", 4, 40, 40, 1, 9, 1.0), ("mlla", 6, 28, 28, 1, 70, 1.0),
         ("pola", 1, 3, 11, 1, 3, 1.0), ("pola", 2, 31, 1, 1, 2, 1.0), ("pola", 3, 4, 8, 1, 1, 2.0 ** -6), ("pola", 4, 1, 1, 1, 2, 1.0),
         ("pola", 8, 13, 5, 1, 3, 1.0), ("pola", 4, 14, 14, 2, 5, 1.0), ("pola", 2, 40, 40, 8, 9, 1.0), ("pola", 4, 28, 28, 1, 70, 1.0),
         ("pola", 4, 40, 40, 1, 2, 1.0),
         ("mlla", 1, 72, 72, 1, 1, 1.0), ("pola", 1, 72, 72, 1, 1, 1.0)]  # (more tiles than a head may leave partials)


@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("kind,heads,H,W,sr,B,values", CASES)
def test_against_float64(kind, heads, H, W, sr, B, values, dtype, counted, monkeypatch):  # noqa: F811
    block, extra = _block(kind, heads, H, W, sr, dtype)
    x = torch.randn(B, H * W, 32 * heads, device="cuda").to(dtype)
    with torch.no_grad():
        if kind == "mlla":
            x *= values
        else:
            block.kv.weight[32 * heads:] *= values
            block.kv.bias[32 * heads:] *= values
    g = torch.randn_like(x)
    results = []
    for whole in (True, False):
        leaf = x.detach().requires_grad_()
        block.zero_grad(set_to_none=True)
        out = block(leaf, *extra) if whole else _steps(block, monkeypatch, lambda b: b(leaf, *extra))
        out.backward(g)
        results.append([out.detach(), leaf.grad] + [p.grad for p in block.parameters()])
    assert len(counted) == 1
    u = UNIT_ROUNDOFF[dtype]
    names = ["out", "x"] + [n for n, _ in block.named_parameters()]
    for name, a, b, e in zip(names, *results, _exact(block, x, extra, g)):
        if H * W == 1 and e.norm() < 1e-6:
            # One token: numerator and denominator are the same product, so the exact gradients of queries and keys are those of
            # eps, next to nothing, and what is left is the rounding of a difference of two equal fp32 terms, sums of 32 products
            # of output and output gradient: below 32 * 2^4 * 2^-23 = 2^-14 an element.
            assert float(a.abs().max()) <= 2.0 ** -14, name
            continue
        assert _distance(a, e) <= 1.25 * _distance(b, e) + 1.3 * u + 2.0 ** -20, (name, _distance(a, e), _distance(b, e))


@pytest.mark.parametrize("kind", ["mlla", "pola"])
def test_nan_stays_in_its_batch(kind, counted):  # noqa: F811
    block, extra = _block(kind, 4, 7, 7, 1, torch.bfloat16)
    x = torch.randn(3, 49, 128, device="cuda").bfloat16()
    bad = x.clone()
    bad[1, 48, 127] = float("nan")
    outs, grads = [], []
    for v in (x, bad):
        leaf = v.requires_grad_()
        out = block(leaf, *extra)
        out.backward(torch.ones_like(out))
        outs.append(out.detach()), grads.append(leaf.grad)
    assert len(counted) == 2 and outs[1][1].isnan().all() and grads[1][1].isnan().all()
    for a, b in (outs, grads):
        assert torch.equal(a[[0, 2]], b[[0, 2]])
