"""The vision blocks' fused elementwise steps against their torch compositions in float64: channel counts that fill one
64-piece block of the gradient kernel, end inside one and need several, heads of one piece and more, fewer keys than queries,
one token, batches that split into groups, zeros and negative zeros, gates that are part of a wider row.

Bounds: a value is computed in fp32 from inputs that are exact in float64 and rounded once (u); the powers' exponent
p log2 a, at most 2^6 here, carries the fp32 functions' 2^-22 to 2^-16 of the value; a turned
channel is a difference of two products, each off by a few 2^-24 of the pair's length: 2^-22 of the largest result; sums over
tokens (a few hundred terms) stay within 2^-16 of the largest result."""
import pytest
import torch

from helpers import UNIT_ROUNDOFF
from flash_bla.layers import FocusedLinearAttention, MambaLikeLinearAttention, PolaLinearAttention
from flash_bla.layers import _features as features

DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _check(function, formula, inputs, dtype):
    """Outputs and gradients of function(*inputs) against formula in float64 on the same values."""
    rest = [t for t in inputs if not torch.is_tensor(t)]
    ours = [t.detach().requires_grad_(t.requires_grad) for t in inputs if torch.is_tensor(t)]
    exact = [t.detach().double().requires_grad_(t.requires_grad) for t in ours]
    out, want = function(*ours, *rest), formula(*exact, *rest)
    assert len(out) == len(want)
    grads = [torch.randn(o.shape, device="cuda").to(dtype) for o in out]
    leaves = [t for t in ours if t.requires_grad]
    got = torch.autograd.grad(out, leaves, grads)
    ref = torch.autograd.grad(want, [t for t in exact if t.requires_grad], [g.double() for g in grads])
    u = UNIT_ROUNDOFF[dtype]
    for name, a, b in [("out", a, b) for a, b in zip(out, want)] + [("grad", a, b) for a, b in zip(got, ref)]:
        assert a.shape == b.shape and a.dtype == dtype
        slack = 2.0 ** -16 * (b.abs() if name == "out" else b.abs().max()) + 2.0 ** -22 * b.abs().max()
        assert ((a.double() - b).abs() <= u * b.abs() + slack).all(), (name, (a.double() - b).abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,N,Nk,heads,d", [(1, 1, 1, 1, 8), (2, 33, 33, 8, 64), (3, 20, 5, 5, 24), (9, 49, 49, 2, 32),
                                            (2, 7, 7, 10, 64), (37, 4, 1, 3, 40)])
def test_polarity_features(B, N, Nk, heads, d, dtype):
    torch.manual_seed(N * heads)
    C = heads * d
    # half-width inputs: fifth powers of the largest stay inside fp16's range
    values = lambda *shape: (0.5 * torch.randn(shape, device="cuda")).to(dtype).requires_grad_()  # noqa: E731
    qg, kv, pe = values(B, N, 2 * C), values(B, Nk, 2 * C), values(1, Nk, C)
    with torch.no_grad():
        qg.view(-1)[::7] = 0.0
        qg.view(-1)[1::11] = -0.0
    scale = (0.5 + torch.rand(1, 1, C, device="cuda")).to(dtype).requires_grad_()
    power = (1 + 4 * torch.rand(1, heads, 1, d, device="cuda")).to(dtype).requires_grad_()
    assert features._takes(heads, C, 1, qg, kv, pe, scale, power)

    _check(features.polarity_features, features.polarity_formula, (qg, kv, pe, scale, power, heads), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,side,heads,d", [(1, 1, 1, 8), (3, 5, 3, 24), (2, 14, 2, 32), (2, 3, 10, 64)])
def test_rotary_features(B, side, heads, d, dtype):
    torch.manual_seed(side)
    C = heads * d
    qk = torch.randn(B, side * side, 2 * C, device="cuda").to(dtype).requires_grad_()
    x = torch.randn(B, side * side, C, device="cuda").to(dtype).requires_grad_()
    angles = torch.randn(side, side, C // 2, device="cuda")
    rotations = torch.stack([angles.cos(), angles.sin()], dim=-1)

    def exact(qk, x, side, heads):
        q, k = (torch.nn.functional.elu(qk) + 1).chunk(2, dim=-1)
        cos, sin = rotations.double().reshape(side * side, C // 2, 2).unbind(-1)
        turn = lambda t: torch.stack([t[..., ::2] * cos - t[..., 1::2] * sin,  # noqa: E731
                                      t[..., ::2] * sin + t[..., 1::2] * cos], dim=-1).flatten(-2)
        return (*(features.split_heads(t, heads) for t in (q, k, turn(q), turn(k), x)), x)
    _check(lambda qk, x, side, heads: features.rotary_features(qk, x, rotations, side, heads), exact, (qk, x, side, heads),
           dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,side,heads,d", [(1, 1, 1, 8), (3, 5, 3, 32), (2, 7, 2, 64), (1, 2, 2, 128)])
def test_turned_heads(B, side, heads, d, dtype):
    torch.manual_seed(side)
    q, k = (torch.randn(B, heads, side * side, d, device="cuda").to(dtype).requires_grad_() for _ in range(2))
    weight = torch.rand(B, heads, side * side, 1, device="cuda").to(dtype).requires_grad_()
    angles = torch.randn(side, side, d // 2, device="cuda")
    rotations = torch.stack([angles.cos(), angles.sin()], dim=-1)

    def exact(q, k, weight):
        cos, sin = rotations.double().reshape(side * side, d // 2, 2).unbind(-1)
        turn = lambda t: torch.stack([t[..., ::2] * cos - t[..., 1::2] * sin,  # noqa: E731
                                      t[..., ::2] * sin + t[..., 1::2] * cos], dim=-1).flatten(-2)
        return k * weight, turn(q), turn(k * weight)
    _check(lambda *t: features.turned_heads(*t, rotations), exact, (q, k, weight), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("halves", [False, True])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("B,N,heads,d", [(1, 1, 1, 16), (3, 21, 5, 48), (2, 50, 10, 64)])
def test_merged_heads(B, N, heads, d, gated, halves, dtype):
    torch.manual_seed(N)
    values = lambda *shape: torch.randn(shape, device="cuda").to(dtype).requires_grad_()  # noqa: E731
    tensors = [values(B, heads, N, d // 2 if halves else d) for _ in range(1 + halves)] + [values(B, N, heads * d)]
    tensors += [values(B, N, 4 * heads * d)] if gated else []

    def arguments(*t):
        return t[0], t[1] if halves else None, t[1 + halves], t[-1][..., -heads * d:] if gated else None
    _check(lambda *t: (features.merge_heads_with(*arguments(*t)),), lambda *t: features.merge_formula(*arguments(*t)),
           tensors, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,n,tokens,C", [(1, 1, 1, 8), (2, 1, 5, 24), (3, 7, 28, 64), (2, 49, 200, 40), (1, 30, 11, 16),
                                          (2, 5, 5, 8), (1, 3, 1, 8)])
def test_interpolated_tokens(B, n, tokens, C, dtype):
    torch.manual_seed(n)
    kv = torch.randn(B, n, 2 * C, device="cuda").to(dtype).requires_grad_()
    _check(lambda t: (features.interpolate_tokens(t[..., C:], tokens),),
           lambda t: features.interpolate_formula(t[..., C:], tokens), [kv], dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,N,Nk,heads,d", [(1, 1, 1, 1, 16), (2, 33, 33, 8, 32), (3, 20, 5, 5, 24), (37, 5, 1, 3, 40),
                                            (2, 7, 7, 10, 64), (1, 9, 4, 16, 64)])
def test_focused_features(B, N, Nk, heads, d, dtype):
    torch.manual_seed(N * heads)
    C = heads * d
    values = lambda *shape: torch.randn(shape, device="cuda").to(dtype).requires_grad_()  # noqa: E731
    q, kv, pe = values(B, N, C), values(B, Nk, 2 * C), values(1, Nk, C)
    scale = (0.5 + torch.rand(1, 1, C, device="cuda")).to(dtype).requires_grad_()
    assert features._takes(heads, C, 1, q, kv, pe, scale)
    _check(lambda *a: features.focused_features(*a, 3), features.focus_formula, (q, kv, pe, scale, heads), dtype)
    for a, b in zip(features.focused_features(q, kv, pe, scale, heads, 2.5),
                    features.focus_formula(q, kv, pe, scale, heads, 2.5)):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(3))
@pytest.mark.parametrize("name", ["polarity", "focused"])
def test_fp32_features_are_no_further_from_exact_than_torch_operators(name, seed):
    """Distance from float64 of the features and of the gradients of the projections' rows and of the positional term, ours
    and the composition's (measured 0.92 to 1.03 of it; with reciprocals in place of quotients 1.13 to 1.30).  The gradients
    of scale and power are sums over all tokens, few and cancelling: not compared."""
    torch.manual_seed(seed)
    B, N, heads, d = 8, 196, 8, 32
    C = heads * d
    values = lambda *shape: (0.5 * torch.randn(shape, device="cuda")).requires_grad_()  # noqa: E731
    scale = (0.5 + torch.rand(1, 1, C, device="cuda")).requires_grad_()
    if name == "polarity":
        power = (1 + 4 * torch.rand(1, heads, 1, d, device="cuda")).requires_grad_()
        inputs, rest = [values(B, N, 2 * C), values(B, N, 2 * C), values(1, N, C), scale, power], (heads,)
        fused, formula, kept = features.polarity_features, features.polarity_formula, 3
    else:
        inputs, rest = [values(B, N, C), values(B, N, 2 * C), values(1, N, C), scale], (heads, 3)
        fused, formula, kept = features.focused_features, features.focus_formula, 2
    assert features._takes(heads, C, 1, *inputs)
    grads = [torch.randn_like(o) for o in fused(*inputs, *rest)]
    exact = [t.detach().double().requires_grad_() for t in inputs]

    def results(function, inputs, grads):
        out = function(*inputs, *rest)
        return [*out[:kept], *torch.autograd.grad(out, inputs, grads)[:3]]
    want = results(formula, exact, [g.double() for g in grads])
    ours, torchs = ([float((a.double() - b).norm() / b.norm()) for a, b in zip(results(f, inputs, grads), want)]
                    for f in (fused, formula))
    assert all(a <= 1.08 * b for a, b in zip(ours, torchs)), (ours, torchs)


@pytest.mark.gpu
def test_not_a_number_and_infinity_pass_through():
    """A NaN reaches both parts, an infinity its own, as relu and pow give them."""
    x = torch.randn(1, 1, 64, device="cuda")
    x[0, 0, 3], x[0, 0, 4], x[0, 0, 5] = float("nan"), float("inf"), -float("inf")
    pe, one = torch.zeros(1, 1, 32, device="cuda"), torch.ones(1, 1, 32, device="cuda")
    args = (x, x.clone(), pe, one, 2 * one.reshape(1, 1, 1, 32), 1)
    for a, b in zip(features.polarity_features(*args), features.polarity_formula(*args)):
        torch.testing.assert_close(a, b, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("power", [1.0, 1.5, 3.0])
def test_gradients_at_infinities_denormals_and_a_power_of_one(power, dtype):
    """One channel each, so that nothing is added to them: as relu and pow give them, in float64 and rounded."""
    x = torch.tensor([float("inf"), -float("inf"), 1e-40, -1e-40, 0.0, 3.0, -3.0, float("nan")], device="cuda")
    zero, one = torch.zeros(1, 1, 8, device="cuda"), torch.ones(1, 1, 8, device="cuda")
    inputs = [t.to(dtype).requires_grad_() for t in (torch.cat([x, x])[None, None], torch.cat([x, x])[None, None], zero, one,
                                                     power * one.reshape(1, 1, 1, 8))]
    exact = [t.detach().double().requires_grad_() for t in inputs]
    out, want = features.polarity_features(*inputs, 1), features.polarity_formula(*exact, 1)
    for a, b in zip(out, want):
        torch.testing.assert_close(a, b.to(dtype), equal_nan=True)
    got = torch.autograd.grad(sum(o.float().sum((0, 1)).sum() for o in out[:3]), inputs)
    ref = torch.autograd.grad(sum(o.sum((0, 1)).sum() for o in want[:3]), exact)
    for name, a, b in zip(("qg", "kv", "pe", "scale", "power"), got, ref):
        torch.testing.assert_close(a, b.to(dtype), equal_nan=True, msg=lambda m: f"{name}: {m}")


@pytest.mark.gpu
@pytest.mark.parametrize("make,extra", [(lambda: PolaLinearAttention(24, 4, num_heads=2), (2, 2)),
                                        (lambda: MambaLikeLinearAttention(24, (2, 2), 2), ())])
def test_heads_that_are_no_whole_pieces_run_as_torch_operators(make, extra):
    """12 channels a head in fp16: no 16-byte pieces, the compositions run."""
    torch.manual_seed(0)
    block = make().cuda().half()
    if hasattr(block, "rope"):
        block.rope.float()
    x = torch.randn(2, 4, 24, device="cuda", dtype=torch.float16, requires_grad=True)
    y = block(x, *extra)
    y.square().sum().backward()
    exact = block.double()(x.detach().double(), *extra, mode="torch") if extra else None
    assert torch.isfinite(x.grad).all() and (exact is None or (y.double() - exact).norm() <= 5e-3 * exact.norm())


@pytest.mark.gpu
def test_gradient_of_the_gradient():
    torch.manual_seed(0)
    results = []
    for f in (features.merge_heads_with, lambda *t: features.merge_formula(*t)[0]):
        t = [torch.linspace(-1, 1, 64, device="cuda").reshape(s).requires_grad_()
             for s in ((1, 2, 4, 8), (1, 4, 16), (1, 4, 16))]
        g = torch.autograd.grad(f(t[0], None, t[1], t[2]).square().sum(), t, create_graph=True)
        results.append(torch.autograd.grad(sum(x.square().sum() for x in g), t))
    for a, b in zip(*results):
        torch.testing.assert_close(a, b)


@pytest.mark.gpu
def test_heads_that_do_not_divide_the_channels_are_not_taken():
    x = torch.zeros(1, 1, 136, device="cuda").half()
    assert features._takes(17, 136, 1, x) and not features._takes(16, 136, 1, x)  # 136 // 16 is one whole piece


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["mlla", "pola", "focused"])
def test_batches_of_gradients(name):
    """is_grads_batched through what follows the attention, where the kernels find no addresses: as one by one."""
    torch.manual_seed(0)
    block, extra = {"mlla": (MambaLikeLinearAttention(64, (4, 4), 2), ()), "pola": (PolaLinearAttention(64, 16, num_heads=2), (4, 4)),
                    "focused": (FocusedLinearAttention(64, 16, num_heads=2), (4, 4))}[name]
    block = block.cuda()
    x = torch.randn(2, 16, 64, device="cuda")
    wanted = [p for n, p in block.named_parameters() if n.startswith(("proj", "dwc", "lepe"))]
    y = block(x, *extra)
    g = torch.randn(3, *y.shape, device="cuda")
    batched = torch.autograd.grad(y, wanted, g, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(batched, torch.autograd.grad(y, wanted, g[i], retain_graph=True)):
            # fp32 sums of 32 products in another order
            assert (a[i] - b).abs().max() <= 2.0 ** -20 * b.abs().max()
