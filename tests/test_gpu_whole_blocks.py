"""Blocks as one native call a direction against the same kernels issued step by step: outputs and every gradient, in each
type, with and without biases, frozen parameters, rows that are no contiguous tensor, expanded gradients; gradients of
gradients and batches of gradients; calls that something looks into run step by step.

Bounds: the two differ in where values are rounded (residuals, normalised rows and gradients that two steps contribute to
are rounded once here, the steps round every part) and in the order of fp32 sums.  Against float64 the whole call is no
further off than the steps, up to the chance of a few thousand roundings (measured 0.7 to 1.1 times; 1.3 u is what two
roundings more would add).  Where the two are compared directly, each is within 8 u of exact in the 2-norm (a value goes
through at most eight roundings one after the other), fp32 sums add 2^-18."""
import copy

import pytest
import torch

from helpers import UNIT_ROUNDOFF
from flash_bla.layers import (FocusedLinearAttention, GeneralizedLinearAttention, MambaLikeLinearAttention,
                              PolaLinearAttention)
from flash_bla.layers import _whole

pytestmark = pytest.mark.gpu

BLOCKS = {
    "mlla": (lambda **k: MambaLikeLinearAttention(64, (6, 6), 2, **k), 36, 64, (), (torch.half, torch.bfloat16, torch.float)),
    "pola": (lambda **k: PolaLinearAttention(64, 36, num_heads=2, **k), 36, 64, (6, 6), (torch.half, torch.bfloat16, torch.float)),
    "pola sr": (lambda **k: PolaLinearAttention(128, 64, num_heads=4, sr_ratio=2, **k), 64, 128, (8, 8), (torch.half, torch.float)),
    "focused": (lambda **k: FocusedLinearAttention(64, 24, num_heads=4, **k), 24, 64, (4, 6), (torch.half, torch.bfloat16, torch.float)),
    "focused sr": (lambda **k: FocusedLinearAttention(64, 64, num_heads=2, sr_ratio=2, **k), 64, 64, (8, 8), (torch.half, torch.float)),
    "linfusion": (lambda qkv_bias=False: GeneralizedLinearAttention(128, heads=2, dim_head=64, bias=qkv_bias), 40, 128, (),
                  (torch.half, torch.bfloat16)),
}
CASES = [(name, dtype) for name in BLOCKS for dtype in BLOCKS[name][-1]]


def _make(name, dtype, seed=0, **kwargs):
    torch.manual_seed(seed)
    make, tokens, dim, extra, _ = BLOCKS[name]
    block = make(**kwargs)
    with torch.no_grad():
        for p in block.parameters():
            if not p.any():
                p.add_(0.1 * torch.randn(p.shape))
    block = block.cuda().to(dtype)
    if hasattr(block, "rope"):
        block.rope.float()
    if name == "linfusion":  # a value whose rounding crosses LeakyReLU's kink changes its gradient by 1 - slope: 0.01 leaves
        for path in (block.to_q_, block.to_k_):  # 2e-2 of a weight's gradient to that chance, 0.9 a tenth of it
            path[2].negative_slope = 0.9
    return block, torch.randn(3, tokens, dim, device="cuda").to(dtype), extra


@pytest.fixture
def counted(monkeypatch):
    """How many calls ran whole, by output."""
    seen = []
    run = _whole._run
    monkeypatch.setattr(_whole, "_run", lambda *a: seen.append(run(*a)) or seen[-1])
    return seen


def _steps(block, monkeypatch, call):
    with monkeypatch.context() as m:
        m.setattr(_whole, "_ordinary", lambda *a: False)
        return call(block)


def _distance(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def _close(a, b, dtype):
    assert a.dtype == b.dtype and a.shape == b.shape and _distance(a, b) <= 16 * UNIT_ROUNDOFF[dtype] + 2.0 ** -18


def _exact(block, x, extra, g):
    """Output and gradients by torch's operators in float64."""
    block = copy.deepcopy(block).double()
    if hasattr(block, "rope"):
        block.rope.float()  # (the rotation is computed in fp32 by the block's own definition)
    leaf = x.detach().double().requires_grad_()
    block.zero_grad(set_to_none=True)
    out = block(leaf, *extra, mode="torch")
    out.backward(g.double())
    return [out.detach(), leaf.grad] + [p.grad for p in block.parameters()]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("name,dtype", CASES)
def test_results_of_the_steps(name, dtype, bias, counted, monkeypatch):
    block, x, extra = _make(name, dtype, qkv_bias=bias)
    x = torch.cat([x, x], dim=-1)[..., :x.shape[-1]]  # rows of twice their length
    g = torch.randn(x.shape[0], 1, x.shape[2], device="cuda").to(dtype).expand(x.shape)
    results = []
    for whole in (True, False):
        leaf = x.detach().requires_grad_()
        block.zero_grad(set_to_none=True)
        out = block(leaf, *extra) if whole else _steps(block, monkeypatch, lambda b: b(leaf, *extra))
        out.backward(g)
        results.append([out.detach(), leaf.grad] + [p.grad for p in block.parameters()])
    assert len(counted) == 1
    u = UNIT_ROUNDOFF[dtype]
    for a, b, e in zip(*results, _exact(block, x, extra, g)):
        assert a.dtype == dtype and a.shape == b.shape
        assert _distance(a, e) <= 1.25 * _distance(b, e) + 1.3 * u + 2.0 ** -20, (_distance(a, e), _distance(b, e))
    with torch.no_grad():
        _close(block(x, *extra), results[0][0], dtype)
    assert len(counted) == 2


@pytest.mark.parametrize("name", sorted(BLOCKS))
def test_frozen_parameters(name, counted, monkeypatch):
    """Every parameter (and the input) alone: the gradients that are asked for, and no others."""
    block, x, extra = _make(name, torch.half)
    named = dict(block.named_parameters())
    for wanted in (None, *named):
        for n, p in named.items():
            p.requires_grad_(n == wanted)
        leaf = x.clone().requires_grad_(wanted is None)
        grads = []
        for whole in (True, False):
            out = block(leaf, *extra) if whole else _steps(block, monkeypatch, lambda b: b(leaf, *extra))
            grads.append(torch.autograd.grad(out, [leaf if wanted is None else named[wanted]], torch.ones_like(out))[0])
        _close(*grads, torch.half)
    assert len(counted) == 1 + len(named)


@pytest.mark.parametrize("name", ["mlla", "pola", "focused", "linfusion"])
def test_gradients_that_the_kernels_cannot_read_come_from_the_steps(name, counted, monkeypatch):
    block, x, extra = _make(name, torch.half if name == "linfusion" else torch.float)
    dtype = x.dtype
    x.requires_grad_()
    wanted = [p for n, p in block.named_parameters() if n.startswith(("proj", "dwc", "lepe", "to_out"))]
    results = []
    for whole in (True, False):
        call = lambda b: b(x, *extra)  # noqa: E731
        y = call(block) if whole else _steps(block, monkeypatch, call)
        gen = torch.Generator(device="cuda").manual_seed(1)
        g = torch.randn(2, *y.shape, device="cuda", generator=gen).to(dtype)
        batched = torch.autograd.grad(y, wanted, g, is_grads_batched=True, retain_graph=True)
        mapped = torch.func.vmap(lambda g: torch.autograd.grad(y, wanted, g, retain_graph=True))(g)
        one_by_one = zip(*(torch.autograd.grad(y, wanted, e, retain_graph=True) for e in g))
        for a, b, c in zip(batched, mapped, one_by_one):
            _close(a, torch.stack(c), dtype)
            _close(b, torch.stack(c), dtype)
        once = torch.autograd.grad(y, wanted, g[0], create_graph=True)
        twice = torch.autograd.grad(sum(t.float().square().sum() for t in once), x, allow_unused=True)
        results.append([*batched, *(t.detach() for t in once), *(t for t in twice if t is not None)])
    assert len(counted) == 1 and len(results[0]) == len(results[1])
    for a, b in zip(*results):
        _close(a, b, dtype)


@pytest.mark.parametrize("name", sorted(BLOCKS))
def test_calls_that_something_looks_into_run_step_by_step(name, counted):
    block, x, extra = _make(name, torch.half)
    plain = block(x, *extra)
    assert len(counted) == 1
    for module in block.modules():
        if module is block or type(module).__name__ in ("Dropout", "ModuleList") or module in (getattr(block, n, None) for n in ("sr", "norm", "elu")):
            continue
        handle = module.register_forward_hook(lambda *a: None)
        if type(module).__name__ != "Dropout":
            _close(block(x, *extra), plain, torch.half)
        handle.remove()
    if name in ("mlla", "linfusion"):  # (the others' features come out of autocast in fp32, the values in fp16: refused)
        with torch.autocast("cuda", dtype=torch.half):
            block(x, *extra)

    class Other(type(block)):
        pass
    block.__class__ = Other
    block(x, *extra)
    assert len(counted) == 1


def test_two_streams():
    """A call on a stream of its own, its tensors freed while it may still run."""
    block, x, extra = _make("pola", torch.half)
    want = block(x, *extra).detach()
    side = torch.cuda.Stream()
    for _ in range(3):
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = block(x.clone().requires_grad_(), *extra)
            y.backward(torch.ones_like(y))
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(y.detach(), want)
        block.zero_grad()


def test_negative_slope(counted):
    """torch takes it, and so does the block: step by step, with the gradients of torch's operators."""
    block, x, _ = _make("linfusion", torch.half)
    for path in (block.to_q_, block.to_k_):
        path[2] = torch.nn.LeakyReLU(-0.5)  # (in place torch refuses the backward)
    leaf, g = x.requires_grad_(), torch.randn_like(x)
    out = block(leaf)
    out.backward(g)
    got = [out.detach(), leaf.grad] + [p.grad for p in block.parameters()]
    assert not counted
    for a, e in zip(got, _exact(block, x, (), g)):  # (a value whose rounding crosses the kink: 1.5 of its gradient, as in _make)
        assert _distance(a, e) <= 0.1


@pytest.mark.parametrize("name", ["mlla", "pola", "focused", "linfusion"])
def test_function_modes_see_the_steps(name, counted):
    block, x, extra = _make(name, torch.half)
    seen = []

    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    with torch.device("cuda"):  # (a default device looks at no operator)
        plain = block(x, *extra)
        assert len(counted) == 1
        with Watch():
            _close(block(x, *extra), plain, torch.half)
    assert len(counted) == 1 and torch.nn.functional.linear in seen


@pytest.mark.parametrize("what", ["outputs", "rows"])
def test_projections_past_the_kernels_limits_run_on_the_library(what, counted, monkeypatch):
    """More outputs than the projections' kernel addresses, rows further apart: the library's GEMM takes them as it always did."""
    block, x, extra = _make("focused" if what == "outputs" else "linfusion", torch.half)
    if what == "outputs":
        block.proj = torch.nn.Linear(64, 65544).cuda().half()
    else:
        row = (1 << 22) + 8
        x = torch.empty(3 * 40 * row, device="cuda", dtype=torch.half).as_strided((3, 40, 128), (40 * row, row, 1)).copy_(x)
    got = []
    for whole in (True, False):
        leaf = x.detach().requires_grad_()
        out = block(leaf, *extra) if whole else _steps(block, monkeypatch, lambda b: b(leaf, *extra))
        got.append([out.detach(), *torch.autograd.grad(out, [leaf, *block.parameters()], torch.ones_like(out))])
    assert len(counted) == 1
    for a, b in zip(*got):
        _close(a, b, torch.half)


@pytest.mark.parametrize("name", ["mlla", "pola", "focused", "linfusion"])  # (torch's own LayerNorm reads strided statistics wrongly)
def test_saved_tensors_that_come_back_elsewhere(name, counted):
    """Saved-tensor hooks may return other strides and addresses that are no multiple of 16 bytes."""
    def unpack(t):
        if t.ndim > 1:
            return torch.cat([t, t + 1], dim=-1)[..., :t.shape[-1]]
        return torch.cat([t[:1], t])[1:]
    block, x, extra = _make(name, torch.half)
    grads = []
    for hooks in (False, True):
        leaf = x.detach().requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack if hooks else lambda t: t):
            out = block(leaf, *extra)
        grads.append(torch.autograd.grad(out, [leaf, *block.parameters()], torch.ones_like(out)))
    assert len(counted) == 2
    for a, b in zip(*grads):
        _close(a, b, torch.half)


@pytest.mark.parametrize("dtype", [torch.half, torch.float])
@pytest.mark.parametrize("make,side", [
    (lambda: MambaLikeLinearAttention(128, (28, 28), 2), ()), (lambda: MambaLikeLinearAttention(128, (28, 28), 4), ()),
    (lambda: PolaLinearAttention(128, 784, num_heads=2), (28, 28)), (lambda: PolaLinearAttention(128, 784, num_heads=4), (28, 28)),
    (lambda: PolaLinearAttention(128, 784, num_heads=2, sr_ratio=2), (28, 28)),
    (lambda: FocusedLinearAttention(128, 784, num_heads=2), (28, 28)),
    (lambda: FocusedLinearAttention(128, 784, num_heads=2, sr_ratio=2), (28, 28)),
    (lambda: GeneralizedLinearAttention(128, heads=2, dim_head=64), ())])
def test_inference_holds_no_more_memory_than_the_steps(make, side, dtype, monkeypatch):
    """Rows of 64 MB and more: what nothing reads any more is given up on the way."""
    torch.manual_seed(0)
    block = make().cuda().to(dtype)
    if hasattr(block, "rope"):
        block.rope.float()
    x = torch.randn(336, 784, 128, device="cuda").to(dtype)

    def peak(block):
        with torch.no_grad():
            block(x, *side)
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            block(x, *side)
        return torch.cuda.max_memory_allocated() - before
    assert peak(block) <= _steps(block, monkeypatch, peak) + (1 << 20)
