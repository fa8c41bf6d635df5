"""Projections of token rows and the norm between them against float64: token counts and channels around the tiles (64 and 128)
and the step of 64, two products, an added tensor, strided rows, several jobs in a launch, rows past the end that hold NaN.

Bound: products of 16-bit values are exact in fp32, a sum of K of them stays within 2^-24 * sqrt(K) * 4 of the root mean square of
its terms times sqrt(K), and the result is rounded once (u)."""
import pytest
import torch

from helpers import UNIT_ROUNDOFF
from flash_bla import _hip

pytestmark = pytest.mark.gpu
DTYPES = [torch.float16, torch.bfloat16]


def _close(got, want, rms, K, dtype):
    slack = 2.0 ** -24 * 4 * K ** 0.5 * rms * K ** 0.5 + 2.0 ** -24
    assert ((got.double() - want).abs() <= UNIT_ROUNDOFF[dtype] * want.abs() + slack).all(), (got.double() - want).abs().max()


def _rows(tokens, channels, dtype, strided=False):
    """Rows that lie in front of NaN."""
    wide = torch.full((tokens + 1, channels + (24 if strided else 0)), float("nan"), device="cuda", dtype=dtype)
    rows = wide[:tokens, :channels]
    rows.copy_(torch.randn(tokens, channels, device="cuda"))
    return rows


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens,K,N", [(1, 8, 8), (63, 72, 64), (64, 64, 128), (65, 56, 136), (129, 128, 72), (1000, 640, 320),
                                        (128 * 257 + 3, 64, 128), (128 * 260, 256, 264), (128 * 256 + 1, 136, 56)])
def test_projection(tokens, K, N, dtype):
    torch.manual_seed(tokens + K)
    x, g = _rows(tokens, K, dtype, strided=True), _rows(tokens, N, dtype, strided=True)
    x2, g2 = _rows(tokens, K, dtype), _rows(tokens, N, dtype)
    w, w2 = (_rows(N, K, dtype) for _ in range(2))
    b = torch.randn(N, device="cuda").to(dtype)
    cases = [([(x, w, None, None, None, None)], False, [(x, w.t(), None, None)]),
             ([(x, w, b, g2, None, None), (x2, w2, None, None, None, None), (x2, w, b, None, None, None)], False,
              [(x, w.t(), None, g2.double() + b.double()), (x2, w2.t(), None, None), (x2, w.t(), None, b.double())]),
             ([(g, w, None, None, None, None), (g2, w2, None, x, None, None)], True,
              [(g, w, None, None), (g2, w2, None, x.double())]),
             ([(g, w, None, x2, g2, w2)], True, [(g, w, (g2, w2), x2.double())]),
             # a job of one product next to one of two: it has no second rows to look at
             ([(g, w, None, None, g2, w2), (g2, w2, None, x, None, None)], True, [(g, w, (g2, w2), None), (g2, w2, None, x.double())]),
             ([(g2, w2, None, x, None, None), (g, w, None, None, g2, w2)], True, [(g2, w2, None, x.double()), (g, w, (g2, w2), None)])]
    for jobs, rows_of_w, wants in cases:
        for got, (a, m, second, more) in zip(_hip.project(jobs, rows_of_w), wants):
            a, m = a.double(), m.double()
            want, power, terms = a @ m, a.square() @ m.square(), m.shape[0]
            if second is not None:
                a2, m2 = (t.double() for t in second)
                want, power, terms = want + a2 @ m2, power + a2.square() @ m2.square(), 2 * terms
            _close(got, want if more is None else want + more, (power / terms).sqrt(), terms, dtype)
            assert got.is_contiguous() and got.dtype == dtype


@pytest.mark.parametrize("rows_of_w", [False, True])
def test_weight_that_ends_with_its_memory(rows_of_w):
    """A weight and rows that fill an allocation of their own: the loads ahead of the last step are past its end."""
    torch.manual_seed(0)
    K, N, tokens = 1536, 4096, 4096  # 12 MiB each
    a, w = (torch.empty(tokens, K, device="cuda", dtype=torch.half).normal_() for _ in range(2))
    m = w.view(K, N) if rows_of_w else w.view(N, K).t()
    got, = _hip.project([(a, m if rows_of_w else m.t(), None, None, None, None)], rows_of_w)
    a, m = a.double(), m.double()
    _close(got, a @ m, (a.square() @ m.square() / K).sqrt(), K, torch.half)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens,C", [(1, 8), (5, 504), (4, 512), (7, 520), (9, 640), (3, 1280), (33, 2048)])
def test_norm_leaky(tokens, C, dtype):
    """fp32 from exact inputs: mean and variance within 2^-20 of the largest normed value, one rounding."""
    torch.manual_seed(C)
    jobs, wants = [], []
    for affine, eps, slope in ((True, 1e-5, 0.01), (False, 1e-3, 0.2)):
        x = (3 * torch.randn(2, tokens, C, device="cuda") + 1).to(dtype)
        w, b = (torch.randn(C, device="cuda").to(dtype) for _ in range(2)) if affine else (None, None)
        jobs.append((x, w, b, eps, slope))
        y = torch.nn.functional.layer_norm(x.double(), (C,), None if w is None else w.double(), None if b is None else b.double(), eps)
        mean, rstd = x.double().mean(-1, keepdim=True), (x.double().var(-1, unbiased=False, keepdim=True) + eps).rsqrt()
        wants.append((torch.nn.functional.leaky_relu(y, slope), mean, rstd))
    for with_stats in (True, False):
        for (y, mean, rstd), want in zip(_hip.norm_leaky(jobs, with_stats), wants):
            assert ((y.double() - want[0]).abs() <= UNIT_ROUNDOFF[dtype] * want[0].abs() + 2.0 ** -20 * want[0].abs().max()).all()
            assert (mean is None) == (rstd is None) == (not with_stats)
            if with_stats:
                torch.testing.assert_close(mean.double(), want[1], rtol=1e-5, atol=1e-5)
                torch.testing.assert_close(rstd.double(), want[2], rtol=1e-5, atol=1e-5)


def test_refusals():
    x, w = torch.zeros(4, 16, device="cuda"), torch.zeros(8, 16, device="cuda")
    with pytest.raises(ValueError):
        _hip.project([(x, w, None, None, None, None)], False)  # fp32
    x, w = x.half(), w.half()
    with pytest.raises(RuntimeError):
        _hip.project([(x, w[:, :8], None, None, None, None)], False)  # another number of channels
    with pytest.raises(ValueError):
        _hip.project([(x[:, :12], w[:, :12], None, None, None, None)], False)  # no whole pieces
    with pytest.raises(ValueError):
        _hip.norm_leaky([(torch.zeros(2, 2056, device="cuda").half(), None, None, 1e-5, 0.01)], False)
    assert [tuple(t.shape) for t in _hip.project([(x[:0], w, None, None, None, None)], False)] == [(0, 8)]
