"""State and mean key of head dims between the kernels' row lengths, which leave and enter them in wider shapes: edges of the
copies' spans of 1024 elements, one row or column, with and without the mean key.

Bound: products of the inputs are exact (16 bits) or rounded once, and summed in fp32: 2^-18 of the matrix in the 2-norm."""
import pytest
import torch

from flash_bla import _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.half, torch.float])
@pytest.mark.parametrize("DK,DV", [(1, 1), (17, 13), (31, 33), (9, 127), (127, 9), (100, 100), (5, 120), (125, 125)])
def test_state_in_the_callers_shape(DK, DV, dtype):
    torch.manual_seed(DK * 128 + DV)
    q, k = (torch.rand(2, 3, 77, DK, device="cuda").to(dtype) for _ in range(2))
    v, g = (torch.randn(2, 3, 77, DV, device="cuda").to(dtype) for _ in range(2))
    want = k.double().transpose(-1, -2).contiguous() @ v.double() / 77
    mean = k.double().mean(2)
    for flags in (0, _hip.NORMALIZE):
        o, s, km = _hip.la_fwd(q, k, v, None, None, 1.0 / 77, 1e-6, flags)
        assert s.shape == want.shape and (s.double() - want).norm() <= 2.0 ** -18 * want.norm()
        if flags:
            assert (km.double().reshape(mean.shape) - mean).norm() <= 2.0 ** -18 * mean.norm()
        else:  # dq = dO S^T, rounded once; S as hi and lo parts
            dq = _hip.la_bwd(q, k, v, None, None, g, s, None, 1.0 / 77, 1e-6, 0)[0]
            exact = g.double() @ want.transpose(-1, -2).contiguous()
            assert (dq.double() - exact).norm() <= (2.0 ** -11 if dtype == torch.half else 2.0 ** -18) * 1.25 * exact.norm()
