"""Problems of few heads, whose token chunks are cut finer than elsewhere: lengths at the edges of the chunks, forward and
backward against the float64 oracle."""
import pytest
import torch

from flash_bla import _hip
from test_gpu_cross_lengths import _check
from test_zz_no_alloc import _call_static

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,dims", [((1, 1), (64, 64)), ((2, 4), (64, 64)), ((1, 2), (128, 128)), ((1, 3), (32, 32)),
                                        ((1, 2), (100, 100)), ((2, 2), (128, 64))])
def test_few_heads(heads, dims, dtype):
    for i, length in enumerate((256, 257, 320, 513, 1024, 1087, 2050)):
        _check("linear", *heads, length, length, *dims, dtype, 31 * i + dims[1])
    _check("simple", *heads, 769, 769, *dims, dtype, 7)


def test_few_heads_that_fit_the_built_in_scratch_with_longer_chunks_only():
    """The same bits with it as with a workspace, and the oracle's values."""
    B, H, L, DK, DV = 3, 3, 1750, 110, 87
    q, k = (torch.rand(B, H, L, DK, device="cuda").half() for _ in range(2))
    v = torch.randn(B, H, L, DV, device="cuda").half()
    rc, *static = _call_static(_hip, q, k, v, 1.0 / L, 1e-6, _hip.NORMALIZE)
    assert rc == 0, _hip.lib().fbla_last_error()
    assert all(torch.equal(a, b) for a, b in zip(static, _hip.la_fwd(q, k, v, None, None, 1.0 / L, 1e-6, _hip.NORMALIZE)))
    _check("linear", B, H, L, L, DK, DV, torch.half, 3)
