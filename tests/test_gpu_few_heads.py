"""Problems of few heads, whose token chunks are cut finer than elsewhere: lengths at the edges of the chunks, forward and
backward against the float64 oracle."""
import pytest
import torch

from test_gpu_cross_lengths import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,dims", [((1, 1), (64, 64)), ((2, 4), (64, 64)), ((1, 2), (128, 128)), ((1, 3), (32, 32)),
                                        ((1, 2), (100, 100)), ((2, 2), (128, 64))])
def test_few_heads(heads, dims, dtype):
    for i, length in enumerate((256, 257, 320, 513, 1024, 1087, 2050)):
        _check("linear", *heads, length, length, *dims, dtype, 31 * i + dims[1])
    _check("simple", *heads, 769, 769, *dims, dtype, 7)
