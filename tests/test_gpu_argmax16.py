"""The argmax of 16-bit logits by integer order: zeros of both signs, NaNs of both signs, infinities, all negative rows,
ties across lanes, pieces, rounds and the ragged end."""
import pytest
import torch

from rdkv_amd import fast_decode
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu


def _rows(n, dtype):
    g = torch.Generator().manual_seed(n)
    x = (torch.randn(n, generator=g) * 3).to(dtype)
    nan = float("nan")
    signed_nan = torch.tensor([-1], dtype=torch.int16).view(dtype)          # all bits set: a negative NaN
    yield x
    yield -x.abs() - 1
    for value in (0.0, -0.0, float("inf"), 50.0, nan):
        for places in ((n - 1,), (0, n - 1), (n // 2, n - 1), (min(n - 1, 8199), n - 1)):
            y = -x.abs() - 1
            y[list(places)] = value
            yield y
    y = -x.abs() - 1
    y[n // 3] = -0.0                        # equal to the +0 behind it
    y[n // 2] = 0.0
    yield y
    y = x.clone()
    y[n // 2] = signed_nan[0]
    yield y
    yield torch.full((n,), -float("inf"), dtype=dtype)
    yield torch.full((n,), torch.finfo(dtype).min, dtype=dtype)
    yield torch.zeros(n, dtype=dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 1023, 8191, 8193, 131072, 131081, 151936])
def test_argmax_of_16_bit_logits(n, dtype):
    require_gpu()
    token = torch.zeros(1, 1, dtype=torch.long, device=DEV)
    for i, row in enumerate(_rows(n, dtype)):
        fast_decode._argmax_advance(row.to(DEV), token)
        assert int(token) == int(row.float().argmax()), i
