"""One-row projections: rows dealt round-robin over the launch's wavefronts.  Sizes where the dealing
can go wrong: fewer rows than a workgroup has wavefronts, one more than a round, around the change from
sixteen to eight wavefronts per compute unit, rows long enough for the wider workgroup, row ends inside
a tile; plain, fp32, normed and SiLU inputs, both types, weights that are a view."""
import pytest
import torch

from rdkv_amd import fast_decode
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,dtype", [
    (1, 512, torch.float16), (3, 4608, torch.bfloat16), (5, 16384, torch.float16), (4095, 512, torch.float16),
    (4097, 1024, torch.bfloat16), (8192, 2560, torch.float16), (8193, 2048, torch.float16), (16387, 512, torch.bfloat16),
    (517, 8192, torch.float16), (517, 8704, torch.bfloat16), (40, 32768, torch.float16)])
def test_rows_dealt_over_wavefronts(N, K, dtype):
    require_gpu()
    g = torch.Generator().manual_seed(N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    W = rnd(N, K + 8)[:, :K] if N < 600 else rnd(N, K)
    x, delta, norm, gate, bias = rnd(1, K), rnd(1, K), rnd(K), rnd(1, K), rnd(N)
    eps = torch.finfo(dtype).eps
    W64 = W.double().cpu()

    def check(y, row, b=0.0):
        """One rounding of the result, and independent roundings of the row's elements (eps / 2 at most, 0.2 eps
        rms) that add up to 0.2 eps sqrt(K) in units of the mean product's 1 / 0.64: twelve times that."""
        row, y = row.double().cpu().reshape(-1), y.double().cpu().reshape(-1)
        exp = W64 @ row + b
        bound = eps * exp.abs() + 4 * eps * (W64.abs() @ row.abs()) / K ** 0.5
        assert bool(((y - exp).abs() <= bound + 1e-6).all())

    check(fast_decode._linear_row(x, W, bias), x, bias.double().cpu())
    check(fast_decode._linear_row(x.float(), W), x)
    act = torch.nn.functional.silu(gate.float()).to(dtype).float() * x.float()
    check(fast_decode._silu_linear_row(gate, x, W), act.to(dtype))
    if K <= 8192:
        r = (x.float() + delta.float()).to(dtype)
        h = r.double() * torch.rsqrt(r.double().pow(2).mean() + 1e-5) * norm.double()
        y, res = fast_decode._norm_linear_row(x, delta, norm, 1e-5, W, None)
        assert torch.equal(res, r)
        check(y, h)
