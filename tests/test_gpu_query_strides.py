"""Queries of any row stride with the rotary embedding inside the launch: the result of the same rows side by side, bit for
bit (the partner channel of a pair is 64 away within the row, wherever the row starts)."""
import pytest
import torch

from rdkv_amd import stream_cache
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [3, 8])
@pytest.mark.parametrize("width,first", [(128, 0), (192, 0), (200, 40), (129, 1), (320, 64)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rotated_queries_of_any_row_stride(G, width, first, dtype):
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(G + width)
    K, V = (torch.randn(1, 2, 150, 128, generator=g, device=DEV).half() for _ in range(2))
    cache = stream_cache.build_stream_cache_from_kv([(K, V, torch.full((2, 150), 4, device=DEV), torch.full((2, 128), 4, device=DEV))], G)
    wide = torch.randn(cache.rows + 2, width, generator=g, device=DEV).to(dtype)       # (a row ahead and one behind)
    q = wide.reshape(-1)[width:][:cache.rows * width].view(cache.rows, width)[:, first:first + 128]
    ang = torch.rand(64, generator=g, device=DEV)
    rope = (ang.cos(), ang.sin())
    zone_c = tuple(torch.randn(2, 5, 128, generator=g, device=DEV) for _ in range(2))
    for kw in ({}, {"zone_c": zone_c}):
        got = stream_cache.decode_attn_fused(cache, q, rope=rope, **kw)
        exp = stream_cache.decode_attn_fused(cache, q.contiguous(), rope=rope, **kw)
        assert torch.equal(got[0], exp[0]) and torch.equal(got[1], exp[1]) and bool(torch.isfinite(got[0]).all())
