"""Units planned by the packer's first launch against the host's, through the blobs they lay out: more heads than the
launch has threads, channel splits whose stragglers move into wider slots, rows stored as 8 bit, heads without tokens."""
import pytest
import torch

from rdkv_amd import _lib, stream_cache
from tests.gpu_util import DEV, record_native, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T,layers", [(1, 65, 1), (300, 70, 1), (24, 200, 9), (8, 5000, 8), (64, 700, 1), (65, 700, 1)])
def test_blobs_equal_the_general_path(H, T, layers, monkeypatch):
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(H)
    splits = [(2, 1, 125), (0, 11, 5), (17, 9, 3), (128, 0, 0), (0, 0, 1), (15, 7, 3), (31, 0, 2), (1, 120, 7)]
    entries = []
    for l in range(layers):
        K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
        vb = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
        if H > 1:
            vb[1] = 0
        kb = torch.zeros(H, 128, dtype=torch.int64)
        for h in range(H):
            kb[h, torch.randperm(128)[:sum(splits[(h + l) % 8])]] = torch.tensor([2, 4, 8]).repeat_interleave(
                torch.tensor(splits[(h + l) % 8]))
        entries.append((K, V, vb, kb.to(DEV)))
    monkeypatch.setattr(stream_cache, "_POISON_BLOBS", True)
    calls = record_native(monkeypatch)
    got = stream_cache.build_stream_cache_from_kv(entries, 2)
    assert "stream_pack" in calls.taken
    monkeypatch.setattr(_lib, "native", None)                            # (the general path)
    exp = stream_cache.build_stream_cache_from_kv(entries, 2)
    assert all(torch.equal(a, b) for a, b in zip(got.blobs, exp.blobs))
    assert (got.unit_scale_max == exp.unit_scale_max).all()
    q = torch.randn(got.rows, 128, device=DEV, dtype=torch.float16, generator=g)
    for a, b in zip(stream_cache.decode_attn_fused(got, q), stream_cache.decode_attn_fused(exp, q)):
        assert torch.equal(a, b)
