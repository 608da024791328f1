"""A layer's rows, tables and mask in one launch, bit for bit against the launches of the general path: token counts
around the 64-row and 128-row workgroups, heads that keep nothing or no channel, padded and full channel segments, every
integer type of the channel widths, K and V as views."""
import pytest
import torch

from rdkv_amd import _lib, packing
from tests.gpu_util import DEV, NativeCalls, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,G,widths,dtype", [(1, 1, 1, (2, 4, 8), torch.uint8), (64, 2, 4, (0, 2, 4, 8, 16), torch.int64),
                                                (127, 3, 5, (2,), torch.int16), (129, 2, 2, (4,), torch.int32),
                                                (400, 8, 4, (8, 16), torch.uint8), (1300, 5, 1, (0, 0, 2, 8), torch.int64),
                                                (5000, 2, 8, (0, 2, 4, 8), torch.int16)])
def test_one_launch_equals_the_general_path(T, H, G, widths, dtype, monkeypatch):
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(T + H)
    wide = torch.randn(1, H, T + 3, 256, device=DEV, dtype=torch.float16, generator=g)
    K, V = wide[:, :, 3:, :128], wide[:, :, 3:, 128:]
    token = torch.tensor([0, 2, 4, 8, 16], device=DEV)
    vb = token[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
    vb[:, 0] = 4
    kb = torch.tensor(widths, device=DEV)[torch.randint(0, len(widths), (H, 128), device=DEV, generator=g)]
    kb[0, 5] = max(widths)
    if H > 2:
        vb[-1], kb[-2] = 0, 0                # a head without tokens, one without channels
    kb = torch.cat([kb, kb], dim=1).to(dtype)[:, :128]
    results, calls = [], NativeCalls(_lib.native)
    for native, early in ((calls, 1), (None, 1 << 30)):
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", native)
            m.setattr(packing, "_EARLY_MINMAX_TOKENS", early)
            results.append(packing.pack_layer_per_head(K, V, vb, kb, G))
    assert calls.taken == ["pack_layer"]
    (a, a16), (b, b16) = results
    assert (a16 is None) == (b16 is None) and (a16 is None or torch.equal(a16, b16))
    for name in a.__dataclass_fields__:
        x, y = getattr(a, name), getattr(b, name)
        if isinstance(x, torch.Tensor):
            assert x.dtype == y.dtype and torch.equal(x, y), name
        else:
            assert x == y, name
