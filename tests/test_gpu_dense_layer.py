"""A packed layer with its padding mask in one launch, bit for bit against the launches of the general path: token
counts around the 64-row tile and past one walk of the workgroups, K rows that begin off a 16-byte address (odd row
widths over several heads), zero points that are no whole numbers, mask rows with and without zeros behind them."""
import pytest
import torch

from rdkv_amd import _lib, packing, trizone_decompress as tz
from tests.gpu_util import DEV, NativeCalls, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,D,extra", [(1, 1, 128, 0), (63, 2, 64, 1), (64, 3, 128, 7), (130, 2, 256, 0), (700, 5, 128, 33),
                                         (40000, 8, 128, 0), (9000, 96, 128, 5)])
@pytest.mark.parametrize("whole", [True, False])
def test_one_launch_equals_the_general_path(T, H, D, extra, whole, monkeypatch):
    require_gpu()
    if not whole and T > 1000:
        pytest.skip("the fractional zero points need no long layer")
    g = torch.Generator(device=DEV).manual_seed(T + H)
    K, V = (torch.randn(1, H, T, D, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    widths = torch.tensor([0, 2, 4, 8, 16], device=DEV)
    vb = widths[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
    vb[:, 0] = 4
    kb = widths[torch.randint(0, 4, (H, D), device=DEV, generator=g)]
    kb[:, 0], kb[:, 1] = 8, 2
    pl, v16 = packing.pack_layer_per_head(K, V, vb, kb, 4)
    if not whole:
        pl.K_ch_zp = pl.K_ch_zp + 0.25
        pl.V_zp = pl.V_zp - 0.5
    assert pl.softmax_mask is not None and pl.softmax_mask.dtype == torch.float32
    pl.softmax_mask[0, 0] = -1e30
    cache = packing.TriZoneCache((pl,), [v16], [None], [None], T)
    results, calls = [], NativeCalls(_lib.native)
    for native in (calls, None):
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", native)
            ((k, v),), (mask,) = tz.unpack_trizone_to_past_kv(cache, head_dim=D, return_masks=True, H_q=4 * H, max_new_tokens=extra)
            results.append((k, v, mask))
    assert calls.taken == ["dense_layer"]
    for a, b in zip(*results):
        assert a.shape == b.shape and a.dtype == b.dtype == torch.float16
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
