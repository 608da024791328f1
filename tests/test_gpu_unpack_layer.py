"""The whole-layer dequantizers (``rdkv_unpack_layer_k`` / ``rdkv_unpack_layer_v``) at the edges of
their tiles and of their fast paths, bit for bit against the oracle's unpackers: token counts around
the 64-row tile, head dimensions that are no multiple of the 8-channel and 32-channel forms or need
several channel chunks, segments that are views of wider tensors, a head without tokens or channels."""
import dataclasses

import numpy as np
import pytest
import torch

from oracle import rdkv_oracle as O
from rdkv_amd import packing, trizone_decompress as tz
from tests.gpu_util import DEV, assert_bits_equal, layer_to_device, require_gpu, t2n, to_dev

pytestmark = pytest.mark.gpu


def _widened(t, dim):
    """The same values as a view into a larger tensor (row stride no longer the row length)."""
    if t is None:
        return None
    shape = list(t.shape)
    shape[dim] += 3
    wide = torch.full(shape, 0xAB, dtype=t.dtype, device=t.device)
    view = wide.narrow(dim, 0, t.shape[dim])
    view.copy_(t)
    return view


@pytest.mark.parametrize("D,T,H", [(128, 1, 1), (128, 63, 2), (128, 64, 3), (128, 65, 2), (128, 1500, 8),
                                   (8, 70, 2), (36, 130, 2), (64, 129, 3), (256, 200, 2), (264, 67, 2)])
def test_whole_layer_dequantizers_against_the_oracle(D, T, H):
    require_gpu()
    rng = np.random.default_rng(1000 * D + T)
    K = rng.standard_normal((1, H, T, D)).astype(np.float16)
    V = rng.standard_normal((1, H, T, D)).astype(np.float16)
    vb = rng.choice(np.array([0, 2, 4, 8, 16]), size=(H, T))
    vb[0, 0] = 4
    kb = rng.choice(np.array([0, 2, 4, 8]), size=(H, D))
    kb[0, :4] = (2, 4, 8, 8)
    if H > 1:
        vb[-1] = 0                       # a head that keeps nothing, with channels all the same
    ora, ora_nvo = O.pack_layer_per_head(K, V, vb, kb, 2)
    pl = layer_to_device(ora)
    exp_k, exp_v = O.unpack_k_mixed(ora, D), O._unpack_v_perhead(ora, head_dim=D)
    strided = dataclasses.replace(pl, **{n: _widened(getattr(pl, n), 3) for n in ("K_2bit", "K_4bit", "K_8bit")},
                                  **{n: _widened(getattr(pl, n), 2) for n in ("V_2bit", "V_4bit", "V_8bit")})
    for layer in (pl, strided):
        assert_bits_equal(t2n(packing.unpack_k_mixed(layer, D=D)), exp_k)
        assert_bits_equal(t2n(tz._unpack_v_perhead(layer, head_dim=D)), exp_v)
        nvo = to_dev(ora_nvo) if ora_nvo is not None else None
        cache = packing.TriZoneCache((layer,), [nvo], [None], [None], T)
        (k, v), = tz.unpack_trizone_to_past_kv(cache, head_dim=D)
        assert_bits_equal(t2n(k), exp_k)
        assert_bits_equal(t2n(v), exp_v if ora_nvo is None else np.concatenate([exp_v, ora_nvo], axis=2))


@pytest.mark.parametrize("D,widths", [(1, (8,)), (3, (8,)), (6, (4, 8)), (6, (8,)), (130, (4, 8)), (131, (8,))])
def test_head_dimensions_that_only_some_widths_pack(D, widths):
    """A class needs whole bytes per row, a class that is not there needs nothing."""
    require_gpu()
    rng = np.random.default_rng(D)
    H, n = 2, 37
    code = {b: rng.integers(0, 1 << b, (1, H, n, D)) for b in widths}
    seg = {8: lambda c: c, 4: lambda c: c[..., :D // 2] | c[..., D // 2:] << 4}
    T = n * len(widths)
    scale = rng.uniform(0.1, 2.0, (1, H, T, 1)).astype(np.float16)
    zp = rng.integers(0, 8, (1, H, T, 1)).astype(np.float16)
    v16 = rng.standard_normal((1, H, 5, D)).astype(np.float16)
    counts = np.array([[0, n if 4 in widths else 0, n]] * H, np.int32)
    none = dict.fromkeys(f.name for f in dataclasses.fields(packing.PackedKVLayer))
    pl = packing.PackedKVLayer(**{**none, **{f"V_{b}bit": to_dev(seg[b](code[b]).astype(np.uint8)) for b in widths},
                                  "V_scale": to_dev(scale), "V_zp": to_dev(zp), "T_eff": T,
                                  "seg_bounds_per_head": to_dev(counts), "T_eff_per_head": to_dev(counts.sum(1).astype(np.int32))})
    codes = np.concatenate([code[b] for b in widths], axis=2).astype(np.float32)
    exp = ((codes - zp.astype(np.float32)) * scale.astype(np.float32)).astype(np.float16)
    assert_bits_equal(t2n(tz._unpack_v_perhead(pl, head_dim=D)), exp)
    assert_bits_equal(t2n(tz._unpack_v_enqueue(pl, to_dev(v16), D)[0]), np.concatenate([exp, v16], axis=2))


def test_zero_points_that_are_not_whole_numbers():
    """Layers of other origin may carry such zero points; they take the fp32 form."""
    require_gpu()
    rng = np.random.default_rng(9)
    K, V = (rng.standard_normal((1, 2, 90, 128)).astype(np.float16) for _ in range(2))
    vb, kb = rng.choice(np.array([2, 4, 8]), size=(2, 90)), rng.choice(np.array([2, 4, 8]), size=(2, 128))
    ora, _ = O.pack_layer_per_head(K, V, vb, kb, 2)
    ora.K_ch_zp[:, 1, :, 5] += np.float16(0.3)
    ora.V_zp[:, 0, 3] += np.float16(0.7)
    ora.V_zp[:, 1, 60:] = np.float16(3000.5)
    pl = layer_to_device(ora)
    assert_bits_equal(t2n(packing.unpack_k_mixed(pl, D=128)), O.unpack_k_mixed(ora, 128))
    assert_bits_equal(t2n(tz._unpack_v_perhead(pl, head_dim=128)), O._unpack_v_perhead(ora, head_dim=128))


def test_counts_that_do_not_fit_the_layer_are_reported():
    require_gpu()
    rng = np.random.default_rng(3)
    K, V = (torch.from_numpy(rng.standard_normal((1, 2, 100, 128)).astype(np.float16)).to(DEV) for _ in range(2))
    vb = torch.from_numpy(rng.choice(np.array([2, 4, 8]), size=(2, 100)))
    kb = torch.from_numpy(rng.choice(np.array([2, 4]), size=(2, 128)))
    pl, nvo = packing.pack_layer_per_head(K, V, vb, kb, 2)
    pl.seg_bounds_per_head = pl.seg_bounds_per_head + 1          # within the rows the kernel clamps to
    cache = packing.TriZoneCache((pl,), [nvo], [None], [None], 100)
    with pytest.raises(AssertionError, match="T_eff_per_head"):
        tz.unpack_trizone_to_past_kv(cache, head_dim=128)
    pl.K_ch_seg_bounds_per_head = pl.K_ch_seg_bounds_per_head + 1          # 8-bit channels, no 8-bit segment
    with pytest.raises(AssertionError, match="segment that is missing"):
        packing.unpack_k_mixed(pl, D=128)
    pl, nvo = packing.pack_layer_per_head(K, V, vb, kb, 2)
    counts = pl.seg_bounds_per_head.clone()
    counts[:, 0] += 100                                          # more 2-bit tokens than the segment has, sums alike
    pl.seg_bounds_per_head, pl.T_eff_per_head = counts, pl.T_eff_per_head + 100
    with pytest.raises(AssertionError, match="V segments"):
        tz._unpack_v_perhead(pl, head_dim=128)
    counts = pl.K_ch_seg_bounds_per_head.clone()
    counts[:, 0] += 200                                          # more 2-bit channels than the segment has
    pl.K_ch_seg_bounds_per_head = counts
    with pytest.raises(AssertionError, match="K segments of"):
        packing.unpack_k_mixed(pl, D=128)


@pytest.mark.parametrize("D", [128, 200])
@pytest.mark.parametrize("channel", [-1, None, 1 << 40])
def test_channels_outside_the_head_are_reported(D, channel):
    """The kernel leaves such a channel out and says so; padding behind the kept channels is not looked at."""
    require_gpu()
    rng = np.random.default_rng(D)
    K, V = (torch.from_numpy(rng.standard_normal((1, 3, 40, D)).astype(np.float16)).to(DEV) for _ in range(2))
    vb, kb = torch.from_numpy(rng.choice(np.array([2, 4, 8]), size=(3, 40))), torch.full((3, D), 4)
    kb[1, :50] = 0
    pl, _ = packing.pack_layer_per_head(K, V, vb, kb, 2)
    exp, index = packing.unpack_k_mixed(pl, D=D), pl.K_ch_sort_idx_per_head
    pl.K_ch_sort_idx_per_head = index.clone()
    pl.K_ch_sort_idx_per_head[1, D - 50:] = D if channel is None else channel
    assert torch.equal(packing.unpack_k_mixed(pl, D=D), exp)
    pl.K_ch_sort_idx_per_head[1, D - 51] = D if channel is None else channel
    with pytest.raises(IndexError, match="1"):
        packing.unpack_k_mixed(pl, D=D)


def _random_k_layer(H, T, D, n_k, counts, seed, strided):
    """A per-head K layer of random codes (no packer: the large sizes are about the launch), head h keeping
    counts[h] channels of the classes, laid out for n_k."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    widths = (-(-n_k[0] // 4) * 4, -(-n_k[1] // 2) * 2, n_k[2])
    segs = [torch.randint(0, 256, (1, H, T, w * b // 8), generator=g, device=DEV).to(torch.uint8) if w else None
            for w, b in zip(widths, (2, 4, 8))]
    Dp, kept = sum(widths), max(map(sum, counts))
    index = torch.stack([torch.randperm(D, generator=g, device=DEV)[:kept] for _ in range(H)])
    scale = torch.rand(1, H, 1, Dp, generator=g, device=DEV).half()
    zp = torch.randint(0, 256, (1, H, 1, Dp), generator=g, device=DEV).half()
    none = dict.fromkeys(f.name for f in dataclasses.fields(packing.PackedKVLayer))
    K = [_widened(s, 3) if strided else s for s in segs]
    layer = packing.PackedKVLayer(**{**none, "K_2bit": K[0], "K_4bit": K[1], "K_8bit": K[2], "K_ch_scale": scale, "K_ch_zp": zp,
                                     "K_ch_seg_bounds": n_k, "K_ch_sort_idx_per_head": index, "T_eff": T, "T_eff_k": T,
                                     "K_ch_seg_bounds_per_head": torch.tensor(counts, dtype=torch.int32, device=DEV)})
    exp = torch.zeros(1, H, T, D, dtype=torch.float16, device=DEV)
    for h in range(H):
        at = slot = 0
        for s, w, b, n in zip(segs, widths, (2, 4, 8), counts[h]):
            if n:
                rows = packing._dequant(s[0, h], w, b, scale[0, h, 0, slot:slot + w], zp[0, h, 0, slot:slot + w], per_row=False)
                exp[0, h].index_copy_(1, index[h, at:at + n], rows[:, :n])
            at, slot = at + n, slot + w
    return layer, exp


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("H,T,D", [(8, 17001, 128), (1, 131137, 128), (3, 43713, 128), (4, 17000, 200)])
def test_workgroups_that_walk_several_tiles(H, T, D, strided):
    """More rows than one tile per workgroup of the launch (64 x 2048 over all heads and channel chunks):
    LDS filled again behind a barrier, another misalignment per tile, a short last tile."""
    require_gpu()
    counts = [[(5 * h) % 14, (7 * h + 3) % 23, (11 * h + 2) % 20] for h in range(H)]
    counts[-1] = [13, 22, 19]
    layer, exp = _random_k_layer(H, T, D, (13, 22, 19), counts, T, strided)
    assert torch.equal(packing.unpack_k_mixed(layer, D=D).view(torch.int16), exp.view(torch.int16))


@pytest.mark.parametrize("missing", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2)])
def test_a_class_without_a_tensor_has_no_slots(missing):
    """Its columns of the scales are skipped as long as no head keeps channels of it."""
    require_gpu()
    counts = [[0 if c in missing else n for c, n in enumerate(row)] for row in ((13, 22, 19), (3, 5, 7))]
    layer, exp = _random_k_layer(2, 70, 128, (13, 22, 19), counts, 4, False)
    layer = dataclasses.replace(layer, **{("K_2bit", "K_4bit", "K_8bit")[c]: None for c in missing})
    assert torch.equal(packing.unpack_k_mixed(layer, D=128).view(torch.int16), exp.view(torch.int16))
