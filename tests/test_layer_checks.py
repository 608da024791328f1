"""What the attention and dequantize entry points refuse before they launch anything, without a device:
the library is a recorder, host tensors play the device's and ``meta`` tensors those of another one.
The kernels take addresses, so a shape or device that slips through is a read or write out of range."""
import ctypes
import dataclasses

import pytest
import torch

from rdkv_amd import _lib, fast_decode, packing, trizone_decompress as tz


class _Recorder:
    """Stands for the library: every entry point succeeds and is noted down."""

    def rdkv_unpack_layer_k_checked(self, *args):
        """Writes what the launch reports: the counts, and whether a kept channel is outside the head."""
        self.calls.append("rdkv_unpack_layer_k_checked")
        sort, stride, counts, H, D, check = (args[i] for i in (12, 13, 15, 22, 24, 26))
        counts, check = (ctypes.c_int32 * (3 * H)).from_address(counts), (ctypes.c_int32 * (4 * H)).from_address(check)
        for h in range(H):
            n = counts[3 * h:3 * h + 3]
            kept = (ctypes.c_int64 * max(sum(n), 0)).from_address(sort + 8 * stride * h)
            check[4 * h:4 * h + 4] = n + [int(any(c < 0 or c >= D for c in kept))]
        return 0

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return 0
        return call


def _one_device(*tensors):
    devices = {t.device.type for t in tensors if t is not None}
    if devices != {"cpu"}:
        raise RuntimeError(f"tensors on different devices: {devices}")
    return torch.device("cpu")


@pytest.fixture
def lib(monkeypatch):
    recorder = _Recorder()
    monkeypatch.setattr(_lib, "load", lambda: recorder)
    monkeypatch.setattr(_lib, "available", lambda: True)
    monkeypatch.setattr(_lib, "require_device", _one_device)
    monkeypatch.setattr(_lib, "stream_of", lambda dev: 0)
    monkeypatch.setattr(_lib, "workspace", lambda dev, n: torch.empty(64, dtype=torch.uint8))
    monkeypatch.setattr(_lib, "download", lambda t: t.numpy())
    return recorder


def _layer(H=2, T=6, D=128, G=4, n16=3, n_k=(4, 6, 5), per_head=True):
    """A layer of T packed and n16 fp16 tokens per head, n_k channels per class, as the packers lay it out."""
    def codes(rows, width):
        return torch.zeros(1, H, rows, width, dtype=torch.uint8)

    def full(n):
        return torch.full((H,), n, dtype=torch.int32)

    v = (T - 2 * (T // 3), T // 3, T // 3)
    widths = (packing._seg_padded_len(n_k[0], 4), packing._seg_padded_len(n_k[1], 2), n_k[2])
    rows, kept = T + n16, sum(n_k)
    sort = torch.arange(kept).expand(H, kept).contiguous()
    layer = packing.PackedKVLayer(
        K_2bit=codes(rows, widths[0] // 4), K_4bit=codes(rows, widths[1] // 2), K_8bit=codes(rows, widths[2]),
        K_ch_scale=torch.ones(1, H, 1, sum(widths)).half(), K_ch_zp=torch.zeros(1, H, 1, sum(widths)).half(),
        K_ch_sort_idx=sort[0], K_ch_seg_bounds=n_k, K_ch_perm_padded_idx=torch.zeros(sum(widths), dtype=torch.long),
        V_2bit=codes(v[0], D // 4), V_4bit=codes(v[1], D // 2), V_8bit=codes(v[2], D),
        V_scale=torch.ones(1, H, T, 1).half(), V_zp=torch.zeros(1, H, T, 1).half(),
        sort_idx=torch.zeros(T, dtype=torch.long), seg_bounds=v, T_eff=T, T_eff_k=rows, n_v16=n16)
    if per_head:
        layer = dataclasses.replace(
            layer, seg_bounds_per_head=torch.tensor([v] * H, dtype=torch.int32), T_eff_per_head=full(T),
            K_ch_sort_idx_per_head=sort, K_ch_seg_bounds_per_head=torch.tensor([n_k] * H, dtype=torch.int32),
            T_eff_k_per_head=full(rows), n_v16_per_head=full(n16))
    return layer


def _attend(layer, lib, H_q=8, H_kv=2, n=5, G=4, width=128, **kw):
    kv = torch.zeros(H_kv, n, 128, dtype=torch.float32)
    v16 = torch.zeros(layer.n_v16_per_head.numel(), int(layer.n_v16), 128).half()
    return fast_decode.trizone_attention(torch.zeros(H_q, width), layer, v16, layer.n_v16_per_head, kv, kv, G, **kw)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("rows", [4, 7, 16])
def test_attention_refuses_an_output_of_other_height(lib, packed, rows):
    layer = _layer() if packed else dataclasses.replace(_layer(), T_eff=0, T_eff_k=0)
    with pytest.raises(RuntimeError):
        _attend(layer, lib, out=torch.empty(rows, 128))
    assert not packed or lib.calls == []
    _attend(layer, lib, out=torch.empty(8, 128))
    assert any(name.startswith("rdkv_v_weighted_sum") for name in lib.calls)


@pytest.mark.parametrize("H_q,G,H_kv", [(8, 4, 2), (8, 2, 4), (16, 8, 2), (4, 4, 1)])
def test_attention_refuses_groups_that_do_not_fit_the_layer(lib, H_q, G, H_kv):
    """The V launch walks the layer's KV heads through the appended values: both must have as many."""
    fits = _layer(H=H_kv)
    for layer in (fits, fast_decode._pre_squeeze_packed((fits,))[0]):
        _attend(layer, lib, H_q=H_q, H_kv=H_kv, G=G)
    lib.calls.clear()
    for H in (1, 2, 4, 8):
        if H == H_kv or H_q % H:
            continue
        other = _layer(H=H)
        for layer in (other, fast_decode._pre_squeeze_packed((other,))[0]):
            with pytest.raises(RuntimeError):
                _attend(layer, lib, H_q=H_q, H_kv=H_kv, G=G)
    assert lib.calls == []


@pytest.mark.parametrize("width", [64, 127, 129, 256])
@pytest.mark.parametrize("packed", [True, False])
def test_attention_refuses_queries_of_other_width(lib, packed, width):
    """The scores of the appended tokens read 128 channels of every query row."""
    layer = _layer() if packed else dataclasses.replace(_layer(), T_eff=0, T_eff_k=0)
    with pytest.raises((RuntimeError, AssertionError)):
        _attend(layer, lib, width=width)
    with pytest.raises((RuntimeError, AssertionError)):
        _attend(layer, lib, width=width, out=torch.empty(8, 128))
    assert lib.calls == []


@pytest.mark.parametrize("name,shape", [("out", (8, 128)), ("scores_buf", (8, 16))])
def test_attention_refuses_buffers_of_another_device(lib, name, shape):
    layer = dataclasses.replace(_layer(), T_eff=0, T_eff_k=0)
    with pytest.raises(RuntimeError):
        _attend(layer, lib, **{name: torch.empty(shape, device="meta")})
    assert lib.calls == []


@pytest.mark.parametrize("make", [lambda: torch.empty(8, 128, dtype=torch.float16), lambda: torch.empty(1, 8, 128),
                                  lambda: torch.empty(3, 8, 128, dtype=torch.float64), lambda: torch.empty(128, 8).t()])
@pytest.mark.parametrize("default", [torch.float32, torch.float64, torch.bfloat16])
def test_attention_without_packed_tokens_fills_outputs_of_any_kind(lib, make, default):
    """The sum goes to a tensor of the kernel's form and from there to what the caller gave."""
    layer, out = dataclasses.replace(_layer(), T_eff=0, T_eff_k=0), make()
    torch.set_default_dtype(default)
    try:
        assert _attend(layer, lib, out=out) is out
    finally:
        torch.set_default_dtype(torch.float32)
    assert "rdkv_v_weighted_sum_new_values" in lib.calls
    with pytest.raises(RuntimeError):
        _attend(layer, lib, out=torch.empty(8, 128, dtype=torch.int64))


def _cut(t, dim, n=1):
    return t.narrow(dim, 0, t.shape[dim] - n)


def _refused(lib, call, layer, **changes):
    with pytest.raises((RuntimeError, IndexError)):
        call(dataclasses.replace(layer, **changes))
    assert not any(name.startswith("rdkv_unpack") for name in lib.calls), "refused behind the launch"


K_TENSORS = ("K_2bit", "K_4bit", "K_8bit", "K_ch_scale", "K_ch_zp")


@pytest.mark.parametrize("per_head", [True, False])
def test_dense_keys_refuse_tensors_that_do_not_fit(lib, per_head):
    layer = _layer(per_head=per_head)
    index = "K_ch_sort_idx_per_head" if per_head else "K_ch_sort_idx"

    def call(pl):
        return packing._unpack_k_enqueue(pl, 128)

    call(layer)
    assert lib.calls == ["rdkv_unpack_layer_k_checked" if per_head else "rdkv_unpack_layer_k"]
    lib.calls.clear()
    for name in K_TENSORS + (index,):
        t = getattr(layer, name)
        _refused(lib, call, layer, **{name: t.to("meta")})                      # of another device
        if name != index:
            _refused(lib, call, layer, **{name: _cut(t, 3)})                    # too few channels
    for name in ("K_2bit", "K_4bit", "K_8bit"):
        _refused(lib, call, layer, **{name: _cut(getattr(layer, name), 1)})     # too few heads
        _refused(lib, call, layer, **{name: _cut(getattr(layer, name), 2)})     # too few tokens
    _refused(lib, call, layer, K_ch_zp=_cut(layer.K_ch_zp, 1))
    _refused(lib, call, layer, **{index: getattr(layer, index).int()})
    if per_head:
        _refused(lib, call, layer, K_ch_sort_idx_per_head=_cut(layer.K_ch_sort_idx_per_head, 0))
        _refused(lib, call, layer, K_ch_seg_bounds_per_head=_cut(layer.K_ch_seg_bounds_per_head, 0))
        _refused(lib, call, layer, K_ch_seg_bounds_per_head=_cut(layer.K_ch_seg_bounds_per_head, 1))


def test_dense_keys_take_scales_and_counts_wider_than_needed(lib):
    """As the layer's fields allow: only the padded channels and the heads that exist are read."""
    layer = _layer()
    wide = torch.nn.functional.pad
    packing._unpack_k_enqueue(dataclasses.replace(
        layer, K_ch_zp=wide(layer.K_ch_zp, (0, 7)), K_8bit=torch.cat([layer.K_8bit] * 2, dim=1),
        K_ch_sort_idx_per_head=torch.cat([layer.K_ch_sort_idx_per_head] * 2),
        K_ch_seg_bounds_per_head=wide(layer.K_ch_seg_bounds_per_head, (0, 0, 0, 1), value=99)), 128)
    assert lib.calls == ["rdkv_unpack_layer_k_checked"]


@pytest.mark.parametrize("listed", [0, 1, 14])
def test_dense_keys_refuse_a_shared_index_that_lists_too_few_channels(lib, listed):
    layer = _layer(per_head=False)                      # keeps 15 channels
    _refused(lib, lambda pl: packing.unpack_k_mixed(pl, 128), layer, K_ch_sort_idx=layer.K_ch_sort_idx[:listed])
    packing.unpack_k_mixed(dataclasses.replace(layer, K_ch_sort_idx=torch.arange(20)), 128)
    assert lib.calls == ["rdkv_unpack_layer_k"]


@pytest.mark.parametrize("counts", [(-2, 6, 5), (4, -1, 5), (4, 6, -3), (-4, 6, 9)])
def test_dense_keys_report_negative_counts(lib, counts):
    layer = _layer()
    bad = layer.K_ch_seg_bounds_per_head.clone()
    bad[1] = torch.tensor(counts)
    with pytest.raises(AssertionError, match="negative"):
        packing.unpack_k_mixed(dataclasses.replace(layer, K_ch_seg_bounds_per_head=bad), 128)


@pytest.mark.parametrize("channel", [-1, 128, 1 << 40])
def test_dense_keys_report_channels_outside_the_head(lib, channel):
    layer = _layer()
    index = layer.K_ch_sort_idx_per_head.clone()
    index[1, 7] = channel
    cache = packing.TriZoneCache((dataclasses.replace(layer, K_ch_sort_idx_per_head=index),),
                                 [torch.zeros(1, 2, 3, 128).half()], [None], [None], 9)
    with pytest.raises(IndexError):
        packing.unpack_k_mixed(cache.packed[0], 128)
    with pytest.raises(IndexError):
        tz.unpack_trizone_to_past_kv(cache, head_dim=128)


V_SEGMENTS = ("V_2bit", "V_4bit", "V_8bit")


def test_dense_values_refuse_tensors_that_do_not_fit(lib):
    layer = _layer()

    def call(pl):
        return tz._unpack_v_enqueue(pl, None, 128)

    call(layer)
    assert lib.calls == ["rdkv_unpack_layer_v"]
    lib.calls.clear()
    for name in V_SEGMENTS + ("V_scale", "V_zp"):
        t = getattr(layer, name)
        _refused(lib, call, layer, **{name: t.to("meta")})                      # of another device
        if name != "V_scale":                                                   # (says how many heads there are)
            _refused(lib, call, layer, **{name: _cut(t, 1)})                    # too few heads
    for name in V_SEGMENTS:
        _refused(lib, call, layer, **{name: getattr(layer, name)[0]})
        _refused(lib, call, layer, **{name: torch.nn.functional.pad(getattr(layer, name), (0, 1))})
    for name in ("V_scale", "V_zp"):
        _refused(lib, call, layer, **{name: _cut(getattr(layer, name), 2)})     # fewer tokens than the stripe
    for name in ("seg_bounds_per_head", "T_eff_per_head"):
        _refused(lib, call, layer, **{name: _cut(getattr(layer, name), 0)})
    _refused(lib, call, layer, seg_bounds_per_head=_cut(layer.seg_bounds_per_head, 1))
    with pytest.raises(RuntimeError):
        tz._unpack_v_enqueue(layer, torch.zeros(1, 2, 3, 128, device="meta").half(), 128)


def test_dense_values_take_tensors_wider_than_needed(lib):
    layer = _layer()
    wide = torch.nn.functional.pad
    _, counts, totals = tz._unpack_v_enqueue(dataclasses.replace(
        layer, V_zp=wide(layer.V_zp, (0, 0, 0, 5)), V_4bit=torch.cat([layer.V_4bit] * 2, dim=1),
        seg_bounds_per_head=wide(layer.seg_bounds_per_head, (0, 0, 0, 1), value=99),
        T_eff_per_head=wide(layer.T_eff_per_head, (0, 1))), None, 128)
    assert lib.calls == ["rdkv_unpack_layer_v"] and counts.shape == (2, 3) and totals.shape == (2,)


@pytest.mark.parametrize("counts,total", [((-3, 4, 5), 6), ((4, -3, 5), 6), ((4, 5, -3), 6), ((-9, 4, 5), 0)])
def test_dense_values_report_more_rows_than_the_stripe(lib, counts, total):
    """A negative count adds no rows, so counts with the right sum may still have more rows than fit."""
    layer = dataclasses.replace(_layer(T=6), **{n: torch.zeros(1, 2, 6, w, dtype=torch.uint8)
                                                for n, w in zip(V_SEGMENTS, (32, 64, 128))})
    bounds, totals = layer.seg_bounds_per_head.clone(), layer.T_eff_per_head.clone()
    bounds[1], totals[1] = torch.tensor(counts), total
    bad = dataclasses.replace(layer, seg_bounds_per_head=bounds, T_eff_per_head=totals)
    with pytest.raises(AssertionError):
        tz._unpack_v_perhead(bad, head_dim=128)


def test_dense_values_of_a_layer_without_a_class_tensor(lib):
    """Tokens counted for a class that has no rows are left out; the rows behind them decide what fits."""
    layer = dataclasses.replace(_layer(T=6), V_2bit=None)                       # 2, 2 and 2 tokens
    out = tz._unpack_v_perhead(layer, head_dim=128)
    assert out.shape == (1, 2, 6, 128)
    counts = torch.tensor([[7, 2, 2]] * 2, dtype=torch.int32)
    tz._unpack_v_perhead(dataclasses.replace(layer, seg_bounds_per_head=counts,
                                             T_eff_per_head=counts.sum(1, dtype=torch.int32)), head_dim=128)


def test_counts_of_layers_on_several_devices_are_read_device_by_device(lib, monkeypatch):
    reads = []
    monkeypatch.setattr(_lib, "download", lambda t: (reads.append((t.device.type, t.numel())),
                                                     torch.arange(t.numel()).numpy())[1])
    seen = []
    note = lambda layer, rows: seen.append((layer, rows))
    tensors = [torch.zeros(2, 4, dtype=torch.int32, device=d) for d in ("cpu", "meta", "cpu", "meta")]
    tz._read_checks([(note, i, (t,)) for i, t in enumerate(tensors)])
    assert sorted(reads) == [("cpu", 16), ("meta", 16)]
    assert sorted(seen) == [(i, [[8 * (i // 2) + 4 * h + c for c in range(4)] for h in range(2)]) for i in range(4)]
