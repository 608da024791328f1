"""Errors and lifetimes in csrc/native.cpp: an allocation that fails is torch's own OutOfMemoryError, which programs catch
to free memory and try again, from every entry point that allocates, and the call after it gives what it gave before;
fields that another thread replaces while a call runs without the interpreter's lock stay whole for that call."""
import contextlib
import dataclasses
import gc

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from rdkv_amd import _lib, knapsack_solver as ks, obkv_fast, packing, stream_cache, trizone_decompress as tz
from tests.gpu_util import DEV, record_native, require_gpu

pytestmark = pytest.mark.gpu
H, T, G = 2, 300, 4


@contextlib.contextmanager
def _no_memory_left():
    """The process may take no more of the device than it has, and the allocator's free pieces are taken."""
    taken = []
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(0.0)
    try:
        for n in (1 << 20, 1 << 16, 512):
            with contextlib.suppress(torch.OutOfMemoryError):
                while True:
                    taken.append(torch.empty(n, dtype=torch.uint8, device=DEV))
        yield
    finally:
        del taken
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.fixture(scope="module")
def calls():
    """By the entry point that it has to reach: the call."""
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(5)
    K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    v_bits = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
    k_bits = torch.full((H, 128), 4, device=DEV)
    scores, channels = torch.rand(H, T, device=DEV, generator=g), torch.rand(H, 128, device=DEV, generator=g)
    options = dict(gqa_factor=G, token_budget=100, k_budget_ratio=0.5, obs_window=32, pool_kernel_size=7, pool_padding="reflect",
                   v_bit_options=None, k_bit_options=None, eps_V=ks.DEFAULT_EPSILON_V, eps_K=ks.DEFAULT_EPSILON_K)
    planned = packing._plan_layers(v_bits, k_bits, K.device, (K,), 256)
    layer, v16 = packing.pack_layer_per_head(K, V, v_bits, k_bits, G)
    cache = stream_cache.build_stream_cache_from_kv([(K, V, v_bits, k_bits)], G)
    q = torch.randn(cache.rows, 128, device=DEV, dtype=torch.float16, generator=g)
    dense = packing.TriZoneCache((layer,), [v16], [None], [None], T)
    return {
        "select_layer": lambda: obkv_fast._perhead_select_and_pack(K, V, scores, channels, **options)[0].V_scale,
        "pack_layer": lambda: packing._pack_planned_layer(K, V, G, planned, 0, H)[0].K_4bit,
        "stream_order": lambda: stream_cache.build_stream_cache_from_kv([(K, V, v_bits, k_bits)], G).blobs[0],
        "dense_layer": lambda: tz.unpack_trizone_to_past_kv(dense, head_dim=128)[0][0],
        "decode_attn": lambda: stream_cache.decode_attn_fused(cache, q)[0],
    }


@pytest.mark.parametrize("name", ["select_layer", "pack_layer", "stream_order", "dense_layer", "decode_attn"])
def test_out_of_memory(calls, name, monkeypatch):
    reached = record_native(monkeypatch)
    want = calls[name]().clone()
    assert name in reached.taken
    reached.asked.clear()
    with _no_memory_left():
        with pytest.raises(torch.OutOfMemoryError):
            calls[name]()
        assert reached.asked == [name]
    assert torch.equal(calls[name](), want)


class _Replacing(TorchDispatchMode):
    """Runs ``change`` under the first allocation, which a native call makes without the lock, as another thread might."""

    def __init__(self, change):
        super().__init__()
        self.change = change

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if self.change is not None:
            change, self.change = self.change, None
            change()
            gc.collect()
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("fields", [("K_ch_scale", "K_ch_zp", "K_ch_sort_idx_per_head", "K_ch_seg_bounds_per_head"),
                                    ("V_scale", "V_zp", "seg_bounds_per_head", "T_eff_per_head", "K_4bit", "V_2bit", "softmax_mask")])
def test_layer_fields_replaced_under_a_call(fields):
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(5)
    K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    v_bits = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
    layer, v16 = packing.pack_layer_per_head(K, V, v_bits, torch.full((H, 128), 4, device=DEV), G)
    dense = packing.TriZoneCache((layer,), [v16], [None], [None], T)
    (want,), (mask,) = tz.unpack_trizone_to_past_kv(dense, head_dim=128, return_masks=True)
    spare = {f: torch.full_like(getattr(layer, f), 1) for f in fields}
    with _Replacing(lambda: layer.__dict__.update(spare)) as mode:
        native = _lib.native.dense_layer(layer.__dict__, (v16, layer.softmax_mask, 0), 128, *_words(layer), _lib.stream_of(K.device))
    assert mode.change is None and all(getattr(layer, f) is spare[f] for f in fields)
    torch.cuda.synchronize()
    for a, b in zip(native, (*want, mask)):
        assert torch.equal(a, b)


def _words(layer):
    n = int(layer.K_ch_scale.shape[1])
    words = _lib.host_words(layer.K_ch_scale.device, 8 * n)
    return words.take(4 * n), words.take(4 * n), words.tag


def test_cache_tables_replaced_under_a_call():
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(6)
    K, V = (torch.randn(1, H, 3000, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    bits = torch.full((H, 3000), 4, device=DEV)
    cache = stream_cache.build_stream_cache_from_kv([(K, V, bits, torch.full((H, 128), 4, device=DEV))], G, n_groups=3)
    assert cache.n_groups != cache.n_work
    q = torch.randn(cache.rows, 128, device=DEV, dtype=torch.float16, generator=g)
    want = stream_cache.decode_attn_fused(cache, q)
    tables = {f: getattr(cache, f).clone() for f in ("units", "work", "groups")}
    with _Replacing(lambda: cache.__dict__.update(tables)) as mode:
        got = stream_cache.decode_attn_fused(cache, q)
    assert mode.change is None and cache.units is tables["units"]
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_parts_of_a_step_that_are_none_are_refused():
    """Given, but empty, is not the same as not given: no step without the rotation or the appended row that was asked for."""
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(7)
    K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    cache = stream_cache.build_stream_cache_from_kv([(K, V, torch.full((H, T), 4, device=DEV), torch.full((H, 128), 4, device=DEV))], G)
    q = torch.randn(cache.rows, 128, device=DEV, dtype=torch.float16, generator=g)
    new = torch.zeros(H, 4, 128, device=DEV)
    zone_c = (new, new.clone(), torch.ones(H, dtype=torch.int32, device=DEV))
    row, x = torch.zeros(1, dtype=torch.int64, device=DEV), torch.zeros(H, 128, device=DEV, dtype=torch.float16)
    for bad in (dict(rope=(None, None)), dict(zone_c=(None, None)), dict(zone_c=(None, None, zone_c[2])), dict(zone_c=zone_c, append=(None, None, None)),
                dict(zone_c=zone_c, append=(None, x, row)), dict(zone_c=zone_c, append=(x, None, row)), dict(zone_c=zone_c, append=(x, x, None)),
                dict(rope=(torch.zeros(64, device=DEV), None)), dict(zone_c=(new, None))):
        with pytest.raises((AttributeError, AssertionError)):
            stream_cache.decode_attn_fused(cache, q, **bad)
    assert not new.any()


def test_layers_without_v_scales_take_no_words_for_them(monkeypatch):
    """As many layers that keep only fp16 tokens, and have no tensor of V scales, as fill the words of one call."""
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(8)
    heads, layers = 8, 128
    K, V = (torch.randn(1, heads, 5, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    layer, v16 = packing.pack_layer_per_head(K, V, torch.full((heads, 5), 16, device=DEV), torch.full((heads, 128), 4, device=DEV), G)
    assert layer.T_eff == 0
    bare = dataclasses.replace(layer, V_scale=None, V_zp=None)
    monkeypatch.setattr(_lib, "_host_words", {})
    assert _lib.host_words(K.device, 4 * heads * layers).size == 4 * heads * layers
    _lib.host_words(K.device, 1).pending = False
    got = tz.unpack_trizone_to_past_kv(packing.TriZoneCache((bare,) * layers, [v16] * layers, [None] * layers, [None] * layers, 5), head_dim=128)
    want, = tz.unpack_trizone_to_past_kv(packing.TriZoneCache((layer,), [v16], [None], [None], 5), head_dim=128)
    assert len(got) == layers and all(torch.equal(k, want[0]) and torch.equal(v, want[1]) for k, v in got)


@pytest.mark.parametrize("extra", [0.0, -1.0, -3, True, 2])
def test_numbers_of_new_tokens(extra):
    """Zero and less, as any number, add nothing to the masks; a layer's sizes may be any numbers too."""
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(9)
    K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
    layer, v16 = packing.pack_layer_per_head(K, V, torch.full((H, T), 4, device=DEV), torch.full((H, 128), 4, device=DEV), G)
    dense = packing.TriZoneCache((layer,), [v16], [None], [None], T)
    layer.T_eff, layer.n_v16 = float(layer.T_eff), torch.tensor(float(layer.n_v16))            # (sizes of a layer made by hand)
    _, (mask,) = tz.unpack_trizone_to_past_kv(dense, head_dim=128, return_masks=True, max_new_tokens=extra)
    assert torch.equal(mask, torch.zeros(1, H * G, 1, T + max(int(extra), 0), dtype=torch.float16, device=DEV))


def test_an_entry_that_keeps_no_channel_leaves_the_plan_to_the_others(monkeypatch):
    """The general path takes the entries with the plan that the native call has made: none is planned again but the one
    that is packed on its own."""
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(10)
    entries = []
    for i in range(3):
        K, V = (torch.randn(1, H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(2))
        v_bits = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (H, T), device=DEV, generator=g)]
        k_bits = torch.tensor([0, 2, 4, 8], device=DEV)[torch.randint(0, 4, (H, 128), device=DEV, generator=g)]
        if i == 1:
            k_bits.zero_()
        entries.append((K, V, v_bits, k_bits))
    plans, plan_layers = [], packing._plan_layers
    monkeypatch.setattr(packing, "_plan_layers", lambda v, *a, **k: (plans.append(len(v)), plan_layers(v, *a, **k))[1])
    got = stream_cache.build_stream_cache_from_kv(entries, G)
    assert plans and set(plans) == {H}
    monkeypatch.setattr(_lib, "native", None)
    exp = stream_cache.build_stream_cache_from_kv(entries, G)
    assert 3 * H in plans
    for a, b in zip(got.blobs, exp.blobs):
        assert torch.equal(a[:-256], b[:-256])
    assert (got.unit_scale_max == exp.unit_scale_max).all()
    q = torch.randn(got.rows, 128, device=DEV, dtype=torch.float16, generator=g)
    for a, b in zip(stream_cache.decode_attn_fused(got, q), stream_cache.decode_attn_fused(exp, q)):
        assert torch.equal(a, b)
