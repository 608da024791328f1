"""The host side in C++ (csrc/native.cpp) against the Python it stands in for, which takes every form that it leaves: the
same tensors, bit for bit, over the layouts, types and options that it takes, and the general path's own results and
errors over those that it does not.  Which of the two took a call is asserted."""
import dataclasses

import pytest
import torch

from rdkv_amd import _lib, knapsack_solver as ks, obkv_fast, packing, stream_cache, trizone_decompress as tz
from tests.gpu_util import DEV, record_native, require_gpu

gpu = pytest.mark.gpu


def _same(a, b):
    if isinstance(a, torch.Tensor):
        return a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
    return a == b


def test_other_forms_are_left_to_python():
    _lib.load()
    n = _lib.native
    x = torch.zeros(1, 2, 4, 128, dtype=torch.float16)                    # not on a device
    assert n.pack_layer(x, x, x, x, x, x, None, [], [], 0, 2, 1, 0) is None
    assert n.select_layer(x, x, x, x, (7, 1, 1), [0.0], [1.0], 1.0, [0.0], [1.0], 1.0, 0, 1, False, 0, 1, 0, 0, 0) is None
    assert n.dense_layer({}, None, 128, 0, 0, 1, 0) is None and n.dense_layer(3, None, 128, 0, 0, 1, 0) is None
    assert n.decode_attn({"units": None}, None, x, *[None] * 10, 0, 0, 0) is None
    with pytest.raises(TypeError):
        n.pack_layer(x)
    with pytest.raises(TypeError):
        n.dense_layer({}, None, "128", 0, 0, 1, 0)
    with pytest.raises(OverflowError):
        n.dense_layer({}, None, 1 << 80, 0, 0, 1, 0)


def _kv(H, T, layout, seed, D=128):
    g = torch.Generator(device=DEV).manual_seed(seed)
    K, V = (torch.randn(1, H, T, D, generator=g, device=DEV).half() for _ in range(2))
    if layout == "tokens first":
        K, V = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (K, V))
    elif layout == "apart":                       # different strides: the general path's
        V = V.transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "wide":
        K, V = (torch.cat([t, t], dim=3)[..., :D] for t in (K, V))
    elif layout == "f32 V":
        V = V.float()
    return K, V


@gpu
@pytest.mark.parametrize("layout", ["dense", "tokens first", "apart", "wide", "f32 V"])
@pytest.mark.parametrize("H,G,T,pool", [(2, 4, 1025, ("avg", 7, "reflect")), (3, 1, 70, ("max", 5, "zero")), (1, 8, 9, ("avg", 1, "reflect")),
                                        (4, 2, 3, ("avg", 7, "reflect")), (2, 2, 29001, ("avg", 7, "zero"))])
def test_selection(monkeypatch, layout, H, G, T, pool):
    require_gpu()
    K, V = _kv(H, T, layout, T)
    g = torch.Generator(device=DEV).manual_seed(7)
    tokens = torch.rand(H, T + 5, generator=g, device=DEV).exp()[:, 2:2 + T]          # rows of a wider tensor
    channels = torch.rand(H, 128, generator=g, device=DEV)
    for k_options in (None, torch.tensor([0.0, 2.0, 4.0, 8.0])):
        args = dict(gqa_factor=G, token_budget=max(T // 3, 1), k_budget_ratio=0.5, obs_window=32, pool_kernel_size=pool[1],
                    pool_padding=pool[2], pool_type=pool[0], v_bit_options=torch.tensor([0.0, 2.0, 4.0, 8.0]) if layout == "f32 V" else None,
                    k_bit_options=k_options, eps_V=ks.DEFAULT_EPSILON_V, eps_K=ks.DEFAULT_EPSILON_K, retain_allocation_metadata=H != 3)
        with monkeypatch.context() as m:
            calls = record_native(m)
            got = obkv_fast._perhead_select_and_pack(K, V, tokens, channels, **args)
            plain = [] if layout == "f32 V" else ["select_layer", "pack_layer"] if K.stride() == V.stride() else ["select_layer"]
            assert calls.taken == plain
        with monkeypatch.context() as m:
            m.setattr(obkv_fast, "_select_and_pack_native", lambda *a: None)
            m.setattr(_lib, "native", None)
            exp = obkv_fast._perhead_select_and_pack(K, V, tokens, channels, **args)
        for f in dataclasses.fields(packing.PackedKVLayer):
            assert _same(getattr(got[0], f.name), getattr(exp[0], f.name)), f.name
        assert _same(got[1], exp[1]) and got[2] == exp[2]
        if "pack_layer" in plain:
            assert got[0]._host_counts == exp[0]._host_counts
        # the dense tensors of that layer
        cache = packing.TriZoneCache((got[0],), [got[1]], [None], [None], T)
        with monkeypatch.context() as m:
            calls = record_native(m)
            a = tz.unpack_trizone_to_past_kv(cache, head_dim=128)
            assert calls.taken == ["dense_layer"]
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", None)
            b = tz.unpack_trizone_to_past_kv(cache, head_dim=128)
        assert _same(a[0][0], b[0][0]) and _same(a[0][1], b[0][1])


@gpu
def test_selection_with_unusual_arguments(monkeypatch):
    """What the general path takes or refuses, through the entry point."""
    require_gpu()
    K, V = _kv(2, 64, "dense", 1)
    tokens, channels = torch.rand(2, 64, device=DEV), torch.rand(2, 128, device=DEV)
    args = dict(gqa_factor=2, token_budget=16, k_budget_ratio=0.5, obs_window=32, pool_kernel_size=7, pool_padding="reflect",
                v_bit_options=None, k_bit_options=None, eps_V=ks.DEFAULT_EPSILON_V, eps_K=ks.DEFAULT_EPSILON_K)
    call = obkv_fast._perhead_select_and_pack
    want = call(K, V, tokens, channels, **args)[0]
    for t, c in ((tokens.cpu(), channels), (tokens, channels.cpu()), (tokens.double(), channels.double())):
        assert _same(call(K, V, t, c, **args)[0].V_scale, want.V_scale)
    timing = {}
    assert _same(call(K, V, tokens, channels, timing=timing, **args)[0].K_ch_scale, want.K_ch_scale) and timing["pooling_ms"] > 0
    with pytest.raises(AssertionError):
        call(K, V, tokens[0], channels, **args)
    with pytest.raises(AssertionError):
        call(K, V, tokens, channels[:, :64], **args)
    with pytest.raises(KeyError):
        call(K, V, tokens, channels, **dict(args, eps_V={0: 1.0}))
    with pytest.raises(AssertionError):
        call(K, V, tokens, channels, **dict(args, k_bit_options=torch.tensor([0.0, 2.5]), eps_K={0: 1.0, 2: 0.3}))


@gpu
@pytest.mark.parametrize("G", [1, 4, 5, 8])
@pytest.mark.parametrize("q_dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
def test_decode_step(monkeypatch, G, q_dtype):
    require_gpu()
    K, V = _kv(2, 300, "dense", G)
    g = torch.Generator(device=DEV).manual_seed(G)
    v_bits = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (2, 300), generator=g, device=DEV)]
    k_bits = torch.full((2, 128), 4, device=DEV)
    cache = stream_cache.build_stream_cache_from_kv([(K, V, v_bits, k_bits)] * 2, G)
    rows, heads = cache.rows, cache.rows // G
    wide = torch.randn(rows, 200, generator=g, device=DEV).to(q_dtype)
    step = torch.randn(2, heads, 140, generator=g, device=DEV)
    ang = torch.rand(64, generator=g, device=DEV)
    counts = torch.randint(1, 30, (heads,), generator=g, device=DEV, dtype=torch.int32)
    row = torch.tensor([4], device=DEV)
    forms = [dict(), dict(rope=(ang.cos(), ang.sin())), dict(rope=(ang.cos().half(), ang.sin().half()), zone_c=2),
             dict(zone_c=3), dict(zone_c=2, q_dense=True), dict(zone_c=3, append=torch.float16, rope=(ang.cos(), ang.sin())),
             dict(zone_c=3, append=torch.float32, out=True), dict(out=True), dict(zone_c=3, append=torch.bfloat16, q_dense=True, out=True),
             dict(one_launch=False)]

    def run(form):
        buf = torch.randn(heads, 40, 264, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV)
        kw = dict(form)
        q = wide[:, :128].contiguous() if kw.pop("q_dense", False) else wide[:, 40:168]
        if "zone_c" in kw:
            kw["zone_c"] = (buf[:, :, :128], buf[:, :, 132:260], counts)[:kw["zone_c"]]
        if "append" in kw:
            dt = kw["append"]
            kw["append"] = (step[0, :, :128].to(dt), step[1, :, 5:133].to(dt), row)
        if kw.pop("out", False):
            kw["out"], kw["lse"] = torch.full((rows, 160), 7.0, device=DEV)[:, :128], torch.empty(rows, device=DEV)
        out, lse = stream_cache.decode_attn_fused(cache, q, **kw)
        assert "out" not in kw or (out is kw["out"] and lse is kw["lse"])
        return out, lse, buf

    for form in forms:
        with monkeypatch.context() as m:
            calls = record_native(m)
            got = run(form)
            assert calls.taken == ([] if q_dtype is torch.float64 else ["decode_attn"])
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", None)
            exp = run(form)
        assert all(_same(a, b) for a, b in zip(got, exp)), form
    stream_cache.decode_attn_fused(cache, wide[:, :128], append=(1, 2))            # (without zone C it is not looked at)
    for bad in (dict(q=wide), dict(zone_c=(step[0, :, None, :128], step[1, :1, None, :128])), dict(zone_c=(step[:, :, None, :128].contiguous()[0], step[:, :, None, :128].contiguous()[1]), append=(1, 2, 3)),
                dict(out=torch.empty(rows, 128, device=DEV, dtype=torch.float16)), dict(rope=(ang[:5], ang[:5]))):
        with pytest.raises((AssertionError, AttributeError)):
            stream_cache.decode_attn_fused(cache, **{"q": wide[:, :128], **bad})


@gpu
@pytest.mark.parametrize("widths", [torch.int64, torch.uint8, torch.int16, torch.float32])
@pytest.mark.parametrize("T,layers,layout", [(1, 1, "dense"), (65, 3, "tokens first"), (300, 2, "apart"), (700, 2, "wide"), (28673, 2, "dense")])
def test_layers_to_the_streaming_format(monkeypatch, widths, T, layers, layout):
    """Blobs (every byte that is written), descriptors, scales and results; the last layer keeps no channel in one form."""
    require_gpu()
    if T > 20000 and widths is not torch.int64:
        pytest.skip("one type is enough for a long layer")
    G, H = 4, 2
    g = torch.Generator(device=DEV).manual_seed(T)
    entries = []
    for i in range(layers):
        K, V = _kv(H, T, layout, 10 * T + i)
        v_bits = torch.tensor([0, 2, 4, 8, 16], device=DEV)[torch.randint(0, 5, (H, T), generator=g, device=DEV)]
        v_bits[:, 0] = 4
        k_bits = torch.tensor([0, 2, 4, 8], device=DEV)[torch.randint(0, 4, (H, 128), generator=g, device=DEV)]
        entries.append((K, V, v_bits.to(widths), k_bits.to(widths)))
    for empty_layer in (False, True) if T == 65 else (False,):
        if empty_layer:
            entries[-1] = (*entries[-1][:3], torch.zeros_like(entries[-1][3]))
        monkeypatch.setattr(stream_cache, "_POISON_BLOBS", True)
        with monkeypatch.context() as m:
            calls = record_native(m)
            got = stream_cache.build_stream_cache_from_kv(entries, G)
            plain = layout != "apart" and widths is not torch.float32
            assert calls.taken == ([] if not plain else ["stream_order"] if empty_layer else ["stream_order", "stream_tables", "stream_pack"])
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", None)                                  # (the general path)
            exp = stream_cache.build_stream_cache_from_kv(entries, G)
        assert len(got.blobs) == len(exp.blobs) == layers
        for i, (a, b) in enumerate(zip(got.blobs, exp.blobs)):
            end = -256 if empty_layer and i == layers - 1 or not plain else None      # (the re-layout leaves its slack)
            assert torch.equal(a[:end], b[:end]) and a.shape == b.shape
        for name in ("n_units", "n_work", "rows", "stream_bytes", "algorithmic_bytes", "max_row_dwords", "row_shape", "n_groups",
                     "kv_algorithmic_bytes", "h_q"):
            assert getattr(got, name) == getattr(exp, name), name
        assert (got.unit_scale_max == exp.unit_scale_max).all()
        addresses = ("k_off", "v_off", "sz_off", "qtab_off")
        for name in got.units_host.dtype.names:
            a, b = got.units_host[name].copy(), exp.units_host[name].copy()
            if name in addresses:
                for u in range(got.n_units):
                    a[u] -= got.blobs[u // H].data_ptr()
                    b[u] -= exp.blobs[u // H].data_ptr()
            assert (a == b).all(), name
        q = torch.randn(got.rows, 128, generator=g, device=DEV)
        for x, y in zip(stream_cache.decode_attn_fused(got, q), stream_cache.decode_attn_fused(exp, q)):
            assert torch.equal(x, y)
