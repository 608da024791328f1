"""Numbers that launches send to the host by themselves (``_lib.HostWords``, ``rdkv_host_words_wait``): the plan of the
packers, with the K min / max that are launched ahead of the host's read of it, and the counts of the dense route."""
import ctypes
import dataclasses
import threading

import pytest
import torch

from rdkv_amd import _lib, fast_decode, packing, stream_cache, trizone_decompress as tz
from tests.gpu_util import DEV, record_native, require_gpu

gpu = pytest.mark.gpu


def _wait(words, n, tag, wait_us=2000):
    out = (ctypes.c_int32 * max(n, 1))()
    return _lib.load().rdkv_host_words_wait(words.data_ptr(), n, tag, out, wait_us), list(out)[:n]


def _tagged(values, tag):
    return (values & 0xFFFFFFFF) | (torch.tensor(tag if tag < 1 << 31 else tag - (1 << 32)) << 32)


@pytest.mark.parametrize("n", [0, 1, 2, 77])
@pytest.mark.parametrize("tag", [1, 0x80000000, 0xFFFFFFFF])
def test_words_are_whole_or_waited_for(n, tag):
    values = torch.arange(n) * 99991 - 3
    words = _tagged(values, tag)
    rc, got = _wait(words, n, tag)
    assert rc == 0 and got == values.tolist()
    for at in {0, n - 1} if n else ():              # one word still of an earlier call
        old = words.clone()
        old[at] = _tagged(values[at], tag - 1 & 0x7FFFFFFF)
        assert _wait(old, n, tag)[0] == _lib.RDKV_EWAIT


def test_words_that_come_late():
    words = torch.zeros(12, dtype=torch.int64)
    t = threading.Timer(0.05, lambda: words.copy_(_tagged(torch.arange(12), 5)))
    t.start()
    rc, got = _wait(words, 12, 5, 5_000_000)
    t.join()
    assert rc == 0 and got == list(range(12))


def _alloc(N, T, D, seed):
    g = torch.Generator().manual_seed(seed)
    vb = torch.tensor([0, 2, 4, 8, 16])[torch.randint(0, 5, (N, T), generator=g)]
    kb = torch.tensor([0, 2, 4, 8])[torch.randint(0, 4, (N, D), generator=g)]
    kb[:, 0] = 4
    return vb, kb


class _Late:
    """The library, whose words are not there on the first look."""

    def __init__(self, lib):
        self.lib, self.looks = lib, []

    def __getattr__(self, name):
        fn = getattr(self.lib, name)
        if name != "rdkv_host_words_wait":
            return fn

        def wait(*args):
            self.looks.append(args[-1])
            return _lib.RDKV_EWAIT if len(self.looks) == 1 else fn(*args)
        return wait


@gpu
@pytest.mark.parametrize("N,T", [(1, 1), (8, 1023), (3, 1025), (600, 40)])
def test_plan_and_its_numbers(monkeypatch, N, T):
    require_gpu()
    vb, kb = (t.to(DEV) for t in _alloc(N, T, 128, N + T))
    for again in range(3):
        order, rank3, plan, counts, info, _, _ = packing._plan_layers(vb, kb, vb.device)
        on_device = plan[:12 * N].tolist()
        assert counts == [on_device[4 * h:4 * h + 4] for h in range(N)]
        assert info == [on_device[4 * N + 8 * h:4 * N + 8 * h + 8] for h in range(N)]
        assert counts == [[int((row == b).sum()) for b in (2, 4, 8, 16)] for row in vb.cpu()]
    late = _Late(_lib.load())                       # the stream's own wait takes over
    monkeypatch.setattr(_lib, "load", lambda: late)
    assert packing._plan_layers(vb, kb, vb.device)[3] == counts
    assert late.looks == [_lib.HostWords.WAIT_US, 0]


@gpu
def test_words_of_a_call_that_was_not_read(monkeypatch):
    """The next call waits for the device first (a launch may still write to them), one that follows a read does not."""
    require_gpu()
    dev = torch.empty(1, device=DEV).device
    waits, sync = [], torch.cuda.synchronize
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: (waits.append(1), sync(*a))[1])
    vb, kb = (t.to(DEV) for t in _alloc(2, 30, 128, 1))
    want = packing._plan_layers(vb, kb, dev)[3]
    assert not waits
    _lib.host_words(dev, 24)
    assert packing._plan_layers(vb, kb, dev)[3] == want and waits == [1]
    assert packing._plan_layers(vb, kb, dev)[3] == want and waits == [1]


@gpu
@pytest.mark.parametrize("late", [False, True])
def test_dense_counts_by_words(monkeypatch, late):
    """The dense tensors and what is refused, whichever way the counts come back."""
    require_gpu()
    vb, kb = _alloc(6, 90, 128, 8)
    g = torch.Generator().manual_seed(4)
    Ks, Vs = ([torch.randn(1, 3, 90, 128, generator=g).half().to(DEV) for _ in range(2)] for _ in range(2))
    layers = packing.pack_layers_per_head(Ks, Vs, vb.view(2, 3, 90), kb.view(2, 3, 128), 2)
    n = len(layers)

    def cache(**changed):
        packed = [layers[0][0], dataclasses.replace(layers[1][0], **changed)]
        return packing.TriZoneCache(tuple(packed), [v for _, v in layers], [None] * n, [None] * n, 90)

    by_words = tz.unpack_trizone_to_past_kv(cache(), head_dim=128)
    monkeypatch.setattr(tz, "_words_of", lambda *a: None)
    by_copy = tz.unpack_trizone_to_past_kv(cache(), head_dim=128)
    monkeypatch.undo()
    for a, b in zip(by_words, by_copy):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    if late:
        slow = _Late(_lib.load())
        monkeypatch.setattr(_lib, "load", lambda: slow)
    pl = layers[1][0]
    with pytest.raises(AssertionError):
        tz.unpack_trizone_to_past_kv(cache(T_eff_per_head=pl.T_eff_per_head + 1), head_dim=128)
    with pytest.raises(AssertionError):
        tz.unpack_trizone_to_past_kv(cache(K_ch_seg_bounds_per_head=pl.K_ch_seg_bounds_per_head - 100), head_dim=128)
    with pytest.raises(IndexError):
        tz.unpack_trizone_to_past_kv(cache(K_ch_sort_idx_per_head=pl.K_ch_sort_idx_per_head + 100), head_dim=128)
    assert len(tz.unpack_trizone_to_past_kv(cache(), head_dim=128)) == n


@gpu
@pytest.mark.parametrize("position", [0, 41, (1 << 32) - 2])
def test_token_words(position):
    """Eager steps and a replayed graph leave each step's token under the position it moved on to."""
    require_gpu()
    logits = torch.randn(3, 1000, device=DEV).half()
    row = logits[0].clone()
    token = torch.zeros(1, 1, dtype=torch.long, device=DEV)
    pos = torch.full((1, 1), position, dtype=torch.long, device=DEV)
    for _ in range(2):
        pos.fill_(position)
        word = _lib.step_word(token.device, 5, position)
        fast_decode._argmax_advance(row, token, pos, word=word)
        assert word.read(position + 1) == int(logits[0].argmax()) == int(token)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            fast_decode._argmax_advance(row, token, pos, word=word)
        for step in range(1, 4):
            row.copy_(logits[step % 3])
            graph.replay()
            assert word.read(position + step + 1) == int(logits[step % 3].argmax()) == int(token)
        row.copy_(logits[0])


def test_words_of_loops_never_share_a_tag(monkeypatch):
    """The ring's words come round with other tags; two loops in a row have words of their own."""
    dev = torch.device("cuda", 63)
    monkeypatch.setattr(_lib, "_step_words", {(63, threading.get_ident()): [torch.zeros(64, dtype=torch.int64), 0, [0] * 64]})
    seen = set()
    for loop in range(200):
        steps, position = 1 + loop % 7, 1000 * loop
        word = _lib.step_word(dev, steps, position)
        tags = {(word.ptr, (word.tag_base + position + k) & 0xFFFFFFFF) for k in range(1, steps + 1)}
        assert len(tags) == steps and not tags & seen and all(tag for _, tag in tags)
        seen |= tags


def _same(a, b):
    for f in dataclasses.fields(a):
        x, y = getattr(a, f.name), getattr(b, f.name)
        assert (torch.equal(x, y) if isinstance(x, torch.Tensor) else x == y), f.name


@gpu
@pytest.mark.parametrize("T,D,form", [(1, 128, "dense"), (511, 128, "dense"), (513, 128, "token major"), (1500, 64, "dense"),
                                      (700, 128, "odd"), (129, 132, "dense")])
def test_minmax_ahead_of_the_read(monkeypatch, T, D, form):
    """The same layers whether the K min / max are launched ahead of the host's read or behind it."""
    require_gpu()
    H, L = 3, 3
    g = torch.Generator().manual_seed(T + D)
    wide = torch.randn(L, 2, 1, T, H, D + 2, generator=g).half().to(DEV)
    kv = wide[..., 2:] if form == "odd" else wide[..., :D].contiguous()
    kv = kv.permute(0, 1, 2, 4, 3, 5)
    if form == "dense":
        kv = kv.contiguous()
    vb, kb = _alloc(L * H, T, D, 3)
    vb[0] = 0                                                    # a head without tokens, one with all of one width
    vb[1] = 8
    if T > 1:
        vb[H:, 0] = 2
    vb, kb = vb.to(DEV).view(L, H, T), kb.to(DEV).view(L, H, D)
    Ks, Vs = list(kv[:, 0]), list(kv[:, 1])
    got = []
    for tokens in (1, 1 << 30):
        monkeypatch.setattr(packing, "_EARLY_MINMAX_TOKENS", tokens)
        assert packing._early_minmax(Ks, Ks[0].device) == (tokens == 1)
        layers = packing.pack_layers_per_head(Ks, Vs, vb, kb, 2)
        layers += [packing.pack_layer_per_head(Ks[1], Vs[1], vb[1], kb[1], 2)]
        cache = None
        if D == 128:            # (the streaming packer takes them ahead always: by its native calls, by the general path)
            with monkeypatch.context() as m:
                if tokens == 1:
                    calls = record_native(m)
                else:
                    m.setattr(_lib, "native", None)
                cache = stream_cache.build_stream_cache_from_kv(
                    [(K, V, vb[l], kb[l]) for l, (K, V) in enumerate(zip(Ks, Vs))], 2)
            assert ("stream_pack" in calls.taken) == (form != "odd")
        got.append((layers, cache))
    for (a, va), (b, vb_) in zip(got[0][0], got[1][0]):
        _same(a, b)
        assert (va is None) == (vb_ is None) and (va is None or torch.equal(va, vb_))
    if got[0][1] is not None:
        a, b = got[0][1], got[1][1]
        assert (a.unit_scale_max == b.unit_scale_max).all() and a.n_work == b.n_work
        for x, y in zip(a.blobs, b.blobs):
            assert torch.equal(x[:-256], y[:-256])
