"""The planning launches' numbers on their way to the host (``rdkv_pack_layer_plan_start`` / ``_wait``), and the
K min / max that are launched ahead of the host's read of them."""
import ctypes
import dataclasses
import threading

import pytest
import torch

from rdkv_amd import _lib, packing, stream_cache
from tests.gpu_util import DEV, require_gpu

gpu = pytest.mark.gpu


def _wait(words, heads, tag, wait_us=2000):
    out = (ctypes.c_int32 * max(12 * heads, 1))()
    return _lib.load().rdkv_pack_layer_plan_wait(words.data_ptr(), heads, tag, out, wait_us), list(out)


@pytest.mark.parametrize("heads", [1, 2, 7])
@pytest.mark.parametrize("tag", [1, 0x80000000, 0xFFFFFFFF])
def test_words_in_plan_order(heads, tag):
    """[heads][4] counts, then [heads][8] further numbers, from twelve words a head; negative values too."""
    values = torch.arange(-3, 12 * heads - 3)
    words = (values & 0xFFFFFFFF) | (torch.tensor(tag if tag < 1 << 31 else tag - (1 << 32)) << 32)
    rc, got = _wait(words, heads, tag)
    v = values.view(heads, 12)
    assert rc == 0 and got == v[:, :4].flatten().tolist() + v[:, 4:].flatten().tolist()
    for at in (0, 12 * heads - 1):                 # one word still of an earlier call
        old = words.clone()
        old[at] = (int(old[at]) & 0xFFFFFFFF) | ((tag - 1 & 0x7FFFFFFF) << 32)
        assert _wait(old, heads, tag)[0] == -5


def test_words_that_come_late():
    words = torch.zeros(12, dtype=torch.int64)
    filled = (torch.arange(12) | (5 << 32))
    t = threading.Timer(0.05, lambda: words.copy_(filled))
    t.start()
    rc, got = _wait(words, 1, 5, 5_000_000)
    t.join()
    assert rc == 0 and got == list(range(12))


def _alloc(N, T, D, seed):
    g = torch.Generator().manual_seed(seed)
    vb = torch.tensor([0, 2, 4, 8, 16])[torch.randint(0, 5, (N, T), generator=g)]
    kb = torch.tensor([0, 2, 4, 8])[torch.randint(0, 4, (N, D), generator=g)]
    kb[:, 0] = 4
    return vb, kb


@gpu
@pytest.mark.parametrize("N,T", [(1, 1), (8, 1023), (3, 1025), (300, 40)])
def test_plan_by_words_and_by_copy(monkeypatch, N, T):
    require_gpu()
    vb, kb = (t.to(DEV) for t in _alloc(N, T, 128, N + T))
    dev = vb.device
    seen = []
    read = packing._read_ints
    monkeypatch.setattr(packing, "_read_ints", lambda *a: (seen.append(1), read(*a))[1])
    for _ in range(3):
        by_words = packing._plan_layers(vb, kb, dev)
    assert not seen

    class Late:                                  # the words are not there in time: the stream's own wait takes over
        def __getattr__(self, name):
            return (lambda *a: -5) if name == "rdkv_pack_layer_plan_wait" else getattr(lib, name)
    lib = _lib.load()
    monkeypatch.setattr(_lib, "load", lambda: Late())
    by_copy = packing._plan_layers(vb, kb, dev)
    assert seen == [1]
    assert by_words[3] == by_copy[3] and by_words[4] == by_copy[4]
    for a, b in zip(by_words[:2], by_copy[:2]):
        assert torch.equal(a, b)


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
        if D == 128:
            cache = stream_cache.build_stream_cache_from_kv(
                [(K, V, vb[l], kb[l]) for l, (K, V) in enumerate(zip(Ks, Vs))], 2)
        got.append((layers, cache))
    for (a, va), (b, vb_) in zip(got[0][0], got[1][0]):
        _same(a, b)
        assert (va is None) == (vb_ is None) and (va is None or torch.equal(va, vb_))
    if got[0][1] is not None:
        a, b = got[0][1], got[1][1]
        assert (a.unit_scale_max == b.unit_scale_max).all() and a.n_work == b.n_work
        for x, y in zip(a.blobs, b.blobs):
            assert torch.equal(x[:-256], y[:-256])
