"""The zone C merge with one, two or all heads of a unit per workgroup (the launch picks by the number
of units): the same bits whichever way, and the exact softmax over the union, at the edges of its
64-token chunks and of the eight tokens of a wavefront, for values that start at any float, for the
step's own token anywhere in the buffer, and for scores of -inf."""
import numpy as np
import pytest
import torch

from rdkv_amd import stream_cache
from tests.gpu_util import DEV, lse_merge, require_gpu, t2n

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 7, 8, 9, 63, 64, 65, 71, 128, 129, 300)


def _cache(G, layers, heads, seed):
    g = torch.Generator().manual_seed(seed)
    entries = []
    for _ in range(layers):
        K, V = (torch.randn(1, heads, 70, 128, generator=g).half().to(DEV) for _ in range(2))
        v_bits = torch.tensor([0, 2, 4, 8, 16])[torch.randint(0, 5, (heads, 70), generator=g)]
        k_bits = torch.tensor([0, 2, 4, 8])[torch.randint(0, 4, (heads, 128), generator=g)]
        v_bits[:, 0], k_bits[:, 0] = 4, 4
        entries.append((K, V, v_bits.to(DEV), k_bits.to(DEV)))
    return stream_cache.build_stream_cache_from_kv(entries, G)


@pytest.mark.parametrize("G,layers,heads", [(1, 1, 2), (2, 2, 8), (3, 1, 4), (4, 1, 8), (5, 2, 3), (8, 1, 4),
                                            (2, 17, 8), (4, 9, 8), (6, 6, 8), (7, 5, 8), (8, 5, 8)])
def test_heads_per_workgroup(G, layers, heads):
    require_gpu()
    cache = _cache(G, layers, heads, 10 * G + layers)
    rows_kv = layers * heads
    g = torch.Generator().manual_seed(G)
    cap = 300
    counts = torch.tensor([COUNTS[(i + G) % len(COUNTS)] for i in range(rows_kv)], dtype=torch.int32)
    wide = torch.randn(rows_kv, cap, 260, generator=g).to(DEV)
    k_buf, v_buf = wide[:, :, :128], wide[:, :, 129:257]              # values at an odd float
    past = torch.arange(cap)[None, :, None] >= counts[:, None, None]
    wide.masked_fill_(past.to(DEV), float("nan"))                      # rows past the count may hold anything
    q = torch.randn(cache.rows, 128, generator=g).to(DEV)
    counts_d = counts.to(DEV)
    out_ab, lse_ab = stream_cache.decode_attn_fused(cache, q)
    out, lse = stream_cache.decode_attn_fused(cache, q, zone_c=(k_buf, v_buf, counts_d))
    w = torch.zeros(cache.rows, cap, device=DEV)
    out_w, lse_w = stream_cache.decode_attn_fused(cache, q, zone_c=(k_buf, v_buf, counts_d), zone_c_weights=w)
    assert torch.equal(out, out_w) and torch.equal(lse, lse_w)
    q64, k64, v64 = (t2n(t).astype(np.float64) for t in (q, k_buf, v_buf))
    for r in range(rows_kv):
        n, at = int(counts[r]), slice(r * G, (r + 1) * G)
        parts = [(t2n(out_ab[at]), t2n(lse_ab[at]))]
        if n:
            s = q64[at] @ k64[r, :n].T / np.sqrt(128.0)
            m = s.max(1, keepdims=True)
            p = np.exp(s - m)
            parts.append((p @ v64[r, :n] / p.sum(1, keepdims=True), m[:, 0] + np.log(p.sum(1))))
        exp_out, exp_lse = lse_merge(parts)
        # 32-bit scores of a few units and sums of up to 300 weights: 2^-24 times some tens
        np.testing.assert_allclose(t2n(out[at]), exp_out, rtol=0, atol=2e-5)
        np.testing.assert_allclose(t2n(lse[at]), exp_lse, rtol=0, atol=2e-5)


@pytest.mark.parametrize("G,layers", [(4, 1), (4, 9), (8, 1)])
@pytest.mark.parametrize("row", [0, 7, 8, 64, 127, 130])
def test_own_token_with_and_without_block_scores(G, layers, row):
    """``append``: with block scores all heads share a workgroup, without them they do not."""
    require_gpu()
    cache = _cache(G, layers, 8, 5)
    rows_kv, cap, block = layers * 8, 131, 32
    g = torch.Generator().manual_seed(row)
    fill = torch.randn(rows_kv, cap, 256, generator=g).to(DEV)
    k, v = (torch.randn(rows_kv, 128, generator=g).half().to(DEV) for _ in range(2))
    q = torch.randn(cache.rows, 128, generator=g).half().to(DEV)
    ang = torch.rand(64, generator=g) * 6.28
    rope = (torch.cos(ang).half().to(DEV), torch.sin(ang).half().to(DEV))
    counts = torch.full((rows_kv,), row + 1, dtype=torch.int32, device=DEV)
    row_t = torch.full((1,), row, dtype=torch.int64, device=DEV)
    got = []
    for scored in (False, True):
        buf = fill.clone()
        buf[:, row] = float("nan")                                      # never read back
        kw = {}
        if scored:
            w = torch.zeros(cache.rows, cap, device=DEV)
            kw = dict(zone_c_weights=w, tail_scores=(torch.zeros(rows_kv, cap, device=DEV),
                                                     torch.zeros(rows_kv, block, device=DEV), None, block))
        out, lse = stream_cache.decode_attn_fused(cache, q, rope=rope, zone_c=(buf[:, :, :128], buf[:, :, 128:], counts),
                                                  append=(k, v, row_t), **kw)
        got.append((out, lse, buf))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert bool(torch.isfinite(got[0][0]).all()) and bool(torch.isfinite(got[0][2]).all())
    # the appended row read back by a later call gives the same result
    again = stream_cache.decode_attn_fused(cache, q, rope=rope, zone_c=(got[0][2][:, :, :128], got[0][2][:, :, 128:], counts))
    assert torch.equal(again[0], got[0][0]) and torch.equal(again[1], got[0][1])


def test_scores_of_minus_infinity_have_no_weight():
    require_gpu()
    cache = _cache(4, 1, 2, 3)
    g = torch.Generator().manual_seed(1)
    q = torch.rand(cache.rows, 128, generator=g).to(DEV) + 0.1          # positive: -inf keys score -inf
    k, v = (torch.randn(2, 80, 128, generator=g).to(DEV) for _ in range(2))
    keep = torch.zeros(80, dtype=torch.bool)
    keep[[3, 70]] = True
    k[:, ~keep] = -float("inf")
    out, lse = stream_cache.decode_attn_fused(cache, q, zone_c=(k, v))
    exp, exp_lse = stream_cache.decode_attn_fused(cache, q, zone_c=(k[:, keep].contiguous(), v[:, keep].contiguous()))
    torch.testing.assert_close(out, exp, rtol=0, atol=1e-6)
    torch.testing.assert_close(lse, exp_lse, rtol=0, atol=1e-6)


@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("layers,heads", [(1, 1), (1, 7), (1, 9), (3, 5), (7, 11), (13, 11), (67, 5)])
def test_same_bits_with_the_heads_apart_and_together(G, layers, heads):
    """The same cache with block scores (all heads of a unit in one workgroup) and without (one, two or
    all of them, by the number of units, here at numbers that are no multiple of eight): every unit is
    merged, with the same bits, and the weights are those of the softmax over the union."""
    require_gpu()
    cache = _cache(G, layers, heads, G + layers)
    n, cap, row = layers * heads, 140, 131
    g = torch.Generator().manual_seed(layers + G)
    counts = torch.tensor([COUNTS[i % 10] if i else row + 1 for i in range(n)], dtype=torch.int32).to(DEV)
    fill = torch.randn(n, cap, 256, generator=g).to(DEV)
    k, v = (torch.randn(n, 128, generator=g).half().to(DEV) for _ in range(2))
    q = torch.randn(cache.rows, 128, generator=g).half().to(DEV)
    row_t = torch.full((1,), row, dtype=torch.int64, device=DEV)
    got = []
    for scored in (True, False):
        buf, w = fill.clone(), torch.full((cache.rows, cap), float("nan"), device=DEV)
        out, lse = torch.full((cache.rows, 128), float("nan"), device=DEV), torch.full((cache.rows,), float("nan"), device=DEV)
        tail = (torch.zeros(n, cap, device=DEV), torch.zeros(n, 256, device=DEV), None, 256) if scored else None
        stream_cache.decode_attn_fused(cache, q, out, lse, zone_c=(buf[:, :, :128], buf[:, :, 128:], counts),
                                       append=(k, v, row_t), zone_c_weights=w, tail_scores=tail)
        got.append((out, lse, w.nan_to_num(nan=-1.0), buf))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    out, lse, w, buf = got[0]
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    s = torch.einsum("ugd,utd->ugt", q.double().view(n, G, 128), buf[:, :, :128].double()).view(cache.rows, cap) / 128 ** 0.5
    there = (torch.arange(cap, device=DEV)[None] < counts[:, None]).repeat_interleave(G, 0)
    exp = torch.where(there, torch.exp(s - lse.double()[:, None]), -1.0)
    # scores of a few units in 32 bits: a few 2^-24 of them, times weights of at most one
    torch.testing.assert_close(w.double(), exp, rtol=1e-5, atol=1e-7)
