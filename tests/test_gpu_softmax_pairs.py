"""``trizone_attention`` over score rows whose softmax comes in pairs from the scores launch, against the three
separate launches (K scores, softmax over [old | new], V sum): tile and walk edges of the scores launch, every
width of its appended keys' workgroups, one to three launches of query heads, masks of every kind."""
import ctypes

import numpy as np
import pytest
import torch

from rdkv_amd import _lib, fast_decode, k_kernel, packing, triton_k_kernel as kk, v_kernel as vk
from tests.gpu_util import DEV, require_gpu, t2n

pytestmark = pytest.mark.gpu


def _layer(H, T, G, seed, kept=128):
    g = torch.Generator().manual_seed(seed)
    K, V = (torch.randn(1, H, T, 128, generator=g).half().to(DEV) for _ in range(2))
    v_bits = torch.tensor([2, 4, 8, 16])[torch.randint(0, 4, (H, T), generator=g)]
    k_bits = torch.tensor([2, 4, 8])[torch.randint(0, 3, (H, 128), generator=g)]
    k_bits[:, kept:] = 0
    layer, v16 = packing.pack_layer_per_head(K, V, v_bits, k_bits, G)
    return fast_decode._pre_squeeze_packed((layer,))[0], v16[0].contiguous()


def _separately(q, layer, v16, kn, vn, G):
    """The weights and the output through a launch for each part."""
    H_q, t_old, n = q.shape[0], int(layer.T_eff_k), kn.shape[1]
    w = torch.empty(H_q, t_old + n, device=DEV)
    kk.k_mixed_qk_dot_into(q, layer, t_old, w[:, :t_old])
    m = layer.softmax_mask
    ws = torch.empty(max(int(_lib.load().rdkv_softmax_rows_workspace_bytes(H_q)), 1), dtype=torch.uint8, device=DEV)
    _lib.check(_lib.load().rdkv_softmax_rows_new_keys(
        w.data_ptr(), w.stride(0), _lib.ptr(m), m.stride(0) if m is not None else 0, t_old, q.data_ptr(),
        _lib.DTYPE_CODE[q.dtype], q.stride(0), kn.data_ptr(), kn.stride(0), kn.stride(1), n, w.data_ptr(), w.stride(0),
        w[:, t_old:].data_ptr(), w.stride(0), H_q, H_q // G, ws.data_ptr(), ws.numel(), _lib.stream_of(q.device)))
    out = torch.empty(H_q, 128, device=DEV)
    vk._weighted_sum_with_new_zone(w[:, :t_old], layer, out, v16, layer.n_v16_per_head, int(layer.T_eff), w[:, t_old:], vn)
    return w, out


def _sum64(w, layer, v16, vn):
    """The weighted sum in 64 bits, over the packed values and the appended ones."""
    H, n = vn.shape[:2]
    T_v, G = int(layer.T_eff), w.shape[0] // H
    out = torch.empty(w.shape[0], 128, dtype=torch.float64, device=DEV)
    for h in range(H):
        V = torch.zeros(w.shape[1], 128, dtype=torch.float64, device=DEV)
        at = 0
        for t, bits, m in zip((layer.V_2bit, layer.V_4bit, layer.V_8bit), (2, 4, 8), layer.seg_bounds_per_head[h].tolist()):
            if m:
                codes = torch.cat([(t[h, :m].long() >> i) & ((1 << bits) - 1) for i in range(0, 8, bits)], dim=1)
                V[at:at + m] = (codes.double() - layer.V_zp[h, at:at + m].double()) * layer.V_scale[h, at:at + m].double()
            at += m
        n16 = int(layer.n_v16_per_head[h])
        V[T_v:T_v + n16] = v16[h, :n16].double()
        V[w.shape[1] - n:] = vn[h].double()
        out[h * G:(h + 1) * G] = w[h * G:(h + 1) * G].double() @ V
    return out


def _pairs(monkeypatch):
    """The number of pairs of every call."""
    seen, load = [], _lib.load()

    class Seen:
        def __getattr__(self, name):
            fn = getattr(load, name)
            if name != "rdkv_attn_scores":
                return fn

            def call(*args):
                rc = fn(*args)
                seen.append(ctypes.c_int.from_address(args[-2]).value)
                return rc
            return call
    monkeypatch.setattr(_lib, "load", lambda: Seen())
    return seen


@pytest.mark.parametrize("H,T,G,n_new,kept,dtype,mask", [
    (1, 1, 1, 1, 128, torch.float32, "own"), (2, 255, 4, 63, 128, torch.float16, "own"), (2, 256, 3, 64, 70, torch.bfloat16, None),
    (3, 257, 5, 65, 128, torch.float16, "odd"), (2, 511, 8, 129, 64, torch.bfloat16, "shared"), (2, 515, 9, 8192, 128, torch.float16, "own"),
    (1, 1030, 16, 8193, 40, torch.float16, "own"), (1, 40, 2, 20000, 128, torch.float32, "odd"),
    # several tiles of a workgroup, its appended keys in front
    (16, 33000, 4, 64, 64, torch.float16, "own"), (16, 33001, 8, 100, 64, torch.float16, "odd"), (64, 5000, 1, 700, 128, torch.bfloat16, "own"),
    (1, 70001, 4, 257, 128, torch.float16, "own")])
def test_rows_in_pairs(monkeypatch, H, T, G, n_new, kept, dtype, mask):
    require_gpu()
    g = torch.Generator().manual_seed(T + n_new)
    layer, v16 = _layer(H, T, G, 11, kept)
    q = torch.randn(H * G, 128, generator=g).to(dtype).to(DEV)
    kn, vn = (torch.randn(H, n_new, 128, generator=g).to(DEV) for _ in range(2))
    t_old = int(layer.T_eff_k)
    if mask is None:
        layer.softmax_mask = None
    elif mask != "own":            # any additive mask, rows at any float or one row for every head
        rows = torch.randn(1 if mask == "shared" else H * G, t_old + 3, generator=g).to(DEV)
        rows[rows > 1.5] = -torch.inf
        layer.softmax_mask = rows[:, 1:1 + t_old].expand(H * G, t_old) if mask == "shared" else rows[:, 3:]
    w, exp = _separately(q, layer, v16, kn, vn, G)
    seen = _pairs(monkeypatch)
    buf = torch.full((H * G, t_old + n_new + 5), 7.0, device=DEV)
    out = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, G, scores_buf=buf)
    again = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, G)
    assert len(seen) == 2 and min(seen) > 0
    # the same fp32 scores; sums of exponentials in another order, an exponential's last bits
    np.testing.assert_allclose(t2n(buf)[:, :t_old + n_new], t2n(w), rtol=1e-5, atol=1e-9)
    assert float((buf[:, t_old + n_new:] - 7.0).abs().max()) == 0
    np.testing.assert_allclose(t2n(out), t2n(exp), rtol=0, atol=1e-5)
    assert torch.equal(out, again)
    # The weights that the sum forms itself: an exponential's last bits (1.2e-7 of the weights in the 2-norm) and some
    # sixty roundings of the sum (sqrt(64) * 2^-25 = 2.4e-7), twice, and rows whose terms cancel to half.
    exact = _sum64(w, layer, v16, vn)
    err = (out.double() - exact).norm(dim=1) / exact.norm(dim=1)
    assert float(err.max()) < 1.5e-6, float(err.max())


def test_wide_keys_come_in_pairs_at_any_length(monkeypatch):
    """One KV head whose tiles are resident at once only in part, every channel 8 bits wide."""
    require_gpu()
    g = torch.Generator().manual_seed(8)
    T, n_new = 300_001, 900
    K, V = (torch.randn(1, 1, T, 128, generator=g).half().to(DEV) for _ in range(2))
    layer, v16 = packing.pack_layer_per_head(K, V, torch.tensor([2, 4, 8, 16])[torch.randint(0, 4, (1, T), generator=g)],
                                             torch.full((1, 128), 8), 4)
    layer, v16 = fast_decode._pre_squeeze_packed((layer,))[0], v16[0].contiguous()
    q = torch.randn(4, 128, generator=g).to(DEV)
    kn, vn = (torch.randn(1, n_new, 128, generator=g).to(DEV) for _ in range(2))
    w, exp = _separately(q, layer, v16, kn, vn, 4)
    seen = _pairs(monkeypatch)
    buf = torch.empty(4, T + n_new, device=DEV)
    out = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, 4, scores_buf=buf)
    assert len(seen) == 1 and seen[0] > 0
    np.testing.assert_allclose(t2n(buf), t2n(w), rtol=1e-5, atol=1e-12)
    err = (out.double() - exp.double()).norm() / exp.double().norm()      # (sums of the same fp32 terms in another order)
    assert float(err) < 2e-6, float(err)


@pytest.mark.parametrize("G", [4, 8])
def test_wide_rows_under_capture(G):
    """Rows whose two tiles take more than 64 KB of LDS, recorded and replayed with other queries in between."""
    require_gpu()
    g = torch.Generator().manual_seed(9)
    H, T, n_new = 2, 140_000, 30
    K, V = (torch.randn(1, H, T, 128, generator=g).half().to(DEV) for _ in range(2))
    layer, v16 = packing.pack_layer_per_head(K, V, torch.tensor([2, 4, 8, 16])[torch.randint(0, 4, (H, T), generator=g)],
                                             torch.full((H, 128), 8), G)
    layer, v16 = fast_decode._pre_squeeze_packed((layer,))[0], v16[0].contiguous()
    q = torch.randn(H * G, 128, generator=g).to(DEV)
    kn, vn = (torch.randn(H, n_new, 128, generator=g).to(DEV) for _ in range(2))
    buf, out = torch.empty(H * G, int(layer.T_eff_k) + n_new, device=DEV), torch.empty(H * G, 128, device=DEV)
    call = lambda: fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, G, scores_buf=buf, out=out)   # noqa: E731
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seed in range(3):
        q.copy_(torch.randn(H * G, 128, generator=g))
        call()
        torch.cuda.synchronize()
        exp, w = out.clone(), buf.clone()
        out.zero_(), buf.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, exp) and torch.equal(buf, w)


@pytest.mark.parametrize("G", [4, 6])
@pytest.mark.parametrize("what", ["row -inf", "all -inf", "new inf", "nan", "inf", "lowest", "tile -inf", "tile nan"])
def test_masked_and_infinite_rows(what, G):
    """Rows of -inf, infinities and NaN end in the same places as by the separate launches."""
    require_gpu()
    g = torch.Generator().manual_seed(5)
    layer, v16 = _layer(2, 1500, G, 3)
    t_old = int(layer.T_eff_k)
    q = torch.randn(2 * G, 128, generator=g).to(DEV)
    kn, vn = (torch.randn(2, 9, 128, generator=g).to(DEV) for _ in range(2))
    m = layer.softmax_mask.clone() if layer.softmax_mask is not None else torch.zeros(2 * G, t_old, device=DEV)
    if what in ("row -inf", "all -inf"):
        m[1] = -torch.inf
    if what in ("all -inf", "new inf"):      # (the key's infinity meets a query of either sign: +-inf or NaN scores)
        kn[0, :, 0] = torch.inf
    if what == "nan":
        m[2, 300] = torch.nan
    if what == "inf":
        m[2, 300] = torch.inf
    if what == "lowest":
        m[1] = torch.finfo(torch.float32).min
        m[2, ::2] = torch.finfo(torch.float32).min
    if what == "tile -inf":
        m[:, 256:512] = -torch.inf
    if what == "tile nan":
        m[3, 256:512] = -torch.inf
        m[3, 400] = torch.nan
    layer.softmax_mask = m
    w, exp = _separately(q, layer, v16, kn, vn, G)
    buf = torch.empty(2 * G, t_old + 9, device=DEV)
    out = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, G, scores_buf=buf)
    np.testing.assert_allclose(t2n(buf), t2n(w), rtol=1e-5, atol=1e-9)
    np.testing.assert_allclose(t2n(out), t2n(exp), rtol=1e-6, atol=1e-5)


def test_other_forms_take_the_separate_softmax(monkeypatch):
    """Strided K rows, no kept channels, diagnosis: the same results without pairs."""
    require_gpu()
    g = torch.Generator().manual_seed(6)
    layer, v16 = _layer(2, 700, 4, 4)
    q, kn, vn = torch.randn(8, 128, generator=g).to(DEV), *(torch.randn(2, 30, 128, generator=g).to(DEV) for _ in range(2))
    call = lambda pl: fast_decode.trizone_attention(q, pl, v16, pl.n_v16_per_head, kn, vn, 4)   # noqa: E731
    exp = call(layer)
    seen = _pairs(monkeypatch)
    wide = torch.zeros(2, layer.K_8bit.shape[1], layer.K_8bit.shape[2] + 16, dtype=torch.uint8, device=DEV)
    wide[:, :, :layer.K_8bit.shape[2]] = layer.K_8bit
    dense, layer.K_8bit = layer.K_8bit, wide[:, :, :layer.K_8bit.shape[2]]
    np.testing.assert_allclose(t2n(call(layer)), t2n(exp), rtol=0, atol=1e-5)
    layer.K_8bit = dense
    assert seen == [0]
    monkeypatch.setattr(k_kernel, "_DIAG_ENABLED", True)
    np.testing.assert_allclose(t2n(call(layer)), t2n(exp), rtol=0, atol=1e-5)
    assert seen == [0]
