"""``trizone_attention``: the appended tokens' scores formed inside the softmax launch and their values
added inside the V launch, against float64 over the packed zones' own K scores and V sums: token
counts around the eight keys of a wavefront and the 128 of a workgroup's pass, rows of every softmax
form, appended rows that are views or start at an odd float, no packed tokens at all."""
import numpy as np
import pytest
import torch

from rdkv_amd import fast_decode, packing, triton_k_kernel as kk, triton_v_kernel as vk
from tests.gpu_util import DEV, require_gpu, t2n

pytestmark = pytest.mark.gpu


def _layer(H, T, G, seed):
    g = torch.Generator().manual_seed(seed)
    K, V = (torch.randn(1, H, T, 128, generator=g).half().to(DEV) for _ in range(2))
    v_bits = torch.tensor([2, 4, 8, 16])[torch.randint(0, 4, (H, T), generator=g)]
    k_bits = torch.tensor([0, 2, 4, 8])[torch.randint(0, 4, (H, 128), generator=g)]
    k_bits[:, :3] = torch.tensor([2, 4, 8])
    layer, v16 = packing.pack_layer_per_head(K, V, v_bits, k_bits, G)
    return fast_decode._pre_squeeze_packed((layer,))[0], v16[0].contiguous()


@pytest.mark.parametrize("H,T,G,n_new,dtype,form", [
    (2, 3, 4, 1, torch.float16, "dense"), (2, 300, 4, 7, torch.bfloat16, "dense"), (3, 1200, 1, 8, torch.float32, "dense"),
    (2, 1200, 2, 9, torch.float16, "kv"), (2, 9000, 5, 127, torch.float16, "odd"), (1, 9000, 8, 128, torch.bfloat16, "dense"),
    (2, 34000, 4, 129, torch.float16, "kv"), (2, 34001, 9, 257, torch.float16, "dense"), (1, 66001, 4, 1, torch.float16, "dense"),
    (1, 66001, 4, 1030, torch.float16, "odd"), (2, 0, 4, 33, torch.float16, "dense"),
    # around the length from which the scores are a launch of their own, and its 256 keys per workgroup
    (2, 300, 4, 1023, torch.float16, "dense"), (2, 300, 4, 1024, torch.float16, "odd"), (3, 9000, 5, 1025, torch.bfloat16, "kv"),
    (1, 34000, 8, 1281, torch.float32, "dense"), (2, 0, 1, 1279, torch.float16, "dense"), (2, 1200, 9, 5000, torch.float16, "kv")])
def test_trizone_attention_new_zone(H, T, G, n_new, dtype, form):
    require_gpu()
    g = torch.Generator().manual_seed(T + n_new)
    wide = torch.randn(H, n_new, 260, generator=g).to(DEV)
    k_new, v_new = {"dense": (wide[:, :, :128].contiguous(), wide[:, :, 128:256].contiguous()),
                    "kv": (wide[:, :, :128], wide[:, :, 128:256]), "odd": (wide[:, :, 1:129], wide[:, :, 130:258])}[form]
    q = torch.randn(H * G, 128, generator=g).to(dtype).to(DEV)
    layer, v16 = _layer(H, max(T, 5), G, 7)
    if T == 0:
        layer.T_eff = layer.T_eff_k = 0
    t_v = int(layer.T_eff)
    t_old = int(layer.T_eff_k) if layer.T_eff_k > 0 else t_v
    buf = torch.empty(H * G, -(-(t_old + n_new) // 4) * 4, device=DEV)
    out = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, k_new, v_new, G, scores_buf=buf)
    q64 = t2n(q.float()).astype(np.float64).reshape(H, G, 128)
    k64, v64 = (t2n(t).astype(np.float64) for t in (k_new, v_new))
    s = (q64 @ k64.transpose(0, 2, 1) / np.sqrt(128.0)).reshape(H * G, n_new)
    if t_old:
        a = t2n(kk.k_mixed_qk_dot(q, layer, t_old)).astype(np.float64)
        if layer.softmax_mask is not None:
            a = a + t2n(layer.softmax_mask)
        s = np.concatenate([a, s], axis=1)
    w = np.exp(s - s.max(1, keepdims=True))
    w /= w.sum(1, keepdims=True)
    exp = (w[:, t_old:].reshape(H, G, n_new) @ v64).reshape(H * G, 128)
    if t_old:
        w_old = torch.from_numpy(w[:, :t_old].astype(np.float32)).to(DEV)
        exp = exp + t2n(vk.v_dequant_weighted_sum_dispatch(w_old, layer, V16=v16, n_v16_per_head=layer.n_v16_per_head,
                                                           max_T_v=t_v))
    # fp32 scores, weights and sums: a few 2^-24 of values of order one
    np.testing.assert_allclose(t2n(out), exp, rtol=0, atol=1e-5)
    np.testing.assert_allclose(t2n(buf)[:, :t_old + n_new], w, rtol=1e-4, atol=1e-7)   # the buffer holds the weights


def test_buffers_and_rows_that_do_not_fit_are_refused():
    require_gpu()
    layer, v16 = _layer(2, 40, 4, 1)
    q, kv = torch.randn(8, 128, device=DEV), torch.randn(2, 6, 128, device=DEV)
    args = (q, layer, v16, layer.n_v16_per_head)
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv, kv, 4, scores_buf=torch.empty(8, 45, device=DEV))
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv.half(), kv, 4)
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv, kv[:, :5], 4)
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv, kv, 4, scores_buf=torch.empty(9, 48, device=DEV))
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv, kv, 4, scores_buf=torch.empty(8, 48, device=DEV, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(torch.randn(10, 128, device=DEV), *args[1:], kv, kv, 4)
    for rows in (4, 16):
        with pytest.raises(RuntimeError):
            fast_decode.trizone_attention(*args, kv, kv, 4, out=torch.empty(rows, 128, device=DEV))
    with pytest.raises(RuntimeError):                                    # the layer has two KV heads, not four or one
        fast_decode.trizone_attention(*args, kv.repeat(2, 1, 1), kv.repeat(2, 1, 1), 2)
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv[:1], kv[:1], 8)
    with pytest.raises(RuntimeError):
        fast_decode.trizone_attention(*args, kv, kv, 4, scores_buf=torch.empty(8, 48))


@pytest.mark.parametrize("T,n_new", [(0, 9), (0, 1500), (50, 9), (50, 1500), (9000, 300), (9000, 1500)])
def test_score_buffers_of_any_alignment(T, n_new):
    """Rows at odd floats take the element-wise softmax: the same weights and output to rounding."""
    require_gpu()
    g = torch.Generator().manual_seed(T + n_new)
    layer, v16 = _layer(2, max(T, 5), 4, 3)
    if T == 0:
        layer.T_eff = layer.T_eff_k = 0
    t_old = int(layer.T_eff_k) if layer.T_eff_k > 0 else int(layer.T_eff)
    q, kn, vn = (torch.randn(*s, generator=g).to(DEV) for s in ((8, 128), (2, n_new, 128), (2, n_new, 128)))
    got = []
    for shift in (0, 1, 3):
        row = -(-(t_old + n_new) // 4) * 4 + shift
        buf = torch.empty(8, row + shift, device=DEV)[:, shift:]
        out = fast_decode.trizone_attention(q, layer, v16, layer.n_v16_per_head, kn, vn, 4, scores_buf=buf)
        got.append((out, buf[:, :t_old + n_new]))
    for out, w in got[1:]:
        torch.testing.assert_close(out, got[0][0], rtol=0, atol=1e-5)
        torch.testing.assert_close(w, got[0][1], rtol=1e-4, atol=1e-7)
