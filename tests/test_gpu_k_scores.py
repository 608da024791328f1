"""K scores by exact int8 products against 64-bit sums over the same codes: channel counts around the 64 of
a block and the bytes of a row, tokens around the 256 of a tile and beyond what is resident at once, rows that
start anywhere, every number of query heads around the four of a product, queries of any size."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from rdkv_amd import k_kernel as kk
from tests.gpu_util import DEV, require_gpu, t2n

pytestmark = pytest.mark.gpu


def _layer(n2, n4, n8, H, T, G, seed, q_scale=1.0, odd_zero_points=False, unused=0):
    """Random packed K (``n2`` / ``n4`` padded to whole bytes, the last ``unused`` channels of every width with
    scale zero) and, per query head, q * scale and the centred codes in float64."""
    rng = np.random.default_rng(seed)
    counts = (n2, n4, n8)
    Dp = n2 + n4 + n8
    codes = [rng.integers(0, 1 << b, (H, T, n), dtype=np.uint8) for b, n in zip((2, 4, 8), counts)]
    scale = (rng.uniform(0.5, 2.0, (H, Dp)) * np.repeat([1.0, 0.2, 0.012], counts)).astype(np.float16)
    zp = np.stack([np.concatenate([rng.integers(0, 1 << b, n) for b, n in zip((2, 4, 8), counts)]) for _ in range(H)]).astype(np.float16)
    if odd_zero_points:
        zp += rng.choice([0.0, 0.25, 30.5, -7.0, 700.0], zp.shape).astype(np.float16)
    at = 0
    for n in counts:
        scale[:, max(at, at + n - unused):at + n] = 0
        at += n
    perm = rng.integers(0, 128, (H * G, Dp))
    q = (rng.standard_normal((H * G, 128)) * q_scale).astype(np.float32)
    n = n2 // 4
    k2 = sum(codes[0][..., i * n:(i + 1) * n] << (2 * i) for i in range(4)).astype(np.uint8)
    n = n4 // 2
    k4 = (codes[1][..., :n] | codes[1][..., n:] << 4).astype(np.uint8)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    layer = SimpleNamespace(
        K_ch_seg_bounds=counts, K_ch_scale=dev(scale[:, None]), K_ch_zp=dev(zp[:, None]), K_2bit=dev(k2) if n2 else None,
        K_4bit=dev(k4) if n4 else None, K_8bit=dev(codes[2]) if n8 else None, K_ch_perm_padded_idx_for_Q=dev(perm))
    terms = np.take_along_axis(q.astype(float), perm, axis=1).reshape(H, G, Dp) * scale[:, None].astype(float)
    centred = np.concatenate(codes, axis=2).astype(float) - zp[:, None].astype(float)
    return layer, q, terms, centred


def _check(got, terms, centred, counts):
    """Roundings of the sum and of the factor 1 / sqrt(128) (itself rounded), and of every term 30 bits against
    the head's largest (each times its width's power of two; the operands hold 46, of which the scales here, like each
    other, need no more: ``test_channels_far_below_the_largest``) with codes below 2^7.  Zero points outside a
    width's codes enter as an fp32 sum: 2^-20 of its magnitude."""
    exp = np.einsum("hgc,htc->hgt", terms, centred) / np.sqrt(128.0)
    sizes = np.abs(terms) * np.repeat([1 / 32, 1 / 8, 1.0], counts)
    tol = 4 * 2.0 ** -24 * np.abs(exp) + (sizes.max(axis=2) * terms.shape[2] * 2.0 ** -31 * 2.0 ** 9)[..., None]
    # (centred - its own codes) is the zero point: what of it lies outside 0 .. 2^b - 1 is the fp32 part
    odd = np.maximum(np.abs(centred).max(axis=1)[:, None] - np.repeat([3.0, 15.0, 255.0], counts), 0.0)
    tol = tol + ((np.abs(terms) * odd).sum(axis=2) * 2.0 ** -20)[..., None]
    err = np.abs(got.reshape(exp.shape) - exp)
    assert (err <= tol).all(), float((err / np.maximum(tol, 1e-300)).max())


@pytest.mark.parametrize("counts", [(4, 0, 0), (0, 2, 0), (0, 0, 1), (64, 0, 0), (68, 0, 0), (128, 0, 0), (0, 64, 0), (0, 66, 0), (0, 128, 0),
                                    (0, 0, 63), (0, 0, 64), (0, 0, 65), (0, 0, 128), (28, 38, 0), (20, 6, 41), (60, 62, 66), (128, 128, 20)])
@pytest.mark.parametrize("T,G", [(1, 4), (255, 1), (257, 5), (700, 9)])
def test_channel_counts(counts, T, G):
    require_gpu()
    layer, q, terms, centred = _layer(*counts, 2, T, G, seed=sum(counts) + T)
    out = torch.full((2 * G, T + 3), 7.0, device=DEV)
    kk.k_mixed_qk_dot_into(torch.from_numpy(q).to(DEV), layer, T, out[:, :T])
    _check(t2n(out[:, :T]), terms, centred, counts)
    assert bool((out[:, T:] == 7.0).all())


@pytest.mark.parametrize("H,T,dtype,G", [(2, 300000, torch.float16, 4), (8, 66000, torch.bfloat16, 8), (3, 90001, torch.float32, 2)])
def test_more_tiles_than_are_resident(H, T, dtype, G):
    require_gpu()
    layer, q, terms, centred = _layer(8, 6, 3, H, T, G, seed=T)
    qd = torch.from_numpy(q).to(dtype)
    q_np = qd.float().numpy()
    perm = t2n(layer.K_ch_perm_padded_idx_for_Q)
    terms = np.take_along_axis(q_np.astype(float), perm, axis=1).reshape(terms.shape) * t2n(layer.K_ch_scale).astype(float)
    _check(t2n(kk.k_mixed_qk_dot(qd.to(DEV), layer, T)), terms, centred, (8, 6, 3))


@pytest.mark.parametrize("counts", [(0, 0, 96), (0, 0, 128), (64, 64, 64), (128, 128, 128)])
@pytest.mark.parametrize("H,T,G", [(8, 33001, 8), (1, 270000, 4)])
def test_wide_rows_over_more_tiles_than_are_resident(counts, H, T, G):
    """Two tiles of up to 57 KB a workgroup; the last of them of 233 and 176 tokens."""
    require_gpu()
    layer, q, terms, centred = _layer(*counts, 1, T, G, seed=sum(counts))
    many = SimpleNamespace(**{k: v.expand(H, *v.shape[1:]).contiguous() if torch.is_tensor(v) and k != "K_ch_perm_padded_idx_for_Q"
                              else v for k, v in vars(layer).items()})
    many.K_ch_perm_padded_idx_for_Q = layer.K_ch_perm_padded_idx_for_Q.repeat(H, 1)
    got = t2n(kk.k_mixed_qk_dot(torch.from_numpy(q).repeat(H, 1).to(DEV), many, T)).reshape(H, G, T)
    _check(got[:1], terms, centred, counts)
    assert (got == got[:1]).all()


@pytest.mark.parametrize("q_scale", [1e-30, 1e-6, 1e6, 1e30])
def test_queries_of_any_size(q_scale):
    require_gpu()
    layer, q, terms, centred = _layer(20, 22, 9, 2, 500, 4, seed=5, q_scale=q_scale)
    _check(t2n(kk.k_mixed_qk_dot(torch.from_numpy(q).to(DEV), layer, 500)), terms, centred, (20, 22, 9))


@pytest.mark.parametrize("G", [4, 9])
@pytest.mark.parametrize("width", [2, 4, 8])
@pytest.mark.parametrize("extreme,n_ext,q_up", [(64, 1, 1), (512, 1, 8), (4096, 1, 8), (4096, 47, 1), (30000, 20, 8)])
def test_channels_far_below_the_largest(extreme, n_ext, q_up, width, G):
    """One token is extreme in some channels, which widens their scales; every other token lies at their zero
    points and its score is the small channels' alone.  Per token: the fp32 products q * scale (2^-24 of each), the
    join of the digits (2^-24 of the part below the upper two) and two roundings of the score; 2^-47 of the
    head's largest (times its width's power of two) for what lies below the last digit, per channel and code."""
    require_gpu()
    H, T, n = 2, 520, 64
    rng = np.random.default_rng(extreme + n_ext + width)
    k = rng.standard_normal((H, T, n))
    k[:, 0, :n_ext] *= extreme
    top = (1 << width) - 1
    lo, hi = k.min(axis=1, keepdims=True), k.max(axis=1, keepdims=True)
    scale = ((hi - lo) / top).astype(np.float16).astype(float)
    zp = np.clip(np.rint(-lo / scale), 0, top)
    codes = np.clip(np.rint(k / scale) + zp, 0, top).astype(np.uint8)
    counts = [0, 0, 0]
    counts[(2, 4, 8).index(width)] = n
    layer, q, _, _ = _layer(*counts, H, T, G, seed=3)
    perm = t2n(layer.K_ch_perm_padded_idx_for_Q)
    perm[:] = rng.permutation(128)[:n]
    q[:, perm[0, :n_ext]] *= q_up
    per, sub = 8 // width, n * width // 8
    rows = sum(codes[..., i * sub:(i + 1) * sub].astype(np.uint8) << (width * i) for i in range(per)).astype(np.uint8)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)   # noqa: E731
    setattr(layer, f"K_{width}bit", dev(rows))
    layer.K_ch_scale, layer.K_ch_zp = dev(scale.astype(np.float16)), dev(zp.astype(np.float16))
    layer.K_ch_perm_padded_idx_for_Q = dev(perm)
    got = t2n(kk.k_mixed_qk_dot(dev(q), layer, T)).astype(float).reshape(H, G, T)
    terms = np.take_along_axis(q.astype(float), perm, axis=1).reshape(H, G, n) * scale
    centred = codes.astype(float) - zp
    parts = np.einsum("hgc,htc->hgt", np.abs(terms), np.abs(centred)) / np.sqrt(128.0)
    exp = np.einsum("hgc,htc->hgt", terms, centred) / np.sqrt(128.0)
    below = np.abs(terms).max(axis=2) * n * 2.0 ** -47 * 255
    tol = 3 * 2.0 ** -24 * np.abs(exp) + 2 * 2.0 ** -24 * parts + below[..., None]
    err = np.abs(got - exp)
    assert (err <= tol).all(), float((err / tol).max())


def test_zero_points_outside_the_codes_and_unused_channels():
    require_gpu()
    for kw in ({"odd_zero_points": True}, {"unused": 7}, {"unused": 300}):
        layer, q, terms, centred = _layer(36, 24, 20, 3, 600, 4, seed=6, **kw)
        _check(t2n(kk.k_mixed_qk_dot(torch.from_numpy(q).to(DEV), layer, 600)), terms, centred, (36, 24, 20))


def test_a_query_that_is_not_finite_stays_in_its_head():
    require_gpu()
    layer, q, terms, centred = _layer(20, 22, 9, 2, 300, 4, seed=7)
    perm = t2n(layer.K_ch_perm_padded_idx_for_Q)
    q[1, perm[1, 3]], q[6, perm[6, 30]] = np.nan, np.inf
    got = t2n(kk.k_mixed_qk_dot(torch.from_numpy(q).to(DEV), layer, 300))
    assert not np.isfinite(got[[1, 6]]).any()
    keep = [0, 2, 3, 4, 5, 7]
    terms = np.where(np.isfinite(terms), terms, 0.0)
    exp = (np.einsum("hgc,htc->hgt", terms, centred) / np.sqrt(128.0)).reshape(8, 300)
    np.testing.assert_allclose(got[keep], exp[keep], rtol=2e-6, atol=1e-4)
