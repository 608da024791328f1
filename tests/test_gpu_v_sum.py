"""The V weighted sum on the matrix cores against 64-bit sums over the same codes: class counts around the
four tokens of a lane group and the 32 / 64 of a step, rows of fewer than four columns, every number of
query heads around the four of a workgroup, weights over fp32's whole range, values that are not finite."""
import numpy as np
import pytest
import torch

from rdkv_amd import v_kernel as vk
from tests.gpu_util import DEV, require_gpu, t2n

pytestmark = pytest.mark.gpu


def _case(counts, n16, G, seed, pad=0):
    """Random packed V of two heads (the second with fewer tokens) and what it stands for in float64."""
    rng = np.random.default_rng(seed)
    H = 2
    seg = np.array([counts, [c // 2 for c in counts]], dtype=np.int32)
    n16h = np.array([n16, max(n16 - 1, 0)], dtype=np.int32)
    T_v = int(sum(counts)) + pad
    codes = {b: rng.integers(0, 1 << b, (H, max(n, 1), 128), dtype=np.uint8) for b, n in zip((2, 4, 8), counts)}
    scale = rng.uniform(0.01, 2.0, (H, max(T_v, 1), 1)).astype(np.float16)
    zp = rng.integers(0, 4, (H, max(T_v, 1), 1)).astype(np.float16)
    v16 = rng.standard_normal((H, max(n16, 1), 128)).astype(np.float16)
    packed = {2: codes[2][..., :32] | codes[2][..., 32:64] << 2 | codes[2][..., 64:96] << 4 | codes[2][..., 96:] << 6,
              4: codes[4][..., :64] | codes[4][..., 64:] << 4, 8: codes[8]}
    dev = {b: torch.from_numpy(packed[b]).to(DEV) if n else None for b, n in zip((2, 4, 8), counts)}
    dense = np.zeros((H, T_v + n16, 128))
    for h in range(H):
        at = 0
        for b, n in zip((2, 4, 8), seg[h]):
            dense[h, at:at + n] = (codes[b][h, :n].astype(float) - zp[h, at:at + n]) * scale[h, at:at + n].astype(float)
            at += n
        dense[h, T_v:T_v + n16h[h]] = v16[h, :n16h[h]]
    args = (dev[2], dev[4], dev[8], torch.from_numpy(scale).to(DEV), torch.from_numpy(zp).to(DEV))
    kw = dict(V16=torch.from_numpy(v16).to(DEV) if n16 else None, n_v16_per_head=torch.from_numpy(n16h).to(DEV), max_T_v=T_v)
    return args, torch.from_numpy(seg).to(DEV), tuple(counts), kw, dense, v16


def _run(w, case):
    args, seg, counts, kw, _, _ = case
    out = torch.full((w.shape[0], 128), 7.0, device=DEV)
    vk.v_dequant_weighted_sum_unified_perhead_into(w, *args, seg, counts, out, **kw)
    return t2n(out).astype(float)


def _close(got, w, dense, G):
    """fp32 weights, codes and sums: 2^-20 of the sum of the products' magnitudes covers the rounding of
    a product (2^-22) and of the sums of this many of them in a few dozen parts."""
    w = w.astype(float).reshape(dense.shape[0], G, -1)
    exp, size = w @ dense, np.abs(w) @ (np.abs(dense) + 4.0)      # (codes and zero points enter apart: up to 4 more)
    err = np.abs(got.reshape(exp.shape) - exp)
    assert (err <= 2.0 ** -20 * size + 1e-38).all(), float((err / np.maximum(size, 1e-38)).max())


@pytest.mark.parametrize("G", [1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("counts,n16", [((1, 0, 0), 0), ((3, 0, 0), 0), ((2, 1, 0), 2), ((0, 0, 0), 1), ((0, 0, 0), 3), ((2, 2, 0), 5),
                                        ((63, 64, 65), 33), ((4, 129, 1), 32), ((0, 67, 130), 0), ((9000, 1, 33), 31)])
def test_class_counts(counts, n16, G):
    require_gpu()
    case = _case(counts, n16, G, seed=G + n16)
    w = np.random.default_rng(5).random((2 * G, sum(counts) + n16)).astype(np.float32)
    _close(_run(torch.from_numpy(w).to(DEV), case), w, case[4], G)


def test_rows_of_any_alignment():
    require_gpu()
    case = _case((70, 67, 129), 35, 4, seed=3, pad=3)
    w = np.random.default_rng(5).random((8, 70 + 67 + 129 + 3 + 35)).astype(np.float32)
    for shift in (0, 1, 2, 3):
        wide = torch.zeros(8, w.shape[1] + 5, device=DEV)[:, shift:shift + w.shape[1]]
        wide.copy_(torch.from_numpy(w))
        _close(_run(wide, case), w, case[4], 4)


@pytest.mark.parametrize("lo,hi", [(-140, -115), (-126, 30), (-60, 60), (60, 110), (-3, 0)])
def test_weights_of_any_size(lo, hi):
    """Weights that grow from token to token (every step rescales), fall, or lie anywhere in fp32."""
    require_gpu()
    case = _case((300, 500, 700), 400, 4, seed=4)
    n = 1900
    ramp = np.linspace(lo, hi, n)
    rng = np.random.default_rng(6)
    w = np.stack([2.0 ** e for e in (ramp, ramp[::-1], rng.permutation(ramp), np.full(n, lo), np.full(n, hi), -ramp.clip(-90, 90),
                                     rng.permutation(ramp), ramp)]).astype(np.float32) * rng.choice([-1, 1], (8, n)).astype(np.float32)
    _close(_run(torch.from_numpy(w).to(DEV), case), w, case[4], 4)


@pytest.mark.parametrize("width", [2, 4, 8, 16])
def test_a_weight_is_used_with_all_its_bits(width):
    """One token counts, of value 1 as code and zero point on the two sides of the middle: its weight is the result."""
    require_gpu()
    G, n = 4, 40
    counts = {2: (n, 0, 0), 4: (0, n, 0), 8: (0, 0, n), 16: (0, 0, 0)}[width]
    args, seg, counts, kw, dense, _ = _case(counts, n if width == 16 else 0, G, seed=1)
    seg[1] = seg[0]
    kw["n_v16_per_head"] = torch.tensor([n if width == 16 else 0] * 2, dtype=torch.int32, device=DEV)
    if width == 16:
        kw["V16"][:] = 1.0
    else:
        codes = {2: 0xAA, 4: 0x88, 8: 0x81}[width]           # code 2, 8, 129 in every field
        args[(2, 4, 8).index(width)].fill_(codes)
        args[3].fill_(1.0)
        args[4].fill_({2: 1.0, 4: 7.0, 8: 128.0}[width])
    w = np.zeros((2 * G, n), dtype=np.float32)
    rng = np.random.default_rng(width)
    for trial in range(20):
        w[:] = 0
        at = rng.integers(0, n, 2 * G)
        value = (rng.random(2 * G) * 2.0 ** rng.uniform(-60, 20, 2 * G)).astype(np.float32)
        w[np.arange(2 * G), at] = value
        got = _run(torch.from_numpy(w).to(DEV), (args, seg, counts, kw, dense, None))
        assert np.array_equal(got, np.repeat(value[:, None].astype(float), 128, axis=1))


def test_small_weights_beside_one_of_no_value():
    """A sink: the weight of one fp16 row is 2^24 .. 2^40 times the others', its values are zero.  fp32 products and sums
    of the others: 2^-20 of the products' magnitudes."""
    require_gpu()
    case = _case((0, 0, 0), 3000, 4, seed=2)
    dense, v16 = case[4], case[5]
    v16[:, 700] = 0
    dense[:, 700] = 0
    case[3]["V16"] = torch.from_numpy(v16).to(DEV)
    rng = np.random.default_rng(3)
    for e in (24, 32, 40):
        w = (rng.random((8, 3000)) * 2.0 ** -e).astype(np.float32)
        w[:, 700] = 1.0
        got = _run(torch.from_numpy(w).to(DEV), case).reshape(2, 4, 128)
        w8 = w.astype(float).reshape(2, 4, -1)
        exp, size = w8 @ dense, w8 @ np.abs(dense)
        assert (np.abs(got - exp) <= 2.0 ** -20 * size).all(), float((np.abs(got - exp) / size).max())


@pytest.mark.parametrize("width", [2, 4, 8, 16])
def test_many_tokens_of_like_weight(width):
    """The error grows as roundings do, without a bias: about 64 additions on a result's way, each off by 2^-25 of a
    partial sum no larger than the results' own size, make sqrt(64) * 2^-25 in the 2-norm; twice that is allowed."""
    require_gpu()
    n = 16000
    counts = {2: (n, 0, 0), 4: (0, n, 0), 8: (0, 0, n), 16: (0, 0, 0)}[width]
    args, seg, counts, kw, dense, v16 = _case(counts, n if width == 16 else 0, 4, seed=9)
    if width < 16:         # values around zero, as the quantizer leaves them
        zp = torch.randint(0, 2, args[4].shape, generator=torch.Generator().manual_seed(4)).half().to(DEV) + (1 << (width - 1)) - 1
        scale = t2n(args[3]).astype(float)
        dense = dense + (t2n(args[4]).astype(float) - t2n(zp).astype(float)) * scale
        dense[1, n // 2:] = 0
        args = (*args[:4], zp)
    w = np.random.default_rng(5).uniform(0.5, 1.5, (8, n)).astype(np.float32)
    got = _run(torch.from_numpy(w).to(DEV), (args, seg, counts, kw, dense, v16)).reshape(2, 4, 128)
    w8 = w.astype(float).reshape(2, 4, -1)
    exp = w8 @ dense
    err = np.linalg.norm(got - exp) / np.linalg.norm(exp)
    assert err < 2 * 8 * 2.0 ** -25, err


def test_infinities_and_nan_stay_where_they_are():
    require_gpu()
    case = _case((100, 100, 100), 200, 4, seed=8)
    v16 = case[5].copy()
    v16[0, 7, 5], v16[0, 9, 6], v16[1, 3, 100] = np.inf, -np.inf, np.nan
    case[3]["V16"] = torch.from_numpy(v16).to(DEV)
    rng = np.random.default_rng(7)
    w = rng.uniform(0.1, 1.0, (8, 500)).astype(np.float32)
    got = _run(torch.from_numpy(w).to(DEV), case).reshape(2, 4, 128)
    assert (got[0, :, 5] == np.inf).all() and (got[0, :, 6] == -np.inf).all() and np.isnan(got[1, :, 100]).all()
    keep = np.ones((2, 128), dtype=bool)
    keep[0, 5] = keep[0, 6] = keep[1, 100] = False
    assert np.isfinite(got[np.broadcast_to(keep[:, None], got.shape)]).all()
    for bad in (np.inf, -np.inf):               # (infinity times a code less infinity times a zero point)
        w[2, 50] = bad
        got = _run(torch.from_numpy(w).to(DEV), case).reshape(2, 4, 128)
        assert np.isnan(got[0, 2]).all() and np.isfinite(got[0, [0, 1, 3]][:, 10:]).all()
    w[2, 50], w[5, 320] = np.nan, np.inf        # head 0: a quantized token; head 1: an fp16 one
    got = _run(torch.from_numpy(w).to(DEV), case).reshape(2, 4, 128)
    assert np.isnan(got[0, 2]).all() and np.isfinite(got[0, [0, 1, 3]][:, 10:]).all()
    sign = np.sign(case[5][1, 20].astype(float))
    assert np.array_equal(got[1, 1, :100], np.where(sign[:100] == 0, np.nan, sign[:100] * np.inf))
    assert np.isfinite(got[1, [0, 2, 3]][:, :100]).all()
