"""Dequantize a packed cache back to dense fp16 K/V (API of obkv_accel/trizone_decompress.py).

This is the "dequantize-then-attend" route of the reference: K via ``unpack_k_mixed``, zone-A
V per head via ``unpack_v_segment``, zone-B V from ``new_v_only``, plus per-head additive
masks for the padded stripe.  All dequantization runs in the HIP kernels.
"""
from __future__ import annotations

from typing import List, Optional, Tuple

import torch
from torch import Tensor

from . import _lib
from .packing import PackedKVLayer, TriZoneCache, _check_k_counts, _int32_on, _unpack_k_enqueue, unpack_v_segment


def _unpack_v_zone_a(pl: PackedKVLayer) -> Tensor:
    """Shared layout: dequantized 2/4/8-bit V segments concatenated in packed order
    (trizone_decompress.py:43-83) -> [1,H_kv,T_v,D] fp16."""
    N = pl.seg_bounds
    T_v = int(pl.T_eff)
    assert sum(N) == T_v, f"V seg_bounds {tuple(N)} must sum to T_v={T_v}"
    H_kv = pl.V_scale.shape[1]
    parts, off = [], 0
    for n, seg, bits in zip(N, (pl.V_2bit, pl.V_4bit, pl.V_8bit), (2, 4, 8)):
        if n > 0 and seg is not None:
            parts.append(unpack_v_segment(seg, pl.V_scale[:, :, off:off + n], pl.V_zp[:, :, off:off + n], bits))
            off += n
    if not parts:
        return torch.empty(1, H_kv, 0, 1, dtype=torch.float16, device=pl.V_scale.device)
    return torch.cat(parts, dim=2)


def _is_perhead_layout(pl: PackedKVLayer) -> bool:
    return pl.seg_bounds_per_head is not None


def _unpack_v_enqueue(pl: PackedKVLayer, zone_b: Optional[Tensor], head_dim: int, words=None) -> tuple:
    """The stripe's dense V, ``zone_b`` rows behind it, in one launch; and the per-head counts, yet to be checked
    (``_check_v_counts``): on the device, [H, 3] by class and [H] in all, or, as the launch read them into the
    next 4 H of ``words``, H."""
    max_T_v = int(pl.T_eff)
    H_kv = pl.V_scale.shape[1]
    # everything the kernel indexes by head, class row and token, before it gets the addresses
    dev = _lib.require_device(pl.V_scale, pl.V_zp, pl.V_2bit, pl.V_4bit, pl.V_8bit, zone_b)
    segs = []
    for seg, bits in zip((pl.V_2bit, pl.V_4bit, pl.V_8bit), (2, 4, 8)):
        if seg is None or seg.numel() == 0:
            segs.append((None, 0, 0))
            continue
        width = head_dim * bits // 8
        if seg.dim() != 4 or seg.shape[1] < H_kv or seg.shape[3] != width:
            raise RuntimeError(f"V segment {tuple(seg.shape)} for {H_kv} heads, rows of {width} bytes")
        seg = seg if seg.stride(3) == 1 and seg.stride(2) == width else seg.contiguous()
        segs.append((seg, seg.stride(1), int(seg.shape[2])))
    sc, zp = pl.V_scale, pl.V_zp
    rows = min(max_T_v, sum(m for _, _, m in segs))      # of a head, at most: the kernel clamps its counts to these
    exact = sc.shape == zp.shape == (1, H_kv, max_T_v, 1)
    if not exact and any(t.dim() < 3 or t.shape[1] < H_kv or t.shape[2] < rows for t in (sc, zp)):
        raise RuntimeError(f"V scales / zero points {tuple(sc.shape)}, {tuple(zp.shape)} for {H_kv} heads of {rows} tokens")
    if rows and not (exact and sc.stride(2) == 1 and zp.stride() == sc.stride()):
        sc, zp = (t[:1, :H_kv, :rows].contiguous() for t in (sc, zp))
    counts, totals = pl.seg_bounds_per_head, pl.T_eff_per_head
    if counts.shape != (H_kv, 3) or totals.shape != (H_kv,):
        if counts.dim() != 2 or counts.shape[0] < H_kv or counts.shape[1] != 3 or totals.numel() < H_kv:
            raise RuntimeError(f"V counts {tuple(counts.shape)}, {tuple(totals.shape)} for {H_kv} heads")
        counts, totals = counts[:H_kv], totals.reshape(-1)[:H_kv]
    counts, totals = _int32_on(dev, counts), _int32_on(dev, totals)
    n16 = 0 if zone_b is None else int(zone_b.shape[2])
    out = torch.empty(1, H_kv, max_T_v + n16, head_dim, dtype=torch.float16, device=dev)
    if zone_b is not None and not (zone_b.stride(3) == 1 and zone_b.stride(2) == head_dim):
        zone_b = zone_b.contiguous()
    (V2, v2h, m2), (V4, v4h, m4), (V8, v8h, m8) = segs
    args = (_lib.ptr(V2), v2h, _lib.ptr(V4), v4h, _lib.ptr(V8), v8h, _lib.ptr(sc), _lib.ptr(zp), sc.stride(1),
            counts.data_ptr(), m2, m4, m8, max_T_v, _lib.ptr(zone_b), zone_b.stride(1) if n16 else 0, n16, H_kv, head_dim,
            _lib.ptr(out))
    if words is not None and max_T_v + n16 > 0:
        _lib.check(_lib.load().rdkv_unpack_layer_v_words(*args, totals.data_ptr(), words.take(4 * H_kv), words.tag,
                                                         _lib.stream_of(dev)))
        return out, H_kv
    _lib.check(_lib.load().rdkv_unpack_layer_v(*args, _lib.stream_of(dev)))
    return out, counts, totals


def _check_v_counts(pl: PackedKVLayer, counts, totals) -> None:
    segs = (pl.V_2bit, pl.V_4bit, pl.V_8bit)
    rows = [0 if seg is None else int(seg.shape[2]) for seg in segs]
    classes = list(zip(*counts))
    if list(map(sum, counts)) == totals and max(totals) <= pl.T_eff and min(map(min, classes)) >= 0 \
            and all(max(c) <= r for c, r in zip(classes, rows)):
        return
    for h, (row, n) in enumerate(zip(counts, totals)):
        assert sum(row) == n, f"head {h}: seg_bounds_per_head {row} != T_eff_per_head {n}"
        # rows that are there: tokens of a class without a tensor are left out, a negative count has none
        there = [max(c, 0) if seg is not None else 0 for c, seg in zip(row, segs)]
        assert all(c <= r for c, r in zip(there, rows)), f"head {h}: {row} tokens in V segments of {rows}"
        assert sum(there) <= pl.T_eff, f"head {h}: {row} tokens in a stripe of {pl.T_eff}"


def _unpack_v_perhead(pl: PackedKVLayer, *, head_dim: int) -> Tensor:
    """Stripe layout: [1,H_kv,max_T_v,D] fp16, head h filled on [0,T_v_h), zeros after
    (trizone_decompress.py:91-144)."""
    if int(pl.T_eff) == 0:
        return torch.zeros(1, pl.V_scale.shape[1], 0, head_dim, dtype=torch.float16, device=pl.V_scale.device)
    out, *found = _unpack_v_enqueue(pl, None, head_dim)
    _read_checks([(_check_v_counts, pl, found)])
    return out


def _words_of(dev: torch.device, words: dict, heads: int):
    """The words of this call on ``dev``, for launches over ``heads`` heads in all (K and V); None where the
    counts come back as tensors (no device, a capture)."""
    if dev.type != "cuda" or torch.cuda.is_current_stream_capturing():
        return None
    if dev not in words:
        words[dev] = _lib.host_words(dev, 4 * heads), []
    return words[dev][0]


def _read_checks(unchecked, words: Optional[dict] = None) -> None:
    """Calls every (check, layer, device tensors) with the tensors' values as lists: one read per device.
    ``words``: by device, what its launches filled and (check, layer, heads) in the order they took theirs."""
    for dev, (filled, entries) in (words or {}).items():
        flat, at = filled.read(dev), 0
        for check, pl, heads in entries:
            rows = [flat[i:i + 4] for i in range(at, at + 4 * heads, 4)]
            at += 4 * heads
            if check is _check_v_counts:
                check(pl, [row[:3] for row in rows], [row[3] for row in rows])
            else:
                check(pl, rows)
    by_device: dict = {}
    for entry in unchecked:
        by_device.setdefault(entry[2][0].device, []).append(entry)
    for entries in by_device.values():
        flat, at = _lib.download(torch.cat([t.reshape(-1) for _, _, ts in entries for t in ts])).tolist(), 0
        for check, pl, ts in entries:
            values = []
            for t in ts:
                end, width = at + t.numel(), t.shape[-1]
                values.append([flat[i:i + width] for i in range(at, end, width)] if t.dim() == 2 else flat[at:end])
                at = end
            check(pl, *values)


def unpack_trizone_to_past_kv(dual_cache: TriZoneCache, *, head_dim: int,
                              device: Optional[torch.device] = None, dtype: torch.dtype = torch.float16,
                              return_masks: bool = False, H_q: Optional[int] = None,
                              max_new_tokens: int = 0, mask_dtype: torch.dtype = torch.float16):
    """TriZoneCache -> tuple of dense (K, V) [1,H_kv,T_eff_k,D] per layer; with
    ``return_masks`` also per-layer [1,H_q,1,T_eff_k+max_new_tokens] additive masks (None for
    shared-layout layers) (trizone_decompress.py:185-333)."""
    past_kv: List[Tuple[Tensor, Tensor]] = []
    masks: List[Optional[Tensor]] = []
    unchecked = []        # (check, layer, per-head counts the launches below read)
    words: dict = {}      # the same from launches that send them to the host
    heads = sum(int(t.shape[1]) for pl in dual_cache.packed for t in (pl.K_ch_scale, pl.V_scale) if t is not None)
    for i, pl in enumerate(dual_cache.packed):
        to = _words_of(pl.K_ch_scale.device, words, heads) if pl.K_ch_scale is not None else None
        zone_b = dual_cache.new_v_only[i] if i < len(dual_cache.new_v_only) else None
        pair = mask = None
        n = 0 if to is None else int(pl.K_ch_scale.shape[1])
        # (words were counted by the scales there are: a layer without V scales has none for V)
        if to is not None and _lib.native is not None and _is_perhead_layout(pl) and to.used + 8 * n <= to.size:
            used = to.used
            if return_masks and mask_dtype == torch.float16 and device is None:
                mask = pl.softmax_mask
            pair = _lib.native.dense_layer(pl.__dict__, zone_b if mask is None else (zone_b, mask, max_new_tokens), head_dim,
                                           to.take(4 * n), to.take(4 * n), to.tag, _lib.stream_of(pl.K_ch_scale.device))
            if pair is None:
                to.used = used
            else:
                K_full, V_full = pair[:2]
                words[pl.K_ch_scale.device][1].extend(((_check_k_counts, pl, n), (_check_v_counts, pl, n)))
        if pair is None:
            K_full, k_check = _unpack_k_enqueue(pl, head_dim, to)
            if isinstance(k_check, int):
                words[pl.K_ch_scale.device][1].append((_check_k_counts, pl, k_check))
            elif k_check is not None:
                unchecked.append((_check_k_counts, pl, (k_check,)))
        if pair is not None:
            pass
        elif _is_perhead_layout(pl):
            rows_b = None
            if int(pl.n_v16) > 0:
                assert zone_b is not None, f"layer {i}: max_n_v16={pl.n_v16} > 0 but new_v_only is None"
                rows_b = zone_b
            if int(pl.T_eff) == 0:
                V_full = rows_b if rows_b is not None else _unpack_v_perhead(pl, head_dim=head_dim)
            else:
                joined = rows_b is not None and rows_b.dtype == torch.float16 and rows_b.shape[:2] == pl.V_scale.shape[:2] \
                    and rows_b.shape[3] == head_dim and rows_b.device == pl.V_scale.device
                V_full, *v_counts = _unpack_v_enqueue(pl, rows_b if joined else None, head_dim,
                                                      _words_of(pl.V_scale.device, words, heads))
                if isinstance(v_counts[0], int):
                    words[pl.V_scale.device][1].append((_check_v_counts, pl, v_counts[0]))
                else:
                    unchecked.append((_check_v_counts, pl, v_counts))
                if rows_b is not None and not joined:
                    V_full = torch.cat([V_full, rows_b], dim=2)
        else:
            zone_a = _unpack_v_zone_a(pl)
            if zone_b is not None and zone_b.shape[2] > 0:
                V_full = zone_b if zone_a.shape[2] == 0 else torch.cat([zone_a, zone_b], dim=2)
            else:
                V_full = zone_a
            if V_full.shape[2] == 0 and V_full.shape[3] != head_dim:
                V_full = torch.empty(1, K_full.shape[1], 0, head_dim, dtype=V_full.dtype, device=V_full.device)
        assert K_full.shape[2] == V_full.shape[2], (
            f"layer {i}: K T-dim {K_full.shape[2]} != V T-dim {V_full.shape[2]}")
        assert K_full.shape[3] == head_dim and V_full.shape[3] == head_dim
        if device is not None:
            K_full, V_full = K_full.to(device), V_full.to(device)
        past_kv.append((K_full.to(dtype).contiguous(), V_full.to(dtype).contiguous()))
        if return_masks:
            if _is_perhead_layout(pl) and pl.softmax_mask is not None:
                m = pl.softmax_mask
                if H_q is not None:
                    assert H_q == int(m.shape[0]), f"layer {i}: caller H_q={H_q} != softmax_mask H_q={m.shape[0]}"
                if mask is not None and pair is not None:      # (left the layer's launch)
                    masks.append(pair[2])
                    continue
                tgt = device if device is not None else m.device
                m4 = m.to(device=tgt, dtype=mask_dtype).view(1, m.shape[0], 1, m.shape[1])
                if max_new_tokens > 0:
                    m4 = torch.cat([m4, torch.zeros(1, m.shape[0], 1, max_new_tokens, dtype=mask_dtype,
                                                    device=tgt)], dim=-1)
                masks.append(m4.contiguous())
            else:
                masks.append(None)
    _read_checks(unchecked, words)        # (behind the launches, which clamp what they follow)
    return (tuple(past_kv), masks) if return_masks else tuple(past_kv)
