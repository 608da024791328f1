"""The framework's work as sized cases: what a program that serves with it calls, and how large.

A case is a dict of plain values.  ``prepare`` makes what such a program holds before the call
(packed caches, queries, allocations, a model), ``run`` is one pass through the public entry
points, ``work`` the bytes and operations of that pass that no implementation can leave out.

Kinds:

* ``step``   - one layer's whole decode attention, as a sequential model loop calls it: rotary
  embedding, packed prompt, the generated tokens with this step's own row appended.
* ``model``  - every layer's packed prompt attention in one call (independent layers / sequences).
* ``batch``  - sequences of differing lengths served together, each with its own generated tokens.
* ``calls``  - one layer through the reference-layout kernels: K scores, softmax, V sum, new tokens.
* ``select`` - prefill of one layer: bit allocation by the knapsack, then quantize + pack.
* ``stream`` - prefill packing of several layers straight into the streaming cache.
* ``dense``  - a packed cache dequantized back to dense K / V with its padding masks.
* ``loop``   - greedy decoding of a few tokens with a model of the 8B layer shape.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rdkv_amd import fast_decode, knapsack_solver, obkv_fast, packing, stream_cache, trizone_decompress

D = 128
DEV = "cuda:0"
KEPT = 64                                             # kept K channels per head (half of them)
V_WIDTHS = (0, 2, 4, 8, 16)
# allocation rules: V fractions over V_WIDTHS, K channel counts (2, 4, 8 bit); None: drawn per head
ALLOC = {
    "mixed": (None, None),
    "even": ((0.2, 0.2, 0.3, 0.2, 0.1), (16, 32, 16)),
    "low": ((0.15, 0.40, 0.30, 0.10, 0.05), (26, 38, 0)),
}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
HIDDEN, INTERMEDIATE, VOCAB = 4096, 14336, 128256     # the decode loop's model (8B layer shape)


def listed():
    return [
        # a short chat prompt, one layer: launches and latency
        {"name": "step_4k", "kind": "step", "context": 4096, "layers": 1, "heads": 8, "group": 4, "tail": 17,
         "alloc": "even", "dtype": "f16"},
        # a document prompt late in a long answer: the generated tokens weigh as much as the prompt
        {"name": "step_32k_long_answer", "kind": "step", "context": 32768, "layers": 1, "heads": 8, "group": 4,
         "tail": 700, "alloc": "mixed", "dtype": "bf16"},
        # the long-context, wide-group model (8 query heads per KV head), ragged prompt length
        {"name": "step_120k_group8", "kind": "step", "context": 120001, "layers": 1, "heads": 8, "group": 8,
         "tail": 200, "alloc": "mixed", "dtype": "f16"},
        # the headline: all 32 layers' packed prompt at 32k
        {"name": "model_32k", "kind": "model", "context": 32768, "layers": 32, "heads": 8, "group": 4, "tail": 0,
         "alloc": "mixed", "dtype": "f16"},
        # serving: 12 sequences of 16k..64k, four of their layers, generated tokens of differing numbers
        {"name": "batch_12_ragged", "kind": "batch", "context": 40960, "layers": 4, "sequences": 12, "heads": 8,
         "group": 4, "tail": 300, "alloc": "mixed", "dtype": "f16"},
        # a program that keeps the reference layout (in-place slots, its own loop) at a document length
        {"name": "calls_32k", "kind": "calls", "context": 32768, "layers": 1, "heads": 8, "group": 4, "tail": 48,
         "alloc": "mixed", "dtype": "f16"},
        # the same at a long, low-bit context
        {"name": "calls_128k_low_bit", "kind": "calls", "context": 131072, "layers": 1, "heads": 8, "group": 4,
         "tail": 257, "alloc": "low", "dtype": "f16"},
        # prefill of one layer of a short prompt
        {"name": "select_4k", "kind": "select", "context": 4096, "layers": 1, "heads": 8, "group": 4, "budget": 1024},
        # prefill of one layer of a document (an odd length)
        {"name": "select_31k", "kind": "select", "context": 31337, "layers": 1, "heads": 8, "group": 4, "budget": 2048},
        # prefill packing for serving: four layers at 32k into the streaming cache
        {"name": "stream_4x32k", "kind": "stream", "context": 32768, "layers": 4, "heads": 8, "group": 4,
         "alloc": "mixed"},
        # the dequantize-then-attend route over two layers
        {"name": "dense_2x16k", "kind": "dense", "context": 16384, "layers": 2, "heads": 8, "group": 4,
         "alloc": "mixed"},
        # decoding itself: eight tokens, four layers of the 8B shape and its LM head, 32k prompt
        {"name": "loop_4_layers_32k", "kind": "loop", "context": 32768, "layers": 4, "heads": 8, "group": 4,
         "tail": 8, "alloc": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "model", "batch", "calls", "calls", "select", "select", "stream",
                       "dense", "loop"])
    case = {"kind": kind, "context": _log_int(rng, 1024, 131072), "layers": 1, "heads": rng.choice([2, 4, 8, 8, 8]),
            "group": rng.choice([1, 2, 4, 4, 4, 5, 7, 8, 8])}
    if kind in ("step", "model", "batch", "calls"):
        case["tail"] = 0 if kind == "model" else _log_int(rng, 1, 1024)
        case["dtype"] = rng.choice(["f16", "bf16"])
    if kind == "model":
        case["context"] = _log_int(rng, 2048, 65536)
        case["layers"] = rng.randint(2, 16)
    elif kind == "batch":
        case["context"] = _log_int(rng, 2048, 40960)
        case["layers"] = rng.randint(1, 4)
        case["sequences"] = rng.randint(2, 12)
        case["tail"] = _log_int(rng, 2, 512)
    elif kind == "select":
        case["budget"] = max(64, int(case["context"] * rng.choice([1 / 16, 1 / 8, 1 / 4])))
    elif kind == "stream":
        case["context"] = _log_int(rng, 1024, 65536)
        case["layers"] = rng.randint(1, 4)
    elif kind == "dense":
        case["context"] = _log_int(rng, 1024, 65536)
        case["layers"] = rng.randint(1, 2)
    elif kind == "loop":
        case.update(context=_log_int(rng, 1024, 32768), layers=rng.randint(1, 4), heads=8, group=4,
                    tail=rng.randint(2, 8))
    if kind != "select":
        case["alloc"] = rng.choice(["mixed", "mixed", "even", "low"])
    return case


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed((seed * 1_000_003 + stream) % (1 << 62))


def _contexts(case):
    """The prompt length of every packed layer of a case."""
    if case["kind"] != "batch":
        return [case["context"]] * case["layers"]
    lengths = np.random.default_rng(case["context"]).uniform(0.4, 1.6, case["sequences"]) * case["context"]
    return [int(n) for n in np.repeat(lengths, case["layers"])]


def _tails(case):
    """The generated tokens of every sequence of a ``batch`` case."""
    return np.random.default_rng(case["context"] + 1).integers(1, case["tail"] + 1, case["sequences"])


def _sizes(case):
    """What fixes the shapes of a case's packed tensors: per layer and head the V class counts over
    V_WIDTHS and the K channel counts (2, 4, 8 bit).  They are the case's own, the same for every
    seed; which tokens and channels fall into a class, and all values, come from the seed."""
    contexts = _contexts(case)
    rng = np.random.default_rng([case["context"], case["layers"], case["heads"], len(contexts)])
    v_fracs, k_counts = ALLOC[case["alloc"]]
    out = []
    for context in contexts:
        v, k = [], []
        for _ in range(case["heads"]):
            n = np.floor((np.asarray(v_fracs) if v_fracs is not None else rng.dirichlet(np.ones(5))) * context)
            n[0] += context - n.sum()
            v.append(n.astype(np.int64))
            k.append(np.asarray(k_counts) if k_counts is not None else rng.multinomial(KEPT, rng.dirichlet(np.ones(3))))
        out.append((np.stack(v), np.stack(k)))
    return out


def _allocation(case, context, sizes, rng, gen):
    """Widths of one layer as the allocator hands them over: v_bits [H, context] and k_bits [H, D]
    (int64), and the four outlier channels of every head (always kept)."""
    H = case["heads"]
    cum = np.cumsum(sizes[0], axis=1)[:, :4]
    k_bits = np.zeros((H, D), dtype=np.int64)
    outliers = np.zeros((H, 4), dtype=np.int64)
    for h in range(H):
        channels = rng.permutation(D)
        outliers[h] = channels[:4]
        kept = rng.permutation(channels[:int(sizes[1][h].sum())])
        k_bits[h, kept] = np.repeat([2, 4, 8], sizes[1][h])
    # the importance ranking of the tokens is random: least important evicted, most important fp16
    position = torch.arange(context, device=DEV)
    cls = (position.view(1, 1, -1) >= torch.from_numpy(cum).to(DEV).unsqueeze(2)).sum(dim=1)
    ranked = torch.tensor(V_WIDTHS, device=DEV)[cls]
    order = torch.rand(H, context, generator=gen, device=DEV).argsort(dim=1)
    v_bits = torch.empty_like(ranked).scatter_(1, order, ranked)
    return v_bits, torch.from_numpy(k_bits).to(DEV), torch.from_numpy(outliers).to(DEV)


def _keys_values(case, context, outliers, gen):
    """fp16 K (four outlier channels per head, eight times as large) and V of one layer."""
    H = case["heads"]
    K = torch.randn(1, H, context, D, generator=gen, device=DEV)
    scale = torch.ones(H, D, device=DEV).scatter_(1, outliers, 8.0)
    K = K.mul_(scale.view(1, H, 1, D)).half()
    V = torch.randn(1, H, context, D, generator=gen, device=DEV).half()
    return K, V


def _entries(case, seed):
    rng = np.random.default_rng(seed)
    gen = _gen(seed, 1)
    out = []
    for context, sizes in zip(_contexts(case), _sizes(case)):
        v_bits, k_bits, outliers = _allocation(case, context, sizes, rng, gen)
        K, V = _keys_values(case, context, outliers, gen)
        out.append((K, V, v_bits, k_bits))
    return out


def _packed(case, seed):
    entries = _entries(case, seed)
    packed = packing.pack_layers_per_head([e[0] for e in entries], [e[1] for e in entries],
                                          torch.stack([e[2] for e in entries]), torch.stack([e[3] for e in entries]),
                                          case["group"])
    return packed


def _rope(position, dtype):
    inv = 1.0 / (500000.0 ** (torch.arange(0, D // 2, device=DEV, dtype=torch.float32) * 2 / D))
    angle = inv * float(position)
    return angle.cos().to(dtype), angle.sin().to(dtype)


class _Norm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.variance_epsilon = 1e-5


class _Linear(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.bias = None


class _Rotary(torch.nn.Module):
    def forward(self, x, position_ids):
        inv = 1.0 / (500000.0 ** (torch.arange(0, D, 2, device=x.device, dtype=torch.float32) / D))
        angle = position_ids.float().unsqueeze(-1) * inv
        angle = torch.cat([angle, angle], dim=-1)
        return angle.cos().to(x.dtype), angle.sin().to(x.dtype)


class _Config:
    def __init__(self, case):
        self.num_attention_heads = case["heads"] * case["group"]
        self.num_key_value_heads = case["heads"]
        self.head_dim = D
        self.hidden_size = HIDDEN


class _Model(torch.nn.Module):
    """A model of the 8B layer shape with random fp16 weights.  The LM head holds the embedding rows
    in another order, so that a next token stands out as it does in a trained model."""

    def __init__(self, case, gen):
        super().__init__()
        self.config = _Config(case)
        q_dim, kv_dim = case["heads"] * case["group"] * D, case["heads"] * D

        def weight(n, k):
            return _Linear(torch.randn(n, k, generator=gen, device=DEV, dtype=torch.float16).mul_(0.02))

        def norm():
            return _Norm(1 + 0.1 * torch.randn(HIDDEN, generator=gen, device=DEV, dtype=torch.float16))

        self.model = torch.nn.Module()
        self.model.layers = torch.nn.ModuleList()
        for _ in range(case["layers"]):
            layer = torch.nn.Module()
            layer.self_attn, layer.mlp = torch.nn.Module(), torch.nn.Module()
            layer.self_attn.q_proj, layer.self_attn.o_proj = weight(q_dim, HIDDEN), weight(HIDDEN, q_dim)
            layer.self_attn.k_proj, layer.self_attn.v_proj = weight(kv_dim, HIDDEN), weight(kv_dim, HIDDEN)
            layer.mlp.gate_proj, layer.mlp.up_proj = weight(INTERMEDIATE, HIDDEN), weight(INTERMEDIATE, HIDDEN)
            layer.mlp.down_proj = weight(HIDDEN, INTERMEDIATE)
            layer.input_layernorm, layer.post_attention_layernorm = norm(), norm()
            self.model.layers.append(layer)
        self.model.norm = norm()
        self.model.rotary_emb = _Rotary()
        table = torch.randn(VOCAB, HIDDEN, generator=gen, device=DEV, dtype=torch.float16)
        self.model.embed_tokens = torch.nn.Embedding(VOCAB, HIDDEN, _weight=table, _freeze=True)
        self.lm_head = _Linear(table[torch.randperm(VOCAB, generator=gen, device=DEV)] * 0.02)


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed, 2)
    H, G, rows = case["heads"], case["group"], case["heads"] * case["group"]

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=gen, device=DEV).to(dtype)

    s = {"case": case}
    if kind == "step":
        dtype, tail = DTYPES[case["dtype"]], case["tail"]
        cache = stream_cache.build_stream_cache_from_kv(_entries(case, seed), G)
        # the zone C buffer of a loop that may generate up to 1024 tokens: K | V side by side
        buf = normal(H, 1024, 2 * D)
        s.update(cache=cache, q=normal(rows, D, dtype=dtype), k=normal(H, D, dtype=dtype), v=normal(H, D, dtype=dtype),
                 rope=_rope(case["context"] + tail - 1, dtype), buf=buf,
                 counts=torch.full((H,), tail, dtype=torch.int32, device=DEV),
                 row=torch.full((1,), tail - 1, dtype=torch.int64, device=DEV),
                 out=torch.empty(rows, D, device=DEV), lse=torch.empty(rows, device=DEV))
    elif kind == "model":
        cache = stream_cache.build_stream_cache_from_kv(_entries(case, seed), G)
        s.update(cache=cache, q=normal(cache.rows, D, dtype=DTYPES[case["dtype"]]),
                 out=torch.empty(cache.rows, D, device=DEV), lse=torch.empty(cache.rows, device=DEV))
    elif kind == "batch":
        tails = np.repeat(_tails(case), case["layers"] * H)
        cache = stream_cache.build_stream_cache_from_kv(_entries(case, seed), G)
        n = len(tails)
        s.update(cache=cache, q=normal(cache.rows, D, dtype=DTYPES[case["dtype"]]),
                 zone_c=(normal(n, case["tail"], D), normal(n, case["tail"], D),
                         torch.from_numpy(tails.astype(np.int32)).to(DEV)),
                 out=torch.empty(cache.rows, D, device=DEV), lse=torch.empty(cache.rows, device=DEV))
    elif kind == "calls":
        layer, v16 = _packed(case, seed)[0]
        layer = fast_decode._pre_squeeze_packed((layer,))[0]
        tail = case["tail"]
        t_old = int(layer.T_eff_k) if layer.T_eff_k > 0 else int(layer.T_eff)
        s.update(layer=layer, v16=v16[0].contiguous() if v16 is not None else None,
                 q=normal(rows, D, dtype=DTYPES[case["dtype"]]), k_new=normal(H, tail, D), v_new=normal(H, tail, D),
                 scores=torch.empty(rows, -(-(t_old + tail) // 64) * 64, device=DEV), out=torch.empty(rows, D, device=DEV))
    elif kind == "select":
        context = case["context"]
        outliers = torch.rand(H, D, generator=gen, device=DEV).argsort(dim=1)[:, :4]
        K, V = _keys_values(case, context, outliers, gen)
        # Attention mass and channel energy, log-normal.  The allocation they lead to sizes the outputs, so
        # the scores are the case's up to what leaves those sizes alone: the seed turns the heads after
        # the first around, and scales everything by a power of two.
        rng = np.random.default_rng([context, H, case["budget"]])
        turned = [0] + [1 + (h + seed) % (H - 1) for h in range(H - 1)]
        scale = 2.0 ** (seed % 7)
        tokens = np.exp(rng.standard_normal((H, context)) * 1.5 + 2.0)[turned] * scale
        channels = np.exp(rng.standard_normal((H, D)))[turned] * scale
        s.update(K=K, V=V, tokens=torch.from_numpy(tokens.astype(np.float32)).to(DEV),
                 channels=torch.from_numpy(channels.astype(np.float32)).to(DEV),
                 k_options=torch.tensor([0.0, 2.0, 4.0, 8.0]))
    elif kind == "stream":
        s.update(entries=_entries(case, seed))
    elif kind == "dense":
        packed = _packed(case, seed)
        n = case["layers"]
        s.update(cache=packing.TriZoneCache(tuple(p for p, _ in packed), [v for _, v in packed], [None] * n, [None] * n,
                                            case["context"]))
    elif kind == "loop":
        packed = _packed(case, seed)
        n = case["layers"]
        s.update(model=_Model(case, gen), first=normal(VOCAB),
                 cache=packing.TriZoneCache(tuple(p for p, _ in packed), [v for _, v in packed], [None] * n, [None] * n,
                                            case["context"]))
    else:
        raise ValueError(kind)
    return s


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
_LAYER_TENSORS = ("K_2bit", "K_4bit", "K_8bit", "K_ch_scale", "K_ch_zp", "V_2bit", "V_4bit", "V_8bit", "V_scale", "V_zp",
                  "sort_idx", "seg_bounds_per_head", "T_eff_per_head", "softmax_mask", "K_ch_sort_idx_per_head",
                  "K_ch_perm_padded_idx_per_head", "K_ch_seg_bounds_per_head", "K_ch_perm_padded_idx_for_Q",
                  "T_eff_k_per_head", "n_v16_per_head", "allocation_v_bits", "allocation_k_bits")


def run(s):
    case = s["case"]
    kind, G = case["kind"], case["group"]
    if kind == "step":
        buf = s["buf"]
        k_buf, v_buf = buf[:, :, :D], buf[:, :, D:]
        out, lse = stream_cache.decode_attn_fused(s["cache"], s["q"], out=s["out"], lse=s["lse"], rope=s["rope"],
                                                  zone_c=(k_buf, v_buf, s["counts"]), append=(s["k"], s["v"], s["row"]))
        return {"out": out, "lse": lse, "appended": buf}
    if kind == "model":
        return stream_cache.decode_attn_fused(s["cache"], s["q"], out=s["out"], lse=s["lse"])
    if kind == "batch":
        return stream_cache.decode_attn_fused(s["cache"], s["q"], out=s["out"], lse=s["lse"], zone_c=s["zone_c"])
    if kind == "calls":
        return fast_decode.trizone_attention(s["q"], s["layer"], s["v16"], s["layer"].n_v16_per_head, s["k_new"],
                                             s["v_new"], G, scores_buf=s["scores"], out=s["out"])
    if kind == "select":
        layer, v16, _ = obkv_fast._perhead_select_and_pack(
            s["K"], s["V"], s["tokens"], s["channels"], gqa_factor=G, token_budget=case["budget"], k_budget_ratio=0.5,
            obs_window=32, pool_kernel_size=7, pool_padding="reflect", v_bit_options=None, k_bit_options=s["k_options"],
            eps_V=knapsack_solver.DEFAULT_EPSILON_V, eps_K=knapsack_solver.DEFAULT_EPSILON_K,
            retain_allocation_metadata=True)
        return {"v16": v16, **{name: getattr(layer, name) for name in _LAYER_TENSORS}}
    if kind == "stream":
        cache = stream_cache.build_stream_cache_from_kv(s["entries"], G)
        # (a blob ends in 256 bytes of slack that loads may touch and nothing writes)
        return {"scales": cache.unit_scale_max, "blobs": [b[:b.numel() - 256] for b in cache.blobs]}
    if kind == "dense":
        return trizone_decompress.unpack_trizone_to_past_kv(s["cache"], head_dim=D, return_masks=True,
                                                            H_q=case["heads"] * G)
    logits = []
    tokens = fast_decode.greedy_decode_fast(
        s["model"], s["cache"], s["first"], case["tail"], [], DEV, case["context"],
        logits_observer=lambda step, row, token, is_eos: logits.append(row))
    return {"tokens": tokens, "logits": logits[1:]}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    kind, H, G, context, layers = case["kind"], case["heads"], case["group"], case["context"], case["layers"]
    if kind == "select":
        # K, V and the scores once; the packed layer at the allocator's budgets, and its widths
        read = 2 * context * H * D * 2 + 4 * context * H
        written = 2 * case["budget"] * H * D * 2 + context * H * 2
        return {"bytes": read + written, "flops": 4 * context * H * D}
    # the packed layers: codes, scales and zero points, fp16 rows; tokens kept, per layer and head
    v = np.stack([n[0] for n in _sizes(case)]).astype(float)
    k = np.stack([n[1] for n in _sizes(case)]).astype(float)
    kept = v[:, :, 1:].sum(axis=2)
    packed = float((kept * (k @ [0.25, 0.5, 1.0]) + 4 * k.sum(axis=2) + v[:, :, 1:] @ [36, 68, 132, 256]).sum())
    kept, prompt = float(kept.sum()), sum(_contexts(case)) * H
    if kind == "stream":
        return {"bytes": 2 * prompt * D * 2 + prompt + packed, "flops": 4 * prompt * D}
    if kind == "dense":
        return {"bytes": packed + kept * (2 * D * 2 + G * 2), "flops": 4 * kept * D}
    tokens = float(_tails(case).sum()) if kind == "batch" else case["tail"] / 2 if kind == "loop" else case["tail"]
    new = H * layers * tokens                             # generated tokens attended over (a loop's: on average)
    rows = v.shape[0] * H * G
    attention = {"bytes": packed + new * 2 * D * 4 + rows * D * 6, "flops": G * (kept + new) * 4 * D}
    if kind != "loop":
        return attention
    weights = layers * HIDDEN * (2 * H * G * D + 2 * H * D + 3 * INTERMEDIATE) + VOCAB * HIDDEN
    return {"bytes": case["tail"] * (attention["bytes"] + 2 * weights),
            "flops": case["tail"] * (attention["flops"] + 2 * weights)}


def tolerance(case):
    """Four times the distance, on the listed cases, to the same attention over the packed values in
    64 bits: 2-norm 2e-4..8.4e-4 for the streaming kernel (its softmax weights enter the matrix cores
    as fp16), largest difference 2.9e-3; under 9e-7 and 5.4e-6 for the reference-layout kernels
    (fp32 throughout).  The loop against the same model in fp32: 1.6e-3 and 7.1e-3 on the logits, the
    same tokens.  Packing, allocation and dequantization are exact."""
    kind = case["kind"]
    if kind in ("select", "stream", "dense"):
        return "exact"
    if kind == "calls":
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "loop":
        return {"rel": 6e-3, "max": 0.03}
    return {"rel": 3.5e-3, "max": 0.012}
