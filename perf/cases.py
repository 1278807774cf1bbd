"""What a user of bitfield attention has it do, as measurable cases through the public entry points.

Kinds of pass (``case["kind"]``):

* ``train``    one attention layer of a training step: ``bitfield_attn_func`` and the gradients of q, k, v.  The flag
               cache is cleared first, as a model's forward does for every batch.
* ``bias``     the same with an additive per-head, per-key bias (ALiBi: slope times key position).
* ``masked``   a training step's layer with a materialized bool mask, ``flash_attn_func(q, k, v, mask=mask)``.
* ``shard``    one rank's layer of a context-parallel training step (zigzag split of the sequence): forward with index
               tensors, backward accumulated into fp32 gradients.
* ``prefill``  the prompt of a generating model through the attention-interface adapter, no gradients.
* ``decode``   one generated token per sequence through the same adapter: a single query against the key / value cache.

Sequences hold text and modality segments; the lengths and head counts are those of this repository's benchmark
workloads and tests, or ordinary ones between them.
"""

import math
import random

import numpy as np
import torch

from cornstarch_amd.kernel.attention import flash_attn_func
from cornstarch_amd.kernel.bitfield_attention import (
    BitfieldUtils,
    _bitfield_attn_backward,
    _bitfield_attn_forward,
    bitfield_attn_func,
)
from cornstarch_amd.kernel.interface import bitfield_attention_forward

# segments: how many modality segments a sequence holds, of seg_min..seg_max tokens, spread over `modalities` kinds;
# pad: padding tokens at the end of every second sequence of the batch
_TEXT = {"segments": 0, "seg_min": 1, "seg_max": 1, "modalities": 1, "pad": 0}


def _case(kind, B, S, Hq, Hkv, D, dtype, **more):
    return {"kind": kind, "B": B, "S": S, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype, **_TEXT, **more}


def listed():
    named = {
        # The smallest calls: short prompts of a small model, the sizes of the parity tests.  Latency and launches.
        "train_short": _case("train", 2, 283, 6, 2, 64, "fp16", segments=2, seg_min=20, seg_max=80, modalities=2),
        # A batch of ordinary fine-tuning samples, padded to an odd common length, grouped kv heads.
        "train_padded_batch": _case("train", 4, 1537, 32, 8, 128, "bf16", segments=2, seg_min=196, seg_max=400,
                                    modalities=2, pad=210),
        # A head dimension between the native ones (vision and language models with 80 or 96).
        "train_head_dim_96": _case("train", 2, 2003, 16, 16, 96, "fp16", segments=3, seg_min=100, seg_max=400, modalities=3),
        # Packed vision-encoder batch: head dim 64, no grouping, one to six segments a sequence (workload C4).
        "train_encoder_batch": _case("train", 8, 4096, 16, 16, 64, "bf16", segments=4, seg_min=256, seg_max=1024, modalities=8),
        # The headline configuration: 8192 tokens, four images of 576 tokens (workload C2).
        "train_8k": _case("train", 1, 8192, 32, 8, 128, "bf16", segments=4, seg_min=576, seg_max=576, modalities=4),
        # Long context with 200 irregular segments, the worst case for partial tiles (workload C5).
        "train_64k": _case("train", 1, 65536, 32, 8, 128, "bf16", segments=200, seg_min=16, seg_max=512, modalities=16),
        # An additive bias per head and key, an ordinary length.
        "bias_2k": _case("bias", 2, 2048, 16, 16, 64, "bf16", segments=2, seg_min=256, seg_max=576, modalities=2),
        # The entry point that takes a bool mask instead of bitfields.
        "masked_4k": _case("masked", 2, 4096, 16, 16, 128, "bf16", segments=3, seg_min=256, seg_max=1024, modalities=3),
        # Rank 0 of two context-parallel ranks on the headline configuration.
        "shard_8k": _case("shard", 1, 8192, 32, 8, 128, "bf16", segments=4, seg_min=576, seg_max=576, modalities=4),
        # The prompt of one request, an odd length.
        "prefill_3k": _case("prefill", 1, 3001, 32, 8, 128, "bf16", segments=2, seg_min=576, seg_max=576, modalities=2),
        # Serving a batch with long caches: bound by reading the cache.
        "decode_batch_8k": _case("decode", 8, 8192, 32, 8, 128, "bf16", window=0, softcap=0.0),
        # One request with a short cache, sliding window and capped logits: bound by latency.
        "decode_single": _case("decode", 1, 1025, 32, 8, 128, "fp16", window=512, softcap=30.0),
    }
    return [dict(c, name=name) for name, c in named.items()]


_HEADS = [(6, 1), (6, 2), (6, 3), (6, 6), (4, 2), (8, 8), (16, 4), (16, 16), (32, 8)]
_HEAD_DIMS = [32, 40, 64, 64, 64, 80, 96, 128, 128, 128, 128]
_MOST_FLOPS = 6e12  # of a drawn case, counted at head dim 128


def _spread(rng, low, high):
    """A whole number of [low, high], spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random):
    while True:
        kind = rng.choice(["train", "train", "train", "train", "prefill", "prefill", "decode", "decode", "decode", "bias", "masked", "shard"])
        Hq, Hkv = rng.choice(_HEADS)
        D, dtype = rng.choice(_HEAD_DIMS), rng.choice(["fp16", "bf16", "bf16"])
        if kind == "decode":
            S = _spread(rng, 17, 65536)
            window = rng.choice([0, 0, 0, _spread(rng, 16, 8192)])
            c = _case(kind, _spread(rng, 1, 32), S, Hq, Hkv, D, dtype, window=window, softcap=rng.choice([0.0, 0.0, 30.0]))
            if 2 * c["B"] * S * Hkv * D * 2 > 4e9:
                continue
            return c
        S = _spread(rng, 57, 8192 if kind == "masked" else 32768)
        if kind == "shard":
            S = max(1024, S // 512 * 512)  # four chunks of whole 128-row blocks
        B = 1 if S > 8192 or kind == "shard" else _spread(rng, 1, 8)
        n = rng.randint(0, 6)
        most = max(8, min(1500, S // (2 * max(n, 1))))
        c = _case(kind, B, S, Hq, Hkv, D, dtype, segments=n, seg_min=max(4, most // 4), seg_max=most, modalities=rng.randint(1, 8),
                  pad=rng.choice([0, 0, S // 9]) if kind in ("train", "prefill") else 0)
        if work(c)["flops"] * (128 / D) > _MOST_FLOPS:
            continue
        return c


def _bitfields(case, seed):
    """int64 (B, S) on the host: text carries bit 62, bit 0 and every modality bit; a segment carries its modality's bit;
    padding carries 0."""
    rng = np.random.default_rng(seed)
    B, S = case["B"], case["S"]
    text = (1 << 62) | 1 | sum(1 << (m + 1) for m in range(case["modalities"]))
    bf = np.full((B, S), text, dtype=np.int64)
    for b in range(B):
        end = S - case["pad"] if b % 2 else S
        lengths = [int(x) for x in rng.integers(case["seg_min"], case["seg_max"] + 1, case["segments"])]
        while sum(lengths) > end:
            lengths.pop()
        cuts, before = np.sort(rng.integers(0, end - sum(lengths) + 1, len(lengths))), 0
        for k, n in enumerate(lengths):
            start = int(cuts[k]) + before
            # distinct modalities as long as there are enough of them
            m = k if case["segments"] <= case["modalities"] else int(rng.integers(0, case["modalities"]))
            bf[b, start : start + n] = 1 << (m + 1)
            before += n
        bf[b, end:] = 0
    return bf


def _allowed(bf, rows=None):
    """Allowed (query, key) pairs: a text row sees itself and everything before it (all of it shares a bit with text),
    a modality row sees the rows of its own modality, padding sees nothing.  ``rows``: only these query rows."""
    pairs = 0
    for one in bf:
        live = np.cumsum(one != 0)
        text = (one & 1) != 0
        pick = np.ones_like(text) if rows is None else np.isin(np.arange(one.size), rows)
        pairs += int(live[text & pick].sum())
        for bits in np.unique(one[~text & (one != 0)]):
            pairs += int((one == bits).sum()) * int(((one == bits) & pick).sum())
    return pairs


def _zigzag(S):
    """Rank 0 of two: chunks 0 and 3 of four; the gathered keys are ordered rank by rank."""
    c = np.split(np.arange(S), 4)
    return np.concatenate([c[0], c[3]]), np.concatenate([c[0], c[3], c[1], c[2]])


def prepare(case, seed):
    dev = torch.device("cuda")
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    B, S, Hq, Hkv, D, kind = (case[k] for k in ("B", "S", "Hq", "Hkv", "D", "kind"))

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=dtype)

    state = {"kind": kind}
    if kind == "decode":
        state.update(module=torch.nn.Module().eval(), q=normal(B, Hq, 1, D), k=normal(B, Hkv, S, D), v=normal(B, Hkv, S, D),
                     options={"scaling": D ** -0.5, "sliding_window": case["window"] or None, "softcap": case["softcap"] or None})
        return state
    bf = torch.from_numpy(_bitfields(case, seed)).to(dev)
    q, k, v, do = normal(B, S, Hq, D), normal(B, S, Hkv, D), normal(B, S, Hkv, D), normal(B, S, Hq, D)
    if kind == "prefill":  # the projections' (B, S, H, D) memory, seen as (B, H, S, D)
        state.update(module=torch.nn.Module().eval(), q=q.transpose(1, 2), k=k.transpose(1, 2), v=v.transpose(1, 2), bf=bf)
        return state
    if kind == "shard":
        iq, ik = (torch.from_numpy(x).to(dev) for x in _zigzag(S))
        BitfieldUtils.clear_cache()
        flags = BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
        # the flags of the shard: rows and columns of the sequence's flags, re-indexed block by block
        flags = flags[:, iq[::128] // 128][:, :, ik[::32] // 32].contiguous()
        BitfieldUtils.clear_cache()
        state.update(q=q[:, iq].contiguous(), k=k[:, ik].contiguous(), v=v[:, ik].contiguous(), do=do[:, iq].contiguous(),
                     bf=bf, flags=flags, iq=iq, ik=ik)
        return state
    state.update(q=q.requires_grad_(True), k=k.requires_grad_(True), v=v.requires_grad_(True), do=do)
    if kind == "masked":
        live = (bf & ((1 << 62) - 1)).unsqueeze(1)  # keys
        rows = live.transpose(1, 2)
        causal = torch.ones(S, S, dtype=torch.bool, device=dev).tril()
        state["mask"] = torch.where((rows & 1) != 0, ((rows & live) != 0) & causal, (rows == live) & (rows != 0))
    else:
        state["bf"] = bf
    if kind == "bias":
        slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / Hq) for h in range(Hq)], device=dev)
        state["bias"] = slopes[None, :, None, None] * torch.arange(1 - S, 1, device=dev, dtype=torch.float32)
    return state


def run(state):
    kind, q, k, v = state["kind"], state["q"], state["k"], state["v"]
    if kind == "decode":
        return bitfield_attention_forward(state["module"], q, k, v, None, **state["options"])[0]
    if kind == "prefill":
        BitfieldUtils.clear_cache()
        with torch.no_grad():
            return bitfield_attention_forward(state["module"], q, k, v, state["bf"])[0]
    if kind == "shard":
        bf, flags, iq, ik = state["bf"], state["flags"], state["iq"], state["ik"]
        o, lse, scale = _bitfield_attn_forward(q, k, v, bf, flags, iq, ik)
        dq, dk, dv = (torch.zeros(x.shape, dtype=torch.float32, device=x.device) for x in (q, k, v))
        _bitfield_attn_backward(state["do"], q, k, v, o, bf, flags, lse, dq, dk, dv, iq, ik, softmax_scale=scale)
        return o, lse, dq, dk, dv
    if kind == "masked":
        o = flash_attn_func(q, k, v, mask=state["mask"])
    else:
        BitfieldUtils.clear_cache()
        o = bitfield_attn_func(q, k, v, state["bf"], state.get("bias"))
    return (o, *torch.autograd.grad(o, (q, k, v), state["do"]))


def work(case):
    """q, k, v (and do) read once, o (and the gradients) written once, the mask read once; 4 D flops per head and allowed
    pair for the forward, 10 D for the backward."""
    B, S, Hq, Hkv, D, kind = (case[k] for k in ("B", "S", "Hq", "Hkv", "D", "kind"))
    if kind == "decode":
        keys = min(S, case["window"] or S)
        return {"bytes": 2 * (2 * B * keys * Hkv * D + 2 * B * Hq * D), "flops": 4 * B * keys * Hq * D}
    bf = _bitfields(case, 0)
    q_rows, kv_rows = B * S * Hq * D, B * S * Hkv * D
    if kind == "prefill":
        return {"bytes": 2 * (2 * q_rows + 2 * kv_rows) + 8 * B * S, "flops": 4 * D * Hq * _allowed(bf)}
    if kind == "shard":
        local = q_rows // 2
        flops = 14 * D * Hq * _allowed(bf, _zigzag(S)[0])
        return {"bytes": 2 * (3 * local + 2 * kv_rows) + 4 * (local + 2 * kv_rows + B * Hq * S // 2) + 8 * B * S, "flops": flops}
    mask = B * S * S if kind == "masked" else 8 * B * S
    bias = 4 * Hq * S if kind == "bias" else 0
    return {"bytes": 2 * (4 * q_rows + 4 * kv_rows) + mask + bias, "flops": 14 * D * Hq * _allowed(bf)}


def tolerance(case):
    """Probabilities and their gradients are rounded to the 16-bit type before they are multiplied."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 3e-3}
