"""dK/dV with four waves a workgroup (head dims up to 64, more than 1024 workgroups), against the oracle: one to several key tiles, odd
counts of slices, head dims below the compiled one, grouped heads and their parts, a bias, index tensors (also fewer rows than keys) and
accumulated gradients, views with other strides, an infinite key."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,Hq,Hkv,D,dtype,form", [
    (72, 100, 16, 16, 64, torch.bfloat16, "plain"),   # one key tile, an odd count of slices
    (36, 129, 16, 16, 40, torch.float16, "plain"),    # a second tile of one key
    (48, 257, 16, 8, 32, torch.bfloat16, "plain"),
    (33, 500, 16, 8, 64, torch.float16, "plain"),     # 1056 workgroups
    (16, 500, 16, 16, 64, torch.bfloat16, "plain"),   # 1024: eight waves
    (12, 700, 16, 16, 24, torch.bfloat16, "bias"),
    (12, 700, 16, 16, 64, torch.bfloat16, "bias"),    # (eight waves)
    (12, 768, 16, 16, 64, torch.bfloat16, "index"),
    (12, 768, 16, 16, 32, torch.float16, "index"),
    (16, 640, 13, 13, 56, torch.bfloat16, "level"),   # nothing hidden
    (3, 3000, 32, 4, 32, torch.bfloat16, "plain"),    # 288 workgroups' work in four parts each: fp32 sums, added up behind
    (36, 129, 16, 16, 40, torch.bfloat16, "views"),
    (18, 515, 16, 16, 64, torch.float16, "views"),
    (9, 1024, 16, 16, 64, torch.bfloat16, "shard"),   # 512 rows, 1024 keys
    (18, 1024, 16, 8, 32, torch.float16, "shard"),
])
def test_gradients_against_the_oracle(B, S, Hq, Hkv, D, dtype, form):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    q, do = ((torch.randn(B, S, Hq, D, generator=g) * 0.5).to(dtype).to(dev) for _ in range(2))
    k, v = ((torch.randn(B, S, Hkv, D, generator=g) * 0.5).to(dtype).to(dev) for _ in range(2))
    bf = random_bitfield(B, S, seed=S, pad=S // 13).to(dev)
    if form == "level":
        bf = torch.full_like(bf, 2)
    bias = torch.randn(1, Hq, 1, S, generator=g).to(dev) if form == "bias" else None
    if form == "views":  # rows of one head one after the other; heads of a wider tensor
        q, do = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, do))
        wide = torch.cat((k, v, k[:, :, :1]), 2)
        k, v = wide[:, :, :Hkv], wide[:, :, Hkv : 2 * Hkv]
    BA.BitfieldUtils.clear_cache()
    if form in ("index", "shard"):  # blocks in another order, gradients accumulated
        rows = keys = torch.arange(S).roll(-128 * (S // 256))
        if form == "shard":  # a rank of a zigzag split
            c = torch.arange(S).chunk(4)
            rows, keys = torch.cat((c[0], c[3])), torch.cat((c[0], c[3], c[1], c[2]))
        flags = O.tile_flags(bf.cpu())[:, rows[::128] // 128][:, :, keys[::32] // 32].contiguous().to(dev)
        rows, keys = rows.to(dev), keys.to(dev)
        q, do, k, v = (t[:, idx].contiguous() for t, idx in ((q, rows), (do, rows), (k, keys), (v, keys)))
        o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags, rows, keys)
        got = [torch.ones(t.shape, dtype=torch.float32, device=dev) for t in (q, k, v)]
        BA._bitfield_attn_backward(do, q, k, v, o, bf, flags, lse, *got, rows, keys, softmax_scale=scale)
        got = [t - 1.0 for t in got]
        want = O.attention_backward(q, k, v, bf, do, idx_q=rows, idx_k=keys)
    else:
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        got = torch.autograd.grad(BA.bitfield_attn_func(*leaves, bf, bias), leaves, do)
        want = O.attention_backward(q, k, v, bf, do, bias=bias) if form == "bias" else O.attention_backward(q, k, v, bf, do)
    # probabilities and dS are rounded to 16 bits before they are multiplied: 2^-9 a term, a few times that in the norm
    for name, x, y in zip(("dq", "dk", "dv"), got, want):
        for b in range(B):
            rel = ((x[b].float() - y[b]).norm() / y[b].norm()).item()
            assert rel <= 1e-2, f"{name} of sequence {b}: {rel}"
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("D", [24, 64])
def test_an_infinity_in_a_key_stays_out_of_the_gradients(D):
    """A key with -inf in one column and queries that are positive there has the weight 0: K operands come from memory here, and the
    columns past the head dim are zeros beside it."""
    dev, B, S, H, col = torch.device("cuda:0"), 72, 128, 16, 3
    g = torch.Generator().manual_seed(D)
    q, k, v, do = ((torch.randn(B, S, H, D, generator=g) * 0.5).bfloat16().to(dev) for _ in range(4))
    q[..., col] = q[..., col].abs() + 0.5
    k[:, [5, 41, S - 2], :, col] = -float("inf")
    bf = torch.full((B, S), (1 << 62) | 1 | 2, dtype=torch.int64, device=dev)
    BA.BitfieldUtils.clear_cache()
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    dq, dk, dv = torch.autograd.grad(BA.bitfield_attn_func(*leaves, bf), leaves, do)
    wq, wk, wv = O.attention_backward(q, k, v, bf, do)
    rest = [c for c in range(D) if c != col]  # (that column of dq is 0 times the infinity)
    for a, b in ((dq[..., rest], wq[..., rest]), (dk, wk), (dv, wv)):
        assert torch.isfinite(b).all() and torch.isfinite(a).all() and ((a.float() - b).norm() / b.norm()).item() <= 1e-2
    BA.BitfieldUtils.clear_cache()
