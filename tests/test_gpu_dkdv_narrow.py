"""dK/dV with four waves a workgroup (head dims up to 64, more than 1024 workgroups), against the oracle: one to several key tiles, odd
counts of slices, head dims below the compiled one, grouped heads, a bias, index tensors and accumulated gradients."""

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
])
def test_gradients_against_the_oracle(B, S, Hq, Hkv, D, dtype, form):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    q, do = ((torch.randn(B, S, Hq, D, generator=g) * 0.5).to(dtype) for _ in range(2))
    k, v = ((torch.randn(B, S, Hkv, D, generator=g) * 0.5).to(dtype) for _ in range(2))
    bf = random_bitfield(B, S, seed=S, pad=S // 13)
    if form == "level":
        bf = torch.full_like(bf, 2)
    bias = torch.randn(1, Hq, 1, S, generator=g) if form == "bias" else None
    qd, kd, vd, dod, bfd = (t.to(dev) for t in (q, k, v, do, bf))
    BA.BitfieldUtils.clear_cache()
    if form == "index":  # the blocks in another order, gradients accumulated
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bfd)
        idx = torch.arange(S).roll(-128 * (S // 256)).to(dev)
        flags = flags[:, idx[::128] // 128][:, :, idx[::32] // 32].contiguous()
        qs, ks, vs, dos = (t[:, idx].contiguous() for t in (qd, kd, vd, dod))
        o, lse, scale = BA._bitfield_attn_forward(qs, ks, vs, bfd, flags, idx, idx)
        grads = [torch.ones(t.shape, dtype=torch.float32, device=dev) for t in (qs, ks, vs)]
        BA._bitfield_attn_backward(dos, qs, ks, vs, o, bfd, flags, lse, *grads, idx, idx, softmax_scale=scale)
        got = [torch.empty_like(t).index_copy_(1, idx, t - 1.0) for t in grads]
    else:
        leaves = [t.requires_grad_(True) for t in (qd, kd, vd)]
        o = BA.bitfield_attn_func(*leaves, bfd, None if bias is None else bias.to(dev))
        got = torch.autograd.grad(o, leaves, dod)
    # (two sequences of the batch: the oracle runs on the CPU)
    for b in (0, B - 1):
        args = [t[b : b + 1] for t in (q, k, v, bf, do)]
        want = O.attention_backward(*args, bias=bias) if form == "bias" else O.attention_backward(*args)
        # probabilities and dS are rounded to 16 bits before they are multiplied: 2^-9 a term, a few times that in the norm
        for name, x, y in zip(("dq", "dk", "dv"), got, want):
            rel = ((x[b : b + 1].float().cpu() - y).norm() / y.norm()).item()
            assert rel <= 1e-2, f"{name}: {rel}"
