"""Head dims between the compiled ones (32, 64, 96, 128): the kernels take every multiple of 8 as it is.  Forward,
gradients written in the input dtype and gradients accumulated in fp32, with and without the dS hand-over (head dims
above 64), against the fp32 oracle at the bars of the other parity tests."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 24, 40, 56, 72, 80, 88, 96, 104, 120])
@pytest.mark.parametrize("B,S,Hq,Hkv", [(2, 57, 2, 1), (1, 333, 4, 2)])
def test_head_dims_between_the_compiled_ones(dtype, D, B, S, Hq, Hkv):
    d = torch.device("cuda:0")
    g = torch.Generator().manual_seed(D + S)
    q, k, v, do = ((torch.randn(B, S, H, D, generator=g) * std).to(dtype)
                   for H, std in ((Hq, 0.5), (Hkv, 0.5), (Hkv, 0.5), (Hq, 1.0)))
    bf = random_bitfield(B, S, seed=S, pad=3)
    o_ref, _ = O.attention_forward(q, k, v, bf)
    want = O.attention_backward(q, k, v, bf, do)
    bfg, dog = bf.to(d), do.to(d)
    qg, kg, vg = (t.to(d).requires_grad_(True) for t in (q, k, v))
    for handover in (True, False):
        BA.BitfieldUtils.clear_cache()
        o = BA.bitfield_attn_func(qg, kg, vg, bfg)
        typed = torch.autograd.grad(o, (qg, kg, vg), dog)
        # the same through the private entry points: fp32 gradients, added to what the buffers hold
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bfg)
        o2, lse, scale = BA._bitfield_attn_forward(qg.detach(), kg.detach(), vg.detach(), bfg, flags)
        acc = [torch.ones(t.shape, dtype=torch.float32, device=d) for t in (q, k, v)]
        mask = bfg if handover else bfg.clone()  # flags of another tensor come without their plan
        BA._bitfield_attn_backward(dog, qg.detach(), kg.detach(), vg.detach(), o2, mask, flags, lse, *acc, softmax_scale=scale)
        torch.cuda.synchronize()
        assert o.shape == q.shape and torch.equal(o, o2)
        assert (o.float().cpu() - o_ref).abs().max().item() <= 2e-2
        for a, b, w in zip(typed, acc, want):
            assert a.shape == w.shape and torch.isfinite(a).all()
            assert rel_l2(a.float().cpu(), w) <= 5e-2 and rel_l2(b.cpu() - 1, w) <= 5e-2
    BA.BitfieldUtils.clear_cache()
