"""Head dims between the compiled ones (32, 64, 96, 128): the kernels take every multiple of 8 as it is.  Forward,
gradients written in the input dtype and gradients accumulated in fp32, with and without the dS hand-over (head dims
above 64), against the fp32 oracle at the bars of the other parity tests."""

import ctypes

import pytest
import torch

from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel import interface
from oracle import bam_oracle as O
from tests import lds_fill
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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 24, 32, 40, 56, 64, 72, 96, 104, 128])
def test_an_infinity_in_a_key_gives_its_scores_and_nothing_else(dtype, D):
    # a key with -inf in one column and queries that are positive there: every score of it is -inf and its weight is 0,
    # also where the tiles have columns past the head dim.  Lengths with and without a ragged last tile.
    d = torch.device("cuda:0")
    for S in (64, 200):
        g = torch.Generator().manual_seed(D + S)
        q, k, v = ((torch.randn(1, S, H, D, generator=g) * 0.5).to(dtype) for H in (4, 2, 2))
        bf = torch.full((1, S), (1 << 62) | 1 | 2, dtype=torch.int64)
        col, keys = 3, torch.tensor([5, 41, S - 2])
        q[..., col] = q[..., col].abs() + 0.5
        k[:, keys, :, col] = -float("inf")
        want, _ = O.attention_forward(q, k, v, bf)
        assert torch.isfinite(want).all()
        BA.BitfieldUtils.clear_cache()
        qd, kd, vd, bfd = (t.to(d) for t in (q, k, v, bf))
        o = BA.bitfield_attn_func(qd, kd, vd, bfd)
        mask = torch.ones(S, S, dtype=torch.bool, device=d).tril()[None]
        for got in (o, A.flash_attn_func(qd, kd, vd, mask=mask)):
            assert (got.float().cpu() - want).abs().max().item() <= 2e-2
        # the decode step: one query against the same keys
        out, _ = interface.bitfield_attention_forward(torch.nn.Module().eval(), qd[:, -1:].transpose(1, 2), kd.transpose(1, 2),
                                                      vd.transpose(1, 2), None)
        assert (out[:, 0].float().cpu() - want[:, -1]).abs().max().item() <= 2e-2
        # gradients: dS of those keys is 0, so only the column of dq that multiplies it by the infinity is not a number.  (Whole
        # tiles of rows only: the zero rows past the end of a ragged one make NaN of a key's infinity in dk and dv.)
        if S % 64:
            continue
        do = torch.randn(1, S, 4, D, generator=g).to(dtype)
        inputs = [t.clone().requires_grad_(True) for t in (qd, kd, vd)]
        dq, dk, dv = torch.autograd.grad(BA.bitfield_attn_func(*inputs, bfd), inputs, do.to(d))
        rest = [c for c in range(D) if c != col]
        wq, wk, wv = O.attention_backward(q, k, v, bf, do)
        for a, b in ((dq[..., rest], wq[..., rest]), (dk, wk), (dv, wv)):
            assert torch.isfinite(b).all() and torch.isfinite(a).all() and rel_l2(a.float().cpu(), b) <= 5e-2
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("D", [24, 40, 56, 72, 104])
def test_columns_past_the_head_dim_do_not_come_from_lds_leftovers(D):
    # after the LDS of every compute unit was filled with NaN patterns: same bits as undisturbed
    d = torch.device("cuda:0")
    fill, sink = lds_fill.load(), torch.zeros(4, dtype=torch.int32, device=d)
    g = torch.Generator().manual_seed(D)
    q, k, v, do = ((torch.randn(2, 200, H, D, generator=g) * 0.5).bfloat16().to(d) for H in (4, 2, 2, 4))
    bf = random_bitfield(2, 200, seed=D, pad=3).to(d)
    BA.BitfieldUtils.clear_cache()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    module = torch.nn.Module().eval()

    def run(disturb):
        def poison():
            if disturb:
                assert fill.lds_fill(ctypes.c_void_p(sink.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0

        acc = [torch.zeros(t.shape, dtype=torch.float32, device=d) for t in (q, k, v)]
        poison()
        o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags)
        poison()
        BA._bitfield_attn_backward(do, q, k, v, o, bf, flags, lse, *acc, softmax_scale=scale)
        poison()
        step = interface.bitfield_attention_forward(module, q[:, -1:].transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), None)[0]
        torch.cuda.synchronize()
        return o, *acc, step

    want = run(False)
    assert all(torch.isfinite(t).all() for t in want)
    for _ in range(4):
        assert all(torch.equal(a, b) for a, b in zip(run(True), want))
    BA.BitfieldUtils.clear_cache()
