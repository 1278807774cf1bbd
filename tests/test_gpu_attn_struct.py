"""The struct form of the backward (``bam_attn_bwd``) called as a C host calls it: the heads taken in runs of whole kv heads,
with and without a dS workspace, give what one run gives and what the oracle gives."""

import ctypes

import pytest
import torch

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu


def tensor(t):
    return _bam_hip.TensorArg(t.data_ptr(), *t.stride()[:3])


def backward(q, k, v, o, do, lse, bf, flags, plan, scale, runs, workspace):
    B, S, Hq, D = q.shape
    grads = [torch.full_like(t, 7.0) for t in (q, k, v)]
    delta = torch.full_like(lse, 7.0)
    a = _bam_hip.Attn()
    for name, t in zip(("q", "k", "v", "o", "dout", "dq", "dk", "dv"), (q, k, v, o, do, *grads)):
        setattr(a, name, tensor(t))
    a.lse, a.delta, a.bf, a.bf_stride_b = lse.data_ptr(), delta.data_ptr(), bf.data_ptr(), bf.stride(0)
    a.flags, a.flags_stride_b, a.flags_stride_m = flags.data_ptr(), flags.stride(0), flags.stride(1)
    a.plan = ctypes.pointer(plan.struct)
    a.mode, a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D = 0, B, S, S, Hq, k.shape[2], D
    a.dtype, a.accumulate, a.head_runs, a.scale = BA._dtype_code(q.dtype), 0, runs, scale
    if workspace:
        pairs = plan.ds_pairs()
        ws = torch.empty((Hq // runs * pairs * 8192,), dtype=torch.uint8, device=q.device)
        a.ds_workspace, a.ds_capacity = ws.data_ptr(), pairs
    _bam_hip.call("bam_attn_bwd", ctypes.byref(a), BA._stream_ptr(q.device))
    torch.cuda.synchronize()
    return grads


# head dims on both sides of 64: up to there the dQ kernel runs first and computes delta from the o of its run's heads
@pytest.mark.parametrize("D,workspace", [(32, False), (40, False), (64, False), (96, False), (96, True), (128, True)])
@pytest.mark.parametrize("B,S,Hq,Hkv", [(1, 200, 4, 4), (2, 331, 8, 4)])
def test_heads_in_runs(D, workspace, B, S, Hq, Hkv):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    q, do = ((torch.randn(B, S, Hq, D, generator=g)).bfloat16() for _ in range(2))
    k, v = ((torch.randn(B, S, Hkv, D, generator=g)).bfloat16() for _ in range(2))
    bf = random_bitfield(B, S, seed=S, pad=5)
    want = O.attention_backward(q, k, v, bf, do)
    q, k, v, do, bf = (t.to(dev) for t in (q, k, v, do, bf))
    BA.BitfieldUtils.clear_cache()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    plan = BA.BitfieldUtils.plan_for(flags, bf)
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags)
    one = backward(q, k, v, o, do, lse, bf, flags, plan, scale, 1, workspace)
    for got, w in zip(one, want):
        assert rel_l2(got.float().cpu(), w) <= 1.2e-2  # probabilities and dS in bf16: 2^-9 a term, a few times that in the norm
    for runs in (2, 4):
        for got, w in zip(backward(q, k, v, o, do, lse, bf, flags, plan, scale, runs, workspace), one):
            assert torch.equal(got, w), runs
    BA.BitfieldUtils.clear_cache()
