"""dK/dV with the lse that the dQ kernel has scaled, against the kernels that scale it themselves: the same bits."""

import ctypes

import pytest
import torch

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from tests.helpers import random_bitfield
from tests.test_gpu_sorted_rows import dev, sorted_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["flags", "sorted", "mask"])
@pytest.mark.parametrize("D", [32, 40, 64, 80])
@pytest.mark.parametrize("S", [1, 33, 200, 517])
def test_gradients_are_the_same_bits(S, D, mode):
    B, Hq, Hkv = 2, 4, 2
    g = torch.Generator(device=dev()).manual_seed(S + D)
    q, k, v, do = (torch.randn(B, S, H, D, generator=g, device=dev()).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(B, S, seed=S, pad=S // 9).to(dev())  # (rows of padding: their lse is -inf)
    flags, plan, ws, _ = sorted_plan(bf)
    o, lse = torch.empty_like(q), torch.empty((B, Hq, -(-S // 128) * 128), device=dev())
    a = _bam_hip.Attn()
    a.lse, a.flags, a.flags_stride_b, a.flags_stride_m = lse.data_ptr(), flags.data_ptr(), flags.stride(0), flags.stride(1)
    a.bf, a.bf_stride_b, a.mode = bf.data_ptr(), bf.stride(0), 0
    if mode == "mask":
        mask = BA.materialize_bitfield_mask(bf).to(torch.bool).contiguous()
        a.mask, a.mode = mask.data_ptr(), 2
    elif mode != "flags":
        a.plan = ctypes.pointer(plan)
    a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D = B, S, S, Hq, Hkv, D
    a.dtype, a.accumulate, a.head_runs, a.scale = BA._dtype_code(q.dtype), 0, 1, D**-0.5

    def backward(scaled):
        grads = [torch.full_like(t, 7.0) for t in (q, k, v)]
        delta = torch.full((2, *lse.shape), float("nan"), device=dev())
        for name, t in zip(("q", "k", "v", "o", "dout", "dq", "dk", "dv"), (q, k, v, o, do, *grads)):
            setattr(a, name, _bam_hip.TensorArg(t.data_ptr(), *t.stride()[:3]))
        a.delta, a.lse_scaled = delta[0].data_ptr(), delta[1].data_ptr() if scaled else None
        _bam_hip.call("bam_attn_bwd", ctypes.byref(a), BA._stream_ptr(dev()))
        torch.cuda.synchronize()
        return grads

    for name, t in zip(("q", "k", "v", "o"), (q, k, v, o)):
        setattr(a, name, _bam_hip.TensorArg(t.data_ptr(), *t.stride()[:3]))
    _bam_hip.call("bam_attn_fwd", ctypes.byref(a), BA._stream_ptr(dev()))
    for x, y in zip(backward(True), backward(False)):
        assert torch.equal(x, y)
