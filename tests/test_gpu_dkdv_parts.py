"""dK / dV with the q heads of a kv head dealt to several workgroups: key tiles that end early, every number of parts
(among them fewer than q heads), typed and accumulated gradients, a bias (indexed by absolute head), strided heads."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu


# (how many parts each of them gets: test_dkdv_parts.py)
@pytest.mark.parametrize("B,S,Hq,Hkv,D", [
    (1, 129, 16, 1, 32), (1, 700, 32, 8, 40), (1, 2100, 6, 3, 56), (4, 400, 6, 1, 64),
    (3, 1000, 24, 4, 64),  # 3 parts of 2 heads
    (1, 4100, 12, 3, 8),   # 4 parts of 1
    (1, 700, 32, 8, 128), (2, 700, 16, 4, 96), (1, 1000, 72, 8, 80),  # with the hand-over of dS
    (2, 900, 16, 4, 96), (1, 2003, 12, 4, 112),  # in one launch with dQ
    (2, 283, 6, 2, 64), (4, 1537, 8, 4, 32),  # one part: too little to share, enough workgroups
])
@pytest.mark.parametrize("bias", [False, True])
def test_parts_against_the_oracle(B, S, Hq, Hkv, D, bias):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    q, do = ((torch.randn(B, S, Hq, D, generator=g) * 0.5).bfloat16() for _ in range(2))
    k, v = ((torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16() for _ in range(2))
    bf = random_bitfield(B, S, seed=S, pad=9)
    bt = torch.randn(1, Hq, 1, S, generator=g) if bias else None
    gq, gk, gv = O.attention_backward(q, k, v, bf, do, bias=bt) if bias else O.attention_backward(q, k, v, bf, do)
    # k, v: heads of a wider tensor
    wide = torch.cat((k, v), 2).to(dev).requires_grad_(True)
    qd, bfd, bd = q.to(dev).requires_grad_(True), bf.to(dev), None if bt is None else bt.to(dev)
    BA.BitfieldUtils.clear_cache()
    kd, vd = wide[:, :, :Hkv], wide[:, :, Hkv:]
    o = BA.bitfield_attn_func(qd, kd, vd, bfd, bd)
    dq, dk, dv = torch.autograd.grad(o, (qd, kd, vd), do.to(dev))
    # probabilities and dS are rounded to bf16 before they are multiplied: 2^-9 a term, a few times that in the norm
    for name, got, want in (("dq", dq, gq), ("dk", dk, gk), ("dv", dv, gv)):
        rel = ((got.float().cpu() - want).norm() / want.norm()).item()
        assert rel <= 1.2e-2, (name, rel)
    # accumulated into fp32 gradients that hold something already: the same sums before they are rounded
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bfd)
    with torch.no_grad():
        o, lse, scale = BA._bitfield_attn_forward(qd, kd, vd, bfd, flags, bias=bd)
        acc = [torch.full(x.shape, 1.0, device=dev) for x in (qd, kd, vd)]
        BA._bitfield_attn_backward(do.to(dev), qd, kd, vd, o, bfd, flags, lse, *acc, bias=bd, softmax_scale=scale)
    for a, t in zip(acc[1:], (dk, dv)):
        err = (a - 1.0 - t.float()).abs() - t.float().abs() * 2.0 ** -8 - 2.0 ** -22
        assert err.max().item() <= 0
    BA.BitfieldUtils.clear_cache()


def test_without_room_for_the_parts_the_backward_runs_in_one_part():
    B, S, Hq, Hkv, D = 1, 512, 8, 1, 64  # 8 parts: 2 MiB, a segment of its own; everything else comes from smaller ones
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(0)
    q, k, v, do = (torch.randn(B, S, H, D, generator=g, device=dev).bfloat16().requires_grad_(n < 3)
                   for n, H in enumerate((Hq, Hkv, Hkv, Hq)))
    bf = random_bitfield(B, S, seed=1).to(dev)
    BA.BitfieldUtils.clear_cache()
    want = torch.autograd.grad(BA.bitfield_attn_func(q, k, v, bf), (q, k, v), do)
    o = BA.bitfield_attn_func(q, k, v, bf)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    small = [torch.empty(1 << 19, dtype=torch.uint8, device=dev) for _ in range(8)]  # room for the gradients
    total = torch.cuda.get_device_properties(dev).total_memory
    hold = []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved(dev) / total)
        while True:  # what is left of larger segments
            try:
                hold.append(torch.empty(2 << 20, dtype=torch.uint8, device=dev))
            except torch.cuda.OutOfMemoryError:
                break
        small = small[:1]  # (keeps their segment)
        got = torch.autograd.grad(o, (q, k, v), do)
        torch.cuda.synchronize()
        with pytest.raises(torch.cuda.OutOfMemoryError):  # there was no room indeed
            torch.empty(2 << 20, dtype=torch.uint8, device=dev)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        del hold, small
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):  # the same sums in another order, rounded to bf16 once
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() <= 2.0 ** -8
    BA.BitfieldUtils.clear_cache()
