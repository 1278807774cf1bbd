"""dK/dV and dQ of small problems in one launch (head dims above 32), against the oracle: either side of the sizes where it starts and
ends, two streams on a list and side by side, one workgroup of dK/dV, parts, a bias, a bool mask, index tensors (also fewer rows than
keys), accumulated gradients; and which of them take a dS workspace."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel.attention import flash_attn_func
from oracle import bam_oracle as O
from tests.helpers import random_bitfield, rel_l2
from tests.test_gpu_ds_handover import inputs, run_backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,Hq,Hkv,D", [
    (1, 128, 2, 1, 64), (1, 129, 2, 1, 64),        # from three key tiles on
    (1, 700, 42, 42, 64), (1, 700, 43, 43, 64),    # 252 and 258 workgroups of dQ: up to 256 with so few keys
    (2, 1030, 21, 3, 40), (1, 1500, 40, 8, 48),    # 378, 480: the plan decides how the streams share the lists; parts
    (1, 1601, 4, 4, 56),
    (1, 767, 4, 4, 96), (1, 768, 4, 2, 72),        # above head dim 64: from 768 keys on
    (1, 1030, 16, 2, 128), (1, 1500, 11, 11, 80),  # parts; 264 workgroups: the count decides (level lists: two launches)
    (1, 2049, 15, 15, 128), (1, 1030, 29, 29, 128),  # 510 and 522 workgroups
])
@pytest.mark.parametrize("form", ["plain", "bias", "mask", "index", "level"])
def test_gradients_against_the_oracle(B, S, Hq, Hkv, D, form):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    q, do = ((torch.randn(B, S, Hq, D, generator=g) * 0.5).bfloat16() for _ in range(2))
    k, v = ((torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16() for _ in range(2))
    bf = random_bitfield(B, S, seed=S, pad=S // 13)
    if form == "level":  # nothing hidden
        bf = torch.full_like(bf, 2)
    bias = torch.randn(1, Hq, 1, S, generator=g) if form == "bias" else None
    want = O.attention_backward(q, k, v, bf, do, bias=bias) if form == "bias" else O.attention_backward(q, k, v, bf, do)
    qd, kd, vd, dod, bfd = (t.to(dev) for t in (q, k, v, do, bf))
    BA.BitfieldUtils.clear_cache()
    if form == "index":  # the rows and keys in another order, gradients accumulated
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bfd)
        order = torch.arange(S).roll(-128 * (S // 256))
        if S % 128:  # (flags of whole blocks can be reordered)
            order = torch.arange(S)
        idx = order.to(dev)
        blocks = order[::128] // 128
        flags = flags[:, blocks.to(dev)][:, :, (order[::32] // 32).to(dev)].contiguous()
        qs, ks, vs, dos = (t[:, idx].contiguous() for t in (qd, kd, vd, dod))
        o, lse, scale = BA._bitfield_attn_forward(qs, ks, vs, bfd, flags, idx, idx)
        grads = [torch.ones(t.shape, dtype=torch.float32, device=dev) for t in (qs, ks, vs)]
        BA._bitfield_attn_backward(dos, qs, ks, vs, o, bfd, flags, lse, *grads, idx, idx, softmax_scale=scale)
        got = [torch.empty_like(t).index_copy_(1, idx, t - 1.0) for t in grads]
    else:
        leaves = [t.requires_grad_(True) for t in (qd, kd, vd)]
        if form == "mask":
            o = flash_attn_func(*leaves, mask=BA.materialize_bitfield_mask(bfd).to(torch.bool).contiguous())
        else:
            o = BA.bitfield_attn_func(*leaves, bfd, None if bias is None else bias.to(dev))
        got = torch.autograd.grad(o, leaves, dod)
    # probabilities and dS are rounded to bf16 before they are multiplied: 2^-9 a term, a few times that in the norm
    for name, x, y in zip(("dq", "dk", "dv"), got, want):
        rel = ((x.float().cpu() - y).norm() / y.norm()).item()
        assert rel <= 1e-2, f"{name}: {rel}"


# a rank of a zigzag split: S / 2 rows, S keys, every row block in another place than its positions say; parts of dK/dV where heads are
# grouped.  Above head dim 64: sizes decide, the count decides, two launches
@pytest.mark.parametrize("S,Hq,Hkv,D", [
    (1536, 4, 4, 64), (2048, 12, 3, 48), (2048, 30, 30, 64),
    (1536, 6, 2, 128), (2048, 8, 8, 96), (2048, 16, 16, 128), (4096, 8, 2, 72), (2048, 24, 24, 96),
])
def test_a_shard_against_the_oracle(S, Hq, Hkv, D):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(S + D)
    c = torch.arange(S).chunk(4)
    rows, keys = torch.cat((c[0], c[3])), torch.cat((c[0], c[3], c[1], c[2]))
    q, do = ((torch.randn(1, S // 2, Hq, D, generator=g) * 0.5).bfloat16().to(dev) for _ in range(2))
    k, v = ((torch.randn(1, S, Hkv, D, generator=g) * 0.5).bfloat16().to(dev) for _ in range(2))
    bf_cpu = random_bitfield(1, S, seed=S, pad=S // 13)
    flags = O.tile_flags_indexed(bf_cpu, rows, keys).to(dev)
    bf, rows, keys = bf_cpu.to(dev), rows.to(dev), keys.to(dev)
    BA.BitfieldUtils.clear_cache()
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags, rows, keys)
    got = [torch.ones(t.shape, dtype=torch.float32, device=dev) for t in (q, k, v)]
    BA._bitfield_attn_backward(do, q, k, v, o, bf, flags, lse, *got, rows, keys, softmax_scale=scale)
    want = O.attention_backward(q, k, v, bf, do, idx_q=rows, idx_k=keys)
    for name, x, y in zip(("dq", "dk", "dv"), got, want):  # (the bar above)
        rel = ((x - 1.0 - y).norm() / y.norm()).item()
        assert rel <= 1e-2, f"{name}: {rel}"
    BA.BitfieldUtils.clear_cache()


def two_launches(q, k, v, do, bf):
    """The gradients by the entry points that launch dK/dV and dQ one by one, dS handed over."""
    BA.BitfieldUtils.clear_cache()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    plan = BA.BitfieldUtils.plan_for(flags, bf)
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags)
    delta = torch.empty_like(lse)
    BA._launch_bwd_preprocess(o, do, delta)
    assert plan.attach_ds_workspace(q.shape[2], q.shape[3], q.shape[1]) is not None
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    BA._launch_bwd_dkdv(q, k, v, do, lse, delta, dk, dv, bf, flags, scale, accumulate=False, plan=plan)
    BA._launch_bwd_dq(q, k, v, do, lse, delta, dq, bf, flags, scale, accumulate=False, plan=plan)
    torch.cuda.synchronize()
    plan.detach_ds_workspace()
    return dq, dk, dv


@pytest.mark.parametrize("S,Hq,Hkv,level,takes", [
    (1100, 32, 32, False, True), (1500, 20, 20, True, True),    # 576 workgroups; 480, nothing hidden
    (1500, 20, 20, False, False), (2048, 8, 8, True, False),    # 480, of which the count says that they are uneven; 256
])
def test_which_sizes_hand_ds_over(S, Hq, Hkv, level, takes, monkeypatch):
    dev = torch.device("cuda:0")
    bf = (torch.full((1, S), 2) if level else random_bitfield(1, S, seed=S, pad=3)).to(dev)
    q, k, v, do = (t.to(dev) for t in inputs(1, S, Hq, Hkv, 128, torch.bfloat16, seed=S))
    got = run_backward(q, k, v, do, bf, True, monkeypatch, hands_over=takes)
    # where dS was handed over, against a call that may not; where it was not, against the two launches that do
    want = run_backward(q, k, v, do, bf, False, monkeypatch) if takes else two_launches(q, k, v, do, bf)
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    assert rel_l2(got[0].float(), want[0].float()) <= 2e-3  # the same rounded dS values, summed in another order
    BA.BitfieldUtils.clear_cache()
