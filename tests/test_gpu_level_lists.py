"""Forward and dQ where every row sees every key, with 257 to 512 workgroups: the two streams of a workgroup take a unit each (bitfields,
bool masks) or there is one stream (no mask).  Either way a row's result is that of one stream, bit for bit: the same sequences in
a call with more than 512 workgroups."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel.attention import _MaskPlan, flash_attn_func
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu


def _run(kind, q, k, v, do):
    x = [t.contiguous().requires_grad_(True) for t in (q, k, v)]
    B, S = q.shape[:2]
    BA.BitfieldUtils.clear_cache()
    _MaskPlan.forget()
    if kind == "bitfield":
        o = BA.bitfield_attn_func(*x, torch.full((B, S), 2, dtype=torch.int64, device="cuda"))
    else:
        o = flash_attn_func(*x, mask=torch.ones(B, S, S, dtype=torch.bool, device="cuda") if kind == "mask" else None)
    return o.detach(), *torch.autograd.grad(o, x, do.contiguous())


# workgroups: 273 (an odd number: the last workgroup has one unit), 320, 510, 512; ragged ends
@pytest.mark.parametrize("kind", ["bitfield", "mask", "none"])
@pytest.mark.parametrize("D", [40, 64, 96, 128])
@pytest.mark.parametrize("S,H,few,many", [(1601, 21, 1, 2), (1300, 10, 3, 6), (2170, 10, 3, 4), (1024, 16, 3, 5), (2048, 32, 1, 2)])
def test_level_lists_equal_one_stream(S, H, few, many, D, kind):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v, do = (torch.randn(many, S, H, D, generator=g, device="cuda").bfloat16() for _ in range(4))
    all_ = _run(kind, q, k, v, do)
    for a, b in zip(all_, _run(kind, *(t[:few] for t in (q, k, v, do)))):
        assert torch.isfinite(b).all() and torch.equal(a[:few], b)
    BA.BitfieldUtils.clear_cache()
    _MaskPlan.forget()


# index tensors, both forms of a bias, grouped heads, nearly level lists (one text row in 300): forward and dQ
@pytest.mark.parametrize("kind", ["indexed", "bias row", "bias matrix", "grouped", "nearly"])
@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("S,H,few,many", [(1601, 21, 1, 2), (1300, 12, 3, 6)])
def test_other_forms_of_level_lists_equal_one_stream(S, H, few, many, D, kind):
    Hkv = H // 3 if kind == "grouped" else H
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v, do = (torch.randn(many, S, h, D, generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv, H))
    bias = torch.randn(1, H, S if kind == "bias matrix" else 1, S, generator=g, device="cuda") if "bias" in kind else None
    rows = torch.arange(S, device="cuda") if kind == "indexed" else None

    def run(n):
        bf = torch.full((n, S), 2, dtype=torch.int64, device="cuda")
        if kind == "nearly":
            bf[:, 150::300] = (1 << 62) | 2
        x = [t[:n].contiguous() for t in (q, k, v, do)]
        BA.BitfieldUtils.clear_cache()
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
        o, lse, scale = BA._bitfield_attn_forward(*x[:3], bf, flags, rows, rows, bias=bias)
        grads = [torch.zeros(t.shape, device="cuda") for t in x[:3]]
        BA._bitfield_attn_backward(x[3], *x[:3], o, bf, flags, lse, *grads, rows, rows, bias=bias, softmax_scale=scale)
        return o, lse, grads[0]

    for a, b in zip(run(many), run(few)):
        assert not torch.isnan(b).any() and torch.equal(a[:few], b)
    BA.BitfieldUtils.clear_cache()


# both forms of the plan builder's last launches
@pytest.mark.parametrize("B,S", [(1, 1), (1, 65), (3, 515), (2, 1300), (5, 2000), (1, 9000), (70, 130)])
def test_the_plan_knows_how_level_its_lists_are(B, S):
    bf = random_bitfield(B, S, seed=S, pad=S // 7).cuda()
    BA.BitfieldUtils.clear_cache()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    plan = BA.BitfieldUtils.plan_for(flags, bf)
    st, ws, num_m = plan.struct, plan.workspace, -(-S // 128)
    at = (st.group_order - ws.data_ptr()) // 4
    order = ws.view(torch.int32)[at : at + B * num_m + 1].tolist()
    fine = plan.fine_classes().cpu() > 0
    slices = plan.slice_order().cpu()
    lengths = {}
    for b in range(B):
        for grp in range(num_m):
            rows = [int(s) & 0x3FFFFFFF for s in slices[b, 4 * grp : 4 * grp + 4] if s >= 0]
            cols = torch.zeros(2 * (-(-fine.shape[2] // 2)), dtype=torch.bool)
            cols[: fine.shape[2]] = fine[b, rows].any(dim=0)
            lengths[b * num_m + grp] = int(cols.view(-1, 2).any(dim=1).sum())
    codes, heads = order[:-1], order[-1]
    assert sorted(codes) == sorted(lengths) and [lengths[c] for c in codes] == sorted(lengths.values(), reverse=True)
    # the fewest q heads for which longest - mean is at most 5 tiles per 512 workgroups (or lists are a handful of tiles anyway)
    n, longest, total = len(lengths), max(lengths.values()), sum(lengths.values())
    assert heads == (0 if longest <= 10 else -(-(longest * n - total) * 512 // (5 * n * n)))
    BA.BitfieldUtils.clear_cache()
