"""Plans with sorted rows (``bam_tile_plan_sorted_counted``; the public functions take them from 32768 tokens on): their contents
against the definition, and attention with them against attention with a plan in natural order."""

import ctypes

import pytest
import torch

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu
M = (1 << 62) - 1


def dev():
    return torch.device("cuda:0")


def sorted_plan(bf):
    """(flags, plan struct, workspace, number of pairs) of a sorted plan."""
    B, S = bf.shape
    n = ctypes.c_int64()
    _bam_hip.call("bam_sorted_plan_workspace_bytes", B, S, ctypes.byref(n))
    ws = torch.full((n.value,), 0xEE, dtype=torch.uint8, device=dev())
    flags = torch.empty((B, -(-S // 128), -(-S // 32)), dtype=torch.int8, device=dev())
    plan = _bam_hip.Plan()
    _bam_hip.call("bam_tile_plan_sorted_counted", bf.data_ptr(), bf.stride(0), flags.data_ptr(), flags.stride(0), flags.stride(1),
                  ws.data_ptr(), ws.numel(), B, S, ctypes.byref(plan), None, 0, BA._stream_ptr(dev()))
    torch.cuda.synchronize()
    at = plan.ds_count - ws.data_ptr()
    return flags, plan, ws, int(ws[at : at + 4].view(torch.int32).item())


def array(ws, address, shape, dtype):
    size = torch.empty((), dtype=dtype).element_size()
    n = 1
    for s in shape:
        n *= s
    at = address - ws.data_ptr()
    return ws[at : at + n * size].view(dtype).reshape(shape).cpu()


@pytest.mark.parametrize("S", [1, 31, 32, 200, 1023, 1025, 3000, 20000])
@pytest.mark.parametrize("wide", [False, True])
def test_contents(S, wide):
    B = 2
    bf = random_bitfield(B, S, seed=S, pad=S // 9, wide=wide)
    bf[0, S // 3 : S // 2] |= 1 << 40  # bitfields of several bits as well
    flags, plan, ws, pairs = sorted_plan(bf.to(dev()))
    assert torch.equal(flags.cpu(), BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf.to(dev())).cpu())
    Sr = -(-S // 128) * 128
    rows = array(ws, plan.rows, (B, Sr), torch.int32)
    moved = array(ws, plan.rows_moved, (B,), torch.int32)
    bits = array(ws, plan.rows_bits, (B, Sr), torch.int64)
    num_n = -(-S // 32)
    fine = array(ws, plan.fine, (B, Sr // 32, plan.fine_stride_s), torch.uint8)
    mask = BA.materialize_bitfield_mask(bf.to(dev())).cpu()
    for b in range(B):
        r = rows[b, :S].long()
        assert torch.equal(r.sort().values, torch.arange(S)) and (rows[b, S:] == S).all() and (bits[b, S:] == 0).all()
        assert torch.equal(bits[b, :S], bf[b][r])
        kinds = torch.where(bf[b] & 1 != 0, 0, torch.where(bf[b] & M == 0, 2, 1))
        slices = torch.nn.functional.pad(kinds, (0, -S % 32), value=2).reshape(-1, 32)
        mixed = int(((slices == 0).any(1) & (slices == 1).any(1)).sum())
        assert moved[b] == (mixed * 32 >= slices.shape[0])
        if not moved[b]:
            assert torch.equal(r, torch.arange(S))
        kind = kinds[r]
        assert not moved[b] or (kind[1:] >= kind[:-1]).all()  # text, modalities, padding
        # every bitfield of a modality is one run, rows of equal kind keep their order inside it
        group = torch.where(kind == 1, bits[b, :S] & M, -kind.long())
        assert (r[1:] > r[:-1])[group[1:] == group[:-1]].all()
        seen = torch.unique_consecutive(group)
        assert wide or not moved[b] or seen.numel() == group.unique().numel()  # (different bitfields may share a sorting class)
        cells = torch.zeros(Sr, num_n * 32)
        cells[:S, :S] = mask[b][r].float()
        count = cells.reshape(Sr // 32, 32, num_n, 32).sum((1, 3))
        inside = torch.zeros(Sr, num_n * 32)
        inside[:S, :S] = 1
        full = inside.reshape(Sr // 32, 32, num_n, 32).sum((1, 3))
        want = torch.where(count == 0, 0, torch.where(count == full, 2, 1))
        assert torch.equal(fine[b, :, :num_n].long(), want.long())
    columns = torch.nn.functional.pad(fine[:, :, :num_n], (0, -num_n % 4)).reshape(B, Sr // 32, -1, 4)
    assert pairs == int((columns != 0).any(-1).sum())


def attention(q, k, v, do, bf, flags, plan, pairs, bias, scale):
    """Forward and backward through the struct entry points with this plan (None: from the flags alone)."""
    B, S, Hq, D = q.shape
    o, lse = torch.full_like(q, 7.0), torch.full((B, Hq, -(-S // 128) * 128), 7.0, device=q.device)
    grads = [torch.full_like(t, 7.0) for t in (q, k, v)]
    delta = torch.full_like(lse, float("nan"))
    a = _bam_hip.Attn()
    for name, t in zip(("q", "k", "v", "o", "dout", "dq", "dk", "dv"), (q, k, v, o, do, *grads)):
        setattr(a, name, _bam_hip.TensorArg(t.data_ptr(), *t.stride()[:3]))
    a.lse, a.delta, a.bf, a.bf_stride_b = lse.data_ptr(), delta.data_ptr(), bf.data_ptr(), bf.stride(0)
    a.flags, a.flags_stride_b, a.flags_stride_m = flags.data_ptr(), flags.stride(0), flags.stride(1)
    if plan is not None:
        a.plan = ctypes.pointer(plan)
    if bias is not None:
        b = _bam_hip.Bias(bias.data_ptr(), 0, bias.stride(1), bias.stride(2) if bias.shape[2] > 1 else 0, 1)
        a.bias = ctypes.pointer(b)
    a.mode, a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D = 0, B, S, S, Hq, k.shape[2], D
    a.dtype, a.accumulate, a.head_runs, a.scale = BA._dtype_code(q.dtype), 0, 1, scale
    stream = BA._stream_ptr(q.device)
    _bam_hip.call("bam_attn_fwd", ctypes.byref(a), stream)
    if pairs:
        ws = torch.full((Hq * pairs * 8192,), 0xFF, dtype=torch.uint8, device=q.device)  # NaN
        a.ds_workspace, a.ds_capacity = ws.data_ptr(), pairs
    _bam_hip.call("bam_attn_bwd", ctypes.byref(a), stream)
    torch.cuda.synchronize()
    return o, lse, *grads


@pytest.mark.parametrize("bias_rows", [None, 1, "S"])
@pytest.mark.parametrize("D,handover", [(32, False), (40, False), (64, False), (96, True), (128, False), (128, True)])
@pytest.mark.parametrize("S", [20, 33, 64, 200, 517, 1100])  # (with one key the gradients of q and k are rounding noise around 0)
def test_attention_does_not_depend_on_the_order_of_the_rows(S, D, handover, bias_rows):
    B, Hq, Hkv = 2, 4, 2
    g = torch.Generator(device=dev()).manual_seed(S + D)
    q, k, v, do = (torch.randn(B, S, H, D, generator=g, device=dev()).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(B, S, seed=S, pad=S // 9)
    bf[1] = random_bitfield(1, S, seed=S)[0] | 1  # all text: a sequence whose rows stay where they are, beside one whose rows move
    bf = bf.to(dev())
    bias = None
    if bias_rows is not None:
        bias = torch.randn(1, Hq, S if bias_rows == "S" else 1, S, generator=g, device=dev())
    flags, plan, ws, pairs = sorted_plan(bf)
    got = attention(q, k, v, do, bf, flags, plan, pairs if handover else 0, bias, D**-0.5)
    want = attention(q, k, v, do, bf, flags, None, 0, bias, D**-0.5)
    names = ("o", "lse", "dq", "dk", "dv")
    for name, a, b in zip(names, got, want):
        if name == "lse":
            a, b = a[..., :S], b[..., :S]  # (rows past the end hold whatever a row without keys gets)
            assert torch.equal(torch.isfinite(a), torch.isfinite(b))
            a, b = a[torch.isfinite(a)], b[torch.isfinite(b)]
            assert (a - b).abs().max() <= 2.0**-8
            continue
        # other rows of a wave decide when its running maximum moves, against which P is rounded to bf16 (2^-9 a term)
        assert torch.isfinite(a).all() and rel_l2(a.float(), b.float()) <= 2.0**-8, name


@pytest.mark.parametrize("S,D", [(32768, 64), (32900, 128)])
def test_the_public_function_takes_it_from_32768_tokens_on(S, D):
    Hq, Hkv = 2, 1
    below = random_bitfield(1, 32767, seed=1).to(dev())
    assert not BA.BitfieldUtils.plan_for(BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(below), below).struct.rows
    g = torch.Generator(device=dev()).manual_seed(S)
    q, k, v, do = (torch.randn(1, S, H, D, generator=g, device=dev()).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(1, S, seed=1).to(dev())
    for start in range(0, S - 100, 307):  # many short segments
        bf[0, start : start + 100] = 1 << (1 + start // 307 % 5)
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    BA.BitfieldUtils.clear_cache()
    o = BA.bitfield_attn_func(q, k, v, bf)
    grads = torch.autograd.grad(o, (q, k, v), do)
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    plan = BA.BitfieldUtils.plan_for(flags, bf)
    assert plan.struct.rows and not plan.struct.row_workloads
    classes = array(plan.workspace, plan.struct.fine, (-(-S // 128) * 4, plan.struct.fine_stride_s), torch.uint8)
    columns = torch.nn.functional.pad(classes[:, : -(-S // 32)], (0, -(-(-S // 32)) % 4)).reshape(classes.shape[0], -1, 4)
    assert plan.ds_pairs() == int((columns != 0).any(-1).sum())  # (the count word says more than the count)
    assert torch.equal(BA.BitfieldUtils.nonempty_tiles_per_row_block(flags), torch.sum(flags > 0, dim=(0, 2)))
    want = attention(q.detach(), k.detach(), v.detach(), do, bf, flags, None, 0, None, D**-0.5)
    for a, b in zip((o, *grads), (want[0], *want[2:])):
        assert rel_l2(a.float(), b.float()) <= 2.0**-8
    BA.BitfieldUtils.clear_cache()


def test_a_sorted_plan_is_for_bitfield_attention_only():
    S, D = 64, 64
    q, k, v = (torch.randn(1, S, 1, D, device=dev()).bfloat16() for _ in range(3))
    bf = random_bitfield(1, S, seed=1).to(dev())
    flags, plan, ws, _ = sorted_plan(bf)
    a = _bam_hip.Attn()
    o, lse = torch.empty_like(q), torch.empty((1, 1, 128), device=dev())
    for name, t in zip("qkvo", (q, k, v, o)):
        setattr(a, name, _bam_hip.TensorArg(t.data_ptr(), *t.stride()[:3]))
    mask = torch.ones(1, S, S, dtype=torch.bool, device=dev())
    a.lse, a.mask, a.mode, a.plan = lse.data_ptr(), mask.data_ptr(), 2, ctypes.pointer(plan)
    a.flags, a.flags_stride_b, a.flags_stride_m = flags.data_ptr(), flags.stride(0), flags.stride(1)
    a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D, a.dtype, a.scale = 1, S, S, 1, 1, D, BA._dtype_code(q.dtype), 1.0
    with pytest.raises(_bam_hip.BamError, match="sorted rows"):
        _bam_hip.call("bam_attn_fwd", ctypes.byref(a), BA._stream_ptr(dev()))
