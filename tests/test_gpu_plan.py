"""The plan (classes of 32 x 32 tiles + slice order) the kernels use to skip masked work: its contents
against a brute-force classification of the oracle's mask, and the attention results with and without it."""

import ctypes
import math
import weakref

import pytest
import torch
import torch.nn.functional as F

from cornstarch_amd import workloads as W
from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def build_plan(bf):
    """flags, fine (B, slots, num_n) and order (B, slots) of a bitfield tensor on the device."""
    BA.BitfieldUtils.clear_cache()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    plan = BA.BitfieldUtils.plan_for(flags, bf)
    assert plan is not None
    fine, order = plan.fine_classes(), plan.slice_order()
    torch.cuda.synchronize()
    return flags, fine.clone(), order.clone(), plan


def flags_only(bf):
    """The flags through bam_tile_flags, the entry point that builds no plan (same kernel, other instantiation)."""
    B, S = bf.shape
    out = torch.empty((B, -(-S // 128), -(-S // 32)), dtype=torch.int8, device=bf.device)
    _bam_hip.call("bam_tile_flags", bf.data_ptr(), bf.stride(0), out.data_ptr(), out.stride(0), out.stride(1), B, S,
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out


def brute_force_fine(mask, S):
    """Class of every 32 x 32 tile from the (B, S, S) bool mask: 0 nothing allowed, 2 every in-range cell."""
    B = mask.shape[0]
    n = -(-S // 32)
    pad = n * 32 - S
    m = F.pad(mask, (0, pad, 0, pad))
    cnt = m.view(B, n, 32, n, 32).sum(dim=(2, 4))
    cells = F.pad(torch.ones_like(mask), (0, pad, 0, pad)).view(B, n, 32, n, 32).sum(dim=(2, 4))
    return torch.where(cnt == 0, 0, torch.where(cnt == cells, 2, 1)).to(torch.uint8)


@pytest.mark.parametrize("S", [1, 31, 57, 128, 144, 283, 1000])
@pytest.mark.parametrize("wide", [False, True])
def test_fine_classes_and_order_on_irregular_bitfields(S, wide):
    bf = random_bitfield(3, S, seed=S, pad=min(5, S - 1), wide=wide)
    flags, fine, order, _ = build_plan(bf.to(dev()))
    assert torch.equal(flags.cpu(), O.tile_flags(bf))  # the public flags are what they were
    n = -(-S // 32)
    want = brute_force_fine(O.materialize_mask(bf), S)
    assert torch.equal(fine[:, :n].cpu(), want)
    assert (fine[:, n:] == 0).all()  # slots past the last row slice need nothing
    for b in range(3):
        o = order[b].cpu().tolist()
        assert sorted(o[:n]) == list(range(n)) and all(x == -1 for x in o[n:])
        # slices holding a text row come first, latest first; modality-only slices are grouped by modality
        rows = F.pad(bf[b], (0, n * 32 - S)).view(n, 32)
        text = ((rows & 1) != 0).any(dim=1)
        sig = torch.zeros(n, dtype=torch.int64)
        for r in range(32):
            sig |= rows[:, r] & ((1 << 62) - 1)
        nt = int(text.sum())
        assert all(text[s] for s in o[:nt]) and o[:nt] == sorted(o[:nt], reverse=True)
        rest = o[nt:n]
        groups = [int(sig[s]) for s in rest]
        assert groups == sorted(groups)
        for gval in set(groups):
            members = [s for s in rest if int(sig[s]) == gval]
            assert members == sorted(members)


@pytest.mark.parametrize("S", [33, 96, 129, 500, 1111])
@pytest.mark.parametrize("max_run", [1, 3])
def test_classes_when_the_bitfield_changes_every_few_rows(S, max_run):
    # up to 32 runs of equal bitfields inside one 32-row slice: text, five modalities (one above bit 31) and 0, at random
    g = torch.Generator().manual_seed(1000 * S + max_run)
    text = (1 << 62) | 1 | (1 << 3) | (1 << 40)
    values = torch.tensor([text, 1 << 1, 1 << 2, 1 << 3, 1 << 4, 1 << 40, 0], dtype=torch.int64)
    bf = torch.empty((2, S), dtype=torch.int64)
    for b in range(2):
        pos = 0
        while pos < S:
            run = int(torch.randint(1, max_run + 1, (1,), generator=g))
            bf[b, pos : pos + run] = values[int(torch.randint(0, len(values), (1,), generator=g))]
            pos += run
    flags, fine, order, _ = build_plan(bf.to(dev()))
    assert torch.equal(flags.cpu(), O.tile_flags(bf))
    assert torch.equal(flags_only(bf.to(dev())).cpu(), O.tile_flags(bf))  # the kernel form that writes no classes
    n = -(-S // 32)
    assert torch.equal(fine[:, :n].cpu(), brute_force_fine(O.materialize_mask(bf), S))
    for b in range(2):
        o = order[b].cpu().tolist()
        assert sorted(o[:n]) == list(range(n)) and all(x == -1 for x in o[n:])


@pytest.mark.parametrize("B,S", [(1, 1000), (3, 700), (8, 4096), (5, 129), (700, 300)])  # up to 2100 groups / tiles
def test_groups_of_slices_are_ranked_by_the_length_of_their_tile_lists(B, S):
    # group_order: codes b * num_m + group of ALL sequences, by falling number of 64-key tiles the group's four
    # slices visit together (ties: lower code first)
    bf = random_bitfield(B, S, seed=7 * B + S, pad=S // 9)
    _, fine, order, plan = build_plan(bf.to(dev()))
    got = plan.group_order()
    num_m, n64 = -(-S // 128), -(-S // 64)
    assert got is not None and got.shape == (B * num_m,)
    fine, order = fine.cpu(), order.cpu()
    weight = []
    for b in range(B):
        cls = F.pad(fine[b], (0, 2 * n64 - fine.shape[2])).view(fine.shape[1], n64, 2).amax(dim=2) > 0
        for grp in range(num_m):
            rows = [int(s) for s in order[b, 4 * grp : 4 * grp + 4] if s >= 0]
            weight.append(int(cls[rows].any(dim=0).sum()) if rows else 0)
    want = sorted(range(B * num_m), key=lambda c: (-weight[c], c))
    assert got.cpu().tolist() == want
    # the key tiles of the same plan, ranked by the number of slices that list them (what dK/dV goes by)
    nkt = -(-S // 128)
    has = (F.pad(fine, (0, 4 * nkt - fine.shape[2])).view(B, fine.shape[1], nkt, 4) != 0).any(dim=3)
    counts = has.sum(dim=1).reshape(-1).tolist()
    st, ws = plan.struct, plan.workspace
    tile_order = torch.as_strided(ws.view(torch.int32), (B * nkt,), (1,), (st.ds_tile_order - ws.data_ptr()) // 4)
    assert tile_order.cpu().tolist() == sorted(range(B * nkt), key=lambda c: (-counts[c], c))


@pytest.mark.parametrize("name", ["C1", "C2", "C4"])
def test_fine_classes_on_the_benchmark_workloads(name):
    bf = W.make_bitfields(name).to(dev())
    flags, fine, order, _ = build_plan(bf)
    S = bf.shape[1]
    n = S // 32
    want = torch.cat([brute_force_fine(O.materialize_mask(bf[b : b + 1]), S) for b in range(bf.shape[0])])
    assert torch.equal(fine[:, :n], want)
    # a 128 x 32 flag is the summary of its four row slices
    f4 = fine[:, :n].view(bf.shape[0], n // 4, 4, n)
    derived = torch.where((f4 == 0).all(dim=2), 0, torch.where((f4 == 2).all(dim=2), 2, 1)).to(torch.int8)
    assert torch.equal(derived, flags)


def _run(q, k, v, do, bf, flags, plan, scale):
    """forward + both backward kernels through the launch helpers, with or without a plan"""
    B, S, Hq, D = q.shape
    with torch.cuda.device(q.device):
        o = torch.empty_like(q)
        # every row of the rounded lse is the kernel's to write, with or without a plan (what the rows past the end
        # of the sequence hold is unspecified, as in the reference, but it is never left-over memory): start from NaN
        lse = torch.full((B, Hq, flags.shape[1] * 128), float("nan"), dtype=torch.float32, device=q.device)
        _bam_hip.call(
            "bam_fwd", q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), bf.data_ptr(),
            flags.data_ptr(), *BA._strides3(q, k, v, o), bf.stride(0), flags.stride(0), flags.stride(1),
            B, S, Hq, k.shape[2], D, float(scale), BA._dtype_code(q.dtype), None,
            plan.byref() if plan is not None else None, BA._stream_ptr(q.device),
        )
    delta = torch.empty_like(lse)
    BA._launch_bwd_preprocess(o, do, delta)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    BA._launch_bwd_dkdv(q, k, v, do, lse, delta, dk, dv, bf, flags, scale, accumulate=False, plan=plan)
    BA._launch_bwd_dq(q, k, v, do, lse, delta, dq, bf, flags, scale, accumulate=False, plan=plan)
    torch.cuda.synchronize()
    assert not torch.isnan(lse).any()
    return o, lse[:, :, :S], dq, dk, dv


@pytest.mark.parametrize("B,S,Hq,Hkv,D", [(2, 517, 4, 2, 128), (1, 1000, 4, 4, 64), (3, 200, 2, 1, 32), (1, 2048, 8, 2, 128), (2, 97, 2, 2, 64)])
def test_results_do_not_depend_on_the_plan(B, S, Hq, Hkv, D):
    d = dev()
    bf = random_bitfield(B, S, seed=S + D, pad=7).to(d)
    g = torch.Generator().manual_seed(S)
    q = (torch.randn(B, S, Hq, D, generator=g) * 0.5).bfloat16().to(d)
    k = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
    v = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
    do = torch.randn(B, S, Hq, D, generator=g).bfloat16().to(d)
    flags, _, _, plan = build_plan(bf)
    scale = 1.0 / math.sqrt(D)
    with_plan = _run(q, k, v, do, bf, flags, plan, scale)
    without = _run(q, k, v, do, bf, flags, None, scale)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), with_plan, without):
        if name in ("dk", "dv"):  # the two row streams add their fp32 partial sums in another order
            assert rel_l2(a.float(), b.float()) <= 2e-3, name
        else:
            assert torch.equal(a, b), name
    o_ref, lse_ref = O.attention_forward(q, k, v, bf)
    assert (with_plan[0].float() - o_ref).abs().max().item() <= 2e-2
    live = torch.isfinite(lse_ref)
    assert torch.equal(torch.isfinite(with_plan[1]), live)
    assert (with_plan[1][live] - lse_ref[live]).abs().max().item() <= 1e-2
    for got, want in zip(with_plan[2:], O.attention_backward(q, k, v, bf, do)):
        assert rel_l2(got.float(), want) <= 5e-2
    BA.BitfieldUtils.clear_cache()


def test_batches_with_more_groups_or_key_tiles_than_are_ranked_run_without_the_rankings():
    # 4200 sequences of 130 rows: 8400 groups of slices and 8400 key tiles, more than the rankings cover (8192); the
    # kernels then walk them in their natural order and the results are what they are without a plan
    d = dev()
    B, S, Hq, Hkv, D = 4200, 130, 2, 1, 32
    bf = random_bitfield(B, S, seed=5, pad=3).to(d)
    g = torch.Generator().manual_seed(5)
    q = (torch.randn(B, S, Hq, D, generator=g) * 0.5).bfloat16().to(d)
    k = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
    v = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
    do = torch.randn(B, S, Hq, D, generator=g).bfloat16().to(d)
    flags, _, _, plan = build_plan(bf)
    assert plan.group_order() is None and not plan.struct.ds_tile_order
    scale = 1.0 / math.sqrt(D)
    with_plan = _run(q, k, v, do, bf, flags, plan, scale)
    without = _run(q, k, v, do, bf, flags, None, scale)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), with_plan, without):
        if name in ("dk", "dv"):
            assert rel_l2(a.float(), b.float()) <= 2e-3, name
        else:
            assert torch.equal(a, b), name
    sub = slice(0, 16)  # the oracle on a few of the sequences
    o_ref, _ = O.attention_forward(q[sub], k[sub], v[sub], bf[sub])
    assert (with_plan[0][sub].float() - o_ref).abs().max().item() <= 2e-2
    BA.BitfieldUtils.clear_cache()


def test_two_host_threads_with_different_masks_share_the_caches():
    # the flag / plan cache is one per process: two threads that alternate between their own masks must each get
    # their own results, bit for bit what a single thread gets
    import threading

    d = dev()
    jobs = []
    for t, (B, S, Hq, Hkv, D) in enumerate([(2, 700, 4, 2, 128), (1, 900, 4, 4, 128)]):
        g = torch.Generator().manual_seed(100 + t)
        q = (torch.randn(B, S, Hq, D, generator=g) * 0.5).bfloat16().to(d)
        k = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
        v = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).bfloat16().to(d)
        do = torch.randn(B, S, Hq, D, generator=g).bfloat16().to(d)
        bf = random_bitfield(B, S, seed=200 + t, pad=5).to(d)
        jobs.append((q, k, v, do, bf))

    def step(job):
        q, k, v, do, bf = job
        qg, kg, vg = (x.clone().requires_grad_(True) for x in (q, k, v))
        o = BA.bitfield_attn_func(qg, kg, vg, bf)
        grads = torch.autograd.grad(o, (qg, kg, vg), do)
        torch.cuda.synchronize()
        return [o.detach()] + list(grads)

    want = [step(job) for job in jobs]
    errors = []

    def worker(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(6):
                    got = step(jobs[i])
                    for name, a, b in zip(("o", "dq", "dk", "dv"), got, want[i]):
                        # (when the other thread has replaced the cached plan between this thread's flag lookup and
                        # its kernels, these run from the flags alone: same o; dk / dv summed in another order, dq
                        # from recomputed instead of stored dS, i.e. equal up to the last bit)
                        if name == "o":
                            assert torch.equal(a, b), name
                        else:
                            assert rel_l2(a.float(), b.float()) <= 2e-3, (name, rel_l2(a.float(), b.float()))
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors
    BA.BitfieldUtils.clear_cache()


def test_a_mask_whose_end_looks_up_other_flags():
    # the cache lets go of the previous mask when it takes a new one; a finalizer of that mask may itself use the cache
    old, new, other = (random_bitfield(1, S, seed=S) for S in (500, 300, 200))
    newd, otherd = new.to(dev()), other.to(dev())
    g = torch.Generator().manual_seed(0)
    q, k, v = ((torch.randn(1, 300, H, 64, generator=g) * 0.5).bfloat16().to(dev()) for H in (4, 2, 2))
    BA.BitfieldUtils.clear_cache()
    want = BA.bitfield_attn_func(q, k, v, newd)
    seen = []

    def remember():
        mask = old.to(dev())
        BA.BitfieldUtils.clear_cache()
        BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(mask)
        weakref.finalize(mask, lambda: seen.append(BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(otherd)))

    remember()
    got = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(newd)
    assert len(seen) == 1 and torch.equal(got.cpu(), O.tile_flags(new)) and torch.equal(seen[0].cpu(), O.tile_flags(other))
    remember()
    assert torch.equal(BA.bitfield_attn_func(q, k, v, newd), want) and len(seen) == 2
    BA.BitfieldUtils.clear_cache()


def test_a_plan_of_another_problem_is_refused():
    d = dev()
    bf = random_bitfield(1, 256, seed=1).to(d)
    flags, _, _, plan = build_plan(bf)
    q = torch.zeros(1, 128, 2, 64, dtype=torch.bfloat16, device=d)
    bf2 = bf[:, :128].contiguous()
    fl2 = torch.zeros(1, 1, 4, dtype=torch.int8, device=d)
    o = torch.empty_like(q)
    lse = torch.empty(1, 2, 128, device=d)
    with pytest.raises(_bam_hip.BamError, match="plan was built for"):
        _bam_hip.call(
            "bam_fwd", q.data_ptr(), q.data_ptr(), q.data_ptr(), o.data_ptr(), lse.data_ptr(), bf2.data_ptr(),
            fl2.data_ptr(), *BA._strides3(q, q, q, o), bf2.stride(0), fl2.stride(0), fl2.stride(1),
            1, 128, 2, 2, 64, 0.125, BA._dtype_code(q.dtype), None, plan.byref(), BA._stream_ptr(d),
        )
    # caller-provided flags (not the cached tensor) never pick up the cached plan
    assert BA.BitfieldUtils.plan_for(flags.clone(), bf) is None
    assert BA.BitfieldUtils.plan_for(flags, bf) is plan
    BA.BitfieldUtils.clear_cache()
    assert BA.BitfieldUtils.plan_for(flags, bf) is None


@pytest.mark.parametrize("S,Hq", [(1024, 8), (1500, 20), (1100, 32)])  # one launch by the sizes, by the count; a dS workspace
def test_a_plan_whose_count_never_arrives_is_refused(S, Hq):
    """The word that the count is stored to is cleared on the host, as if the last launch of the plan builder had failed: every
    backward that takes such a plan for a hand-over of dS, or may take it for one, raises once the stream has run dry."""
    bf = random_bitfield(1, S, seed=S, pad=3).to(dev())
    flags, _, _, plan = build_plan(bf)
    q, k, v, do = (torch.randn(1, S, Hq, 128, device=dev(), dtype=torch.bfloat16) for _ in range(4))
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags)
    torch.cuda.synchronize()
    # (the word's address and tag follow the bam_plan inside the plan object; the tag is in the word's upper half)
    behind = ctypes.addressof(plan.struct) + ctypes.sizeof(_bam_hip.Plan)
    tag = ctypes.c_uint32.from_address(behind + 8).value
    word = ctypes.c_uint64.from_address(ctypes.c_uint64.from_address(behind).value)
    stored = word.value
    assert stored >> 32 == tag
    try:
        word.value = 0
        with pytest.raises(_bam_hip.BamError, match="pair count of a plan never arrived"):
            BA._bitfield_attn_backward_overwrite(do, q, k, v, o, bf, flags, lse, scale)
    finally:
        word.value = stored
    got = BA._bitfield_attn_backward_overwrite(do, q, k, v, o, bf, flags, lse, scale)
    assert plan.ds_pairs() == stored & 0xFFFFFFFF and all(torch.isfinite(g).all() for g in got)
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("B,S,H,D", [(1, 100, 2, 128), (2, 283, 4, 64), (1, 700, 4, 128), (36, 129, 32, 64)])  # the last: four-wave dK/dV
@pytest.mark.parametrize("offset", [0, 1])
def test_classes_laid_out_by_the_caller(B, S, H, D, offset):
    """Rows of ceil(S/32) class bytes without padding, at any address: dK/dV must not read them as words.  Bytes around them say
    "full", the results are those of the builder's rows of 16-byte multiples."""
    bf = random_bitfield(B, S, seed=S, pad=3).to(dev())
    flags, fine, _, plan = build_plan(bf)
    slots, num_n = 4 * flags.shape[1], fine.shape[2]
    assert fine.shape[1] == slots
    room = torch.full((fine.numel() + 64,), 2, dtype=torch.uint8, device=dev())
    room[16 + offset : 16 + offset + fine.numel()] = fine.reshape(-1)
    own = _bam_hip.Plan.from_buffer_copy(plan.struct)
    own.fine, own.fine_stride_b, own.fine_stride_s = room.data_ptr() + 16 + offset, slots * num_n, num_n

    class Own:
        def byref(self):
            return ctypes.byref(own)

    q, k, v, do = (torch.randn(B, S, H, D, device=dev(), dtype=torch.bfloat16) for _ in range(4))
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, flags)
    delta = torch.empty_like(lse)
    BA._launch_bwd_preprocess(o, do, delta)
    got = []
    for p in (plan, Own()):
        got.append((torch.empty_like(k), torch.empty_like(v)))
        BA._launch_bwd_dkdv(q, k, v, do, lse, delta, *got[-1], bf, flags, scale, accumulate=False, plan=p)
    torch.cuda.synchronize()
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and torch.equal(a, b)
    BA.BitfieldUtils.clear_cache()
