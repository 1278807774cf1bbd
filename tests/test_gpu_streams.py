"""Cached flags, plans and gathered index arrays used on another stream than the one that computes them, and by graphs.  The first stream is kept
busy (`_sleep`), so that the launches that fill them are still queued when the second stream's call is made."""

import time

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel.attention import _MaskPlan, flash_attn_func
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu

BUSY = 40_000_000  # cycles: some 20 ms
B, S, HQ, HKV, D = 2, 700, 8, 2, 128


def _inputs():
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v, do = (torch.randn(B, S, h, D, generator=g, device="cuda").bfloat16() for h in (HQ, HKV, HKV, HQ))
    return q, k, v, do, random_bitfield(B, S, seed=9, pad=40).cuda()


def _forget():
    BA.BitfieldUtils.clear_cache()
    _MaskPlan.forget()


def _bitfield(q, k, v, do, bf):
    x = [t.detach().requires_grad_(True) for t in (q, k, v)]
    o = BA.bitfield_attn_func(*x, bf)
    return o.detach(), *torch.autograd.grad(o, x, do)


def _flags_and_plan(q, k, v, do, bf):
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    assert BA.BitfieldUtils.plan_for(flags, bf) is not None
    return BA._bitfield_attn_forward(q, k, v, bf, flags)[:2]


def _mask(q, k, v, do, bf):
    x = [t.detach().requires_grad_(True) for t in (q, k, v)]
    o = flash_attn_func(*x, mask=_mask.of)
    return o.detach(), *torch.autograd.grad(o, x, do)


def _indexed(q, k, v, do, bf):
    o, lse, scale = BA._bitfield_attn_forward(q, k, v, bf, _indexed.flags, _indexed.rows, _indexed.rows)
    grads = [torch.zeros(t.shape, device=t.device) for t in (q, k, v)]
    BA._bitfield_attn_backward(do, q, k, v, o, bf, _indexed.flags, lse, *grads, _indexed.rows, _indexed.rows, softmax_scale=scale)
    return o, *grads


CALLS = [_bitfield, _flags_and_plan, _mask, _indexed]


@pytest.fixture
def inputs():
    x = _inputs()
    _mask.of = BA.materialize_bitfield_mask(x[4])
    _indexed.rows = torch.arange(S, device="cuda")
    _indexed.flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(x[4]).clone()
    torch.cuda.synchronize()
    yield x
    torch.cuda.synchronize()
    _forget()


def _external():
    return torch.cuda.ExternalStream(torch.cuda.Stream().cuda_stream)  # (a stream that torch takes for the program's own)


STREAMS = {
    "default to side": (torch.cuda.default_stream, torch.cuda.Stream),
    "side to default": (torch.cuda.Stream, torch.cuda.default_stream),
    "side to side": (torch.cuda.Stream, torch.cuda.Stream),
    "external to side": (_external, torch.cuda.Stream),
    "side to external": (torch.cuda.Stream, _external),
}


@pytest.mark.parametrize("call", CALLS, ids=lambda f: f.__name__)
@pytest.mark.parametrize("streams", STREAMS)
def test_a_hit_on_another_stream_waits_for_what_it_uses(inputs, call, streams):
    first, second = (make() for make in STREAMS[streams])
    want = call(*inputs)
    torch.cuda.synchronize()
    for _ in range(2):
        _forget()
        with torch.cuda.stream(first):
            torch.cuda._sleep(BUSY)
            call(*inputs)
        with torch.cuda.stream(second):
            got = call(*inputs)
            again = call(*inputs)
        torch.cuda.synchronize()
        for a, b, c in zip(want, got, again):
            assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("call", CALLS, ids=lambda f: f.__name__)
def test_memory_of_a_dropped_entry_is_not_reused_before_another_stream_is_done(inputs, call):
    want = call(*inputs)
    _forget()
    call(*inputs)  # the entry: computed on the default stream
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(BUSY)
        got = call(*inputs)
    _forget()
    junk = [torch.full((n,), 255, dtype=torch.uint8, device="cuda") for n in (1 << 10, 1 << 12, 1 << 14, 1 << 16, 1 << 18) for _ in range(16)]
    torch.cuda.synchronize()
    del junk
    for a, b in zip(want, got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("call", [_flags_and_plan, _mask, _indexed], ids=lambda f: f.__name__)
@pytest.mark.parametrize("streams", ["default to side", "side to side", "external to side"])
def test_a_capture_finds_finished_plans_only(inputs, call, streams):
    first, second = (make() for make in STREAMS[streams])
    want = call(*inputs)
    with torch.cuda.stream(second):  # (first use of whatever a capture must not set up)
        call(*inputs)
    torch.cuda.synchronize()
    _forget()
    with torch.cuda.stream(first):
        call(*inputs)
        torch.cuda.synchronize()
        _forget()
        torch.cuda._sleep(BUSY)
        call(*inputs)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(second):
        graph.capture_begin()
        try:
            got = call(*inputs)
        finally:
            graph.capture_end()
    for _ in range(3):
        with torch.cuda.stream(second):
            graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(want, got):
            assert torch.equal(a, b)
            b.zero_()
        torch.cuda.synchronize()


def _until(done):
    """The runtime may let go of a destroyed graph from a thread of its own."""
    for _ in range(500):
        if done():
            return
        time.sleep(0.01)
    assert done()


@pytest.mark.parametrize("call", CALLS, ids=lambda f: f.__name__)
def test_a_graph_owns_the_plans_it_reads(inputs, call):
    """The caches hold one entry each: what a graph was captured with stays its own, and goes when the graph goes."""
    from cornstarch_amd.kernel._bam_hip import host

    want = call(*inputs)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    before = host.held_by_graphs()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(*inputs)
        got = call(*inputs)  # a second layer
    assert host.held_by_graphs() == before + 1
    kept = _mask.of, _indexed.flags, _indexed.rows
    for other in (S, S // 2):  # other masks take the entries, their memory and that of the old ones
        q, k, v, do = (t[:, :other].contiguous() for t in inputs[:4])
        bf = torch.flip(inputs[4], (1,))[:, :other].contiguous()
        _mask.of = BA.materialize_bitfield_mask(bf)
        _indexed.rows = torch.arange(other, device="cuda")
        _indexed.flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf).clone()
        call(q, k, v, do, bf)
        junk = [torch.full((n,), 255, dtype=torch.uint8, device="cuda") for n in (1 << 10, 1 << 12, 1 << 14, 1 << 16, 1 << 18) for _ in range(16)]
        torch.cuda.synchronize()
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(want, got):
            assert torch.equal(a, b)
        del junk
    _mask.of, _indexed.flags, _indexed.rows = kept
    del graph
    _until(lambda: host.held_by_graphs() == before)


def test_an_entry_made_anew_is_owned_by_the_next_graph(inputs):
    from cornstarch_amd.kernel._bam_hip import host

    want = _flags_and_plan(*inputs)
    before, graphs = host.held_by_graphs(), []
    for _ in range(3):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            got = _flags_and_plan(*inputs)
    assert host.held_by_graphs() == before + 3
    _forget()
    del graphs[:2]
    _until(lambda: host.held_by_graphs() == before + 1)
    graphs[0].replay()
    torch.cuda.synchronize()
    for a, b in zip(want, got):
        assert torch.equal(a, b)


def test_a_backward_up_to_head_dim_64_does_not_wait_for_the_gpu():
    """Sorted rows (32768 tokens on) are launched as they come: the host does not need to know whether they were moved."""
    n, h, d = 32768, 1, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    x = [torch.randn(1, n, h, d, generator=g, device="cuda").bfloat16().requires_grad_(True) for _ in range(3)]
    do = torch.randn(1, n, h, d, generator=g, device="cuda").bfloat16()
    bf = random_bitfield(1, n, seed=4).cuda()

    def step():
        _forget()
        return torch.autograd.grad(BA.bitfield_attn_func(*x, bf), x, do)

    want = step()
    torch.cuda.synchronize()
    held = torch.cuda.Event()
    torch.cuda._sleep(20 * BUSY)
    held.record()
    got = step()
    waited = held.query()
    torch.cuda.synchronize()
    assert not waited
    for a, b in zip(want, got):
        assert torch.equal(a, b)
    _forget()


@pytest.mark.parametrize("indexed", [False, True])
def test_what_a_capture_computes_stays_out_of_the_caches(indexed):
    """Beyond 131072 rows there is no plan, so flags and index views can be made in a capture: in the graph's memory, by its replays."""
    n = 131200
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(1, rows, 1, 32, generator=g, device="cuda").bfloat16() for rows in (n, 256, 256))
    bf = torch.full((1, n), 2, dtype=torch.int64, device="cuda")
    bf[:, ::40000] = (1 << 62) | 3
    rows = torch.arange(n, device="cuda")

    def call():
        if not indexed:
            return BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
        view = BA._IndexView.get(bf, rows, rows[:256])
        assert view.plan is None
        flags = torch.full((1, -(-n // 128), 8), 1, dtype=torch.int8, device="cuda")
        return BA._bitfield_attn_forward(q, k, v, bf, flags, rows, rows[:256])[0]

    want = call().clone()
    torch.cuda.synchronize()
    _forget()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    eager = call()  # nothing has been replayed yet
    torch.cuda.synchronize()
    assert torch.equal(eager, want)
    for _ in range(3):
        got.zero_()
        _forget()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    _forget()
