"""The C ABI under HIP graph capture: the library allocates nothing, synchronizes nothing and uses only the stream it
is handed, so a whole step -- flags + plan, forward, delta, dK/dV + dQ with the dS hand-over -- can be recorded once
and replayed.  Every replay is compared, bit for bit, with the same entry points called eagerly on the same inputs;
the replays are separated by eager work and synchronizations of the program itself."""

import ctypes
import math

import pytest
import torch

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel.interface import bitfield_attention_forward
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def make_inputs(B, S, Hq, Hkv, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(B, S, Hq, D, generator=g) * 0.5).to(dtype)
    k = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).to(dtype)
    v = (torch.randn(B, S, Hkv, D, generator=g) * 0.5).to(dtype)
    do = torch.randn(B, S, Hq, D, generator=g).to(dtype)
    return q, k, v, do


class _Step:
    """Static buffers of one fwd+bwd step and the five C ABI calls that make it, on a given stream."""

    def __init__(self, B, S, Hq, Hkv, D, dtype, pairs_capacity):
        d = dev()
        self.shape = (B, S, Hq, Hkv, D)
        self.q, self.k, self.v, self.do = (torch.zeros(s, dtype=dtype, device=d)
                                           for s in ((B, S, Hq, D), (B, S, Hkv, D), (B, S, Hkv, D), (B, S, Hq, D)))
        self.bf = torch.zeros((B, S), dtype=torch.int64, device=d)
        self.flags = torch.zeros((B, -(-S // 128), -(-S // 32)), dtype=torch.int8, device=d)
        lib = _bam_hip.load()
        self.plan_ws = torch.zeros((lib.bam_plan_workspace_bytes(B, S),), dtype=torch.uint8, device=d)
        self.plan = _bam_hip.Plan()
        self.o = torch.zeros_like(self.q)
        self.lse = torch.zeros((B, Hq, -(-S // 128) * 128), dtype=torch.float32, device=d)
        self.delta = torch.zeros_like(self.lse)
        self.dq, self.dk, self.dv = torch.zeros_like(self.q), torch.zeros_like(self.k), torch.zeros_like(self.v)
        self.pairs_capacity = pairs_capacity
        nbytes = lib.bam_ds_workspace_bytes(Hq, pairs_capacity) if D == 128 else 0
        self.ds_ws = torch.zeros((max(nbytes, 16),), dtype=torch.uint8, device=d)
        self.use_ds = nbytes > 0

    def load(self, q, k, v, do, bf):
        for dst, src in ((self.q, q), (self.k, k), (self.v, v), (self.do, do), (self.bf, bf)):
            dst.copy_(src)

    def enqueue(self, stream):
        B, S, Hq, Hkv, D = self.shape
        st = stream.cuda_stream
        scale = 1.0 / math.sqrt(D)
        code = BA._dtype_code(self.q.dtype)
        _bam_hip.call("bam_tile_plan", self.bf.data_ptr(), self.bf.stride(0), self.flags.data_ptr(), self.flags.stride(0),
                      self.flags.stride(1), self.plan_ws.data_ptr(), self.plan_ws.numel(), B, S, ctypes.byref(self.plan), st)
        if self.use_ds:  # the caller's part of the plan: where dK/dV leaves dS for dQ
            self.plan.ds_workspace = self.ds_ws.data_ptr()
            self.plan.ds_capacity = self.pairs_capacity
        _bam_hip.call("bam_fwd", self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.o.data_ptr(),
                      self.lse.data_ptr(), self.bf.data_ptr(), self.flags.data_ptr(),
                      *BA._strides3(self.q, self.k, self.v, self.o), self.bf.stride(0), self.flags.stride(0),
                      self.flags.stride(1), B, S, Hq, Hkv, D, scale, code, None, ctypes.byref(self.plan), st)
        _bam_hip.call("bam_bwd_preprocess", self.o.data_ptr(), self.do.data_ptr(), self.delta.data_ptr(),
                      *BA._strides3(self.o, self.do), B, S, Hq, D, code, st)
        _bam_hip.call("bam_bwd", self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.do.data_ptr(),
                      self.lse.data_ptr(), self.delta.data_ptr(), self.dq.data_ptr(), self.dk.data_ptr(), self.dv.data_ptr(),
                      self.bf.data_ptr(), self.flags.data_ptr(),
                      *BA._strides3(self.q, self.k, self.v, self.do, self.dq, self.dk, self.dv), self.bf.stride(0),
                      self.flags.stride(0), self.flags.stride(1), B, S, Hq, Hkv, D, scale, code, 0, None,
                      ctypes.byref(self.plan), st)

    def results(self):
        return [t.clone() for t in (self.flags, self.o, self.lse, self.dq, self.dk, self.dv)]


@pytest.mark.parametrize("B,S,Hq,Hkv,D", [(2, 640, 8, 2, 128), (3, 333, 4, 4, 64)])
def test_a_recorded_step_replays_bit_for_bit(B, S, Hq, Hkv, D):
    dtype = torch.bfloat16
    # room for every (32-row slice, 128-key tile) pair: the count is device data and cannot be read during capture
    capacity = B * 4 * (-(-S // 128)) * (-(-S // 128))
    step = _Step(B, S, Hq, Hkv, D, dtype, capacity)
    cases = []
    for seed in (1, 2, 3):
        q, k, v, do = (t.to(dev()) for t in make_inputs(B, S, Hq, Hkv, D, dtype, seed=10 * seed + S))
        bf = random_bitfield(B, S, seed=seed + S, pad=7 * seed).to(dev())
        cases.append((q, k, v, do, bf))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # once eagerly on the capture stream (loads the code objects)
        step.load(*cases[0])
        step.enqueue(side)
    side.synchronize()

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        step.enqueue(side)

    for case in cases + cases[:1]:
        step.load(*case)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        replayed = step.results()
        # eager work of the program between the replays: the same step through the same entry points
        for t in (step.flags, step.o, step.lse, step.dq, step.dk, step.dv):
            t.zero_()
        step.enqueue(torch.cuda.current_stream())
        torch.cuda.synchronize()
        for name, a, b in zip(("flags", "o", "lse", "dq", "dk", "dv"), replayed, step.results()):
            assert torch.equal(a, b), name
        # and the replay is what the public entry point computes
        BA.BitfieldUtils.clear_cache()
        qg, kg, vg = (t.clone().requires_grad_(True) for t in case[:3])
        o = BA.bitfield_attn_func(qg, kg, vg, case[4])
        dq, dk, dv = torch.autograd.grad(o, (qg, kg, vg), case[3])
        torch.cuda.synchronize()
        assert torch.equal(replayed[1], o.detach())
        for a, b in zip(replayed[3:], (dq, dk, dv)):
            assert torch.equal(a, b)


def test_decode_first_seen_in_a_capture_leaves_eager_calls_alone():
    """A stream's merge counters are never made by a capture: replays and eager calls on the capture stream agree."""
    torch.manual_seed(3)
    q, k, v = (torch.randn(1, h, s, 128, device=dev(), dtype=torch.bfloat16) for h, s in ((8, 1), (2, 2100), (2, 2100)))
    module = torch.nn.Module().eval()
    want = bitfield_attention_forward(module, q, k, v, None)[0]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = bitfield_attention_forward(module, q, k, v, None)[0]
    for _ in range(3):
        with torch.cuda.stream(side):
            eager = bitfield_attention_forward(module, q, k, v, None)[0]
        torch.cuda.synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (eager.float() - want.float()).abs().max() == 0
        # two launches merge the same partial results here: equal up to the rounding of the output
        assert (out.float() - want.float()).abs().max() <= 2.0 ** -8 * want.float().abs().max()


def test_a_plan_is_not_built_by_a_capture():
    """A replay would store the pair count to a word that has another owner by then: refused before anything is launched."""
    q, k, v = (torch.randn(1, 200, 2, 64, device=dev(), dtype=torch.bfloat16) for _ in range(3))
    bf = torch.full((1, 200), (1 << 62) | 1, dtype=torch.int64, device=dev())
    BA.BitfieldUtils.clear_cache()
    want = BA.bitfield_attn_func(q, k, v, bf)  # also loads the code objects
    BA.BitfieldUtils.clear_cache()
    torch.cuda.synchronize()
    with pytest.raises(_bam_hip.BamError, match="captured"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            BA.bitfield_attn_func(q, k, v, bf)
    torch.cuda.synchronize()
    BA.bitfield_attn_func(q, k, v, bf)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = BA.bitfield_attn_func(q, k, v, bf)  # with the plan built before
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("S,Hq,Hkv,D", [(700, 8, 2, 64), (1024, 8, 8, 128), (1030, 8, 2, 96), (2048, 16, 16, 128)])
def test_the_one_launch_backward_in_a_capture(S, Hq, Hkv, D):
    """dK/dV and dQ in one launch (with parts; by the sizes, by the count), with a plan that was built before the capture."""
    q, k, v, do = (t.to(dev()).requires_grad_(n < 3) for n, t in enumerate(make_inputs(1, S, Hq, Hkv, D, torch.bfloat16, seed=S)))
    bf = random_bitfield(1, S, seed=S, pad=5).to(dev())

    def step():
        o = BA.bitfield_attn_func(q, k, v, bf)
        return o.detach(), *torch.autograd.grad(o, (q, k, v), do)

    BA.BitfieldUtils.clear_cache()
    step()  # builds the plan, loads the code objects
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for seed in range(3):
        with torch.no_grad():
            for dst, src in zip((q, k, v, do), make_inputs(1, S, Hq, Hkv, D, torch.bfloat16, seed=seed)):
                dst.copy_(src)
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(("o", "dq", "dk", "dv"), out, step()):
            assert torch.equal(a, b), name
    BA.BitfieldUtils.clear_cache()
