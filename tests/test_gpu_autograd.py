"""The native autograd node under what a training program does around it: saved-tensor hooks, activation checkpointing, graphs
kept or freed, gradients of some inputs only, tensor subclasses, inference mode, and the transforms it has no rule for."""

import threading

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.utils.checkpoint import checkpoint

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA
from tests.helpers import random_bitfield

pytestmark = pytest.mark.gpu


class Problem:
    def __init__(self, B=2, S=200, Hq=4, Hkv=2, D=64, dtype=torch.bfloat16, bias=False):
        dev = torch.device("cuda:0")
        g = torch.Generator(device=dev).manual_seed(S + D)
        self.q, self.k, self.v, self.do = (torch.randn(B, S, H, D, generator=g, device=dev).to(dtype).requires_grad_(n < 3)
                                           for n, H in enumerate((Hq, Hkv, Hkv, Hq)))
        self.bf = random_bitfield(B, S, seed=S, pad=3).to(dev)
        self.bias = torch.randn(1, Hq, 1, S, generator=g, device=dev) if bias else None
        BA.BitfieldUtils.clear_cache()

    @property
    def inputs(self):
        return self.q, self.k, self.v

    def forward(self, q=None, k=None, v=None):
        return BA.bitfield_attn_func(*(x if x is not None else y for x, y in zip((q, k, v), self.inputs)), self.bf, self.bias)

    def grads(self, o=None, **kw):
        return torch.autograd.grad(self.forward() if o is None else o, self.inputs, self.do, **kw)


def same(xs, ys):
    return all(torch.equal(x, y) for x, y in zip(xs, ys))


def wide(t):
    """The same values with another layout: twice the stride along the last dimension."""
    return torch.stack((t, t), -1).flatten(-2)[..., ::2]


def shifted(t):
    """The same values at an address that is a multiple of the element size and of nothing more."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    return flat[1:].view(t.shape).copy_(t)


def hooks(change):
    return torch.autograd.graph.saved_tensors_hooks(lambda t: t, change)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias", [False, True])
def test_saved_tensor_hooks_that_move_or_lay_out_the_tensors(D, bias):
    p = Problem(D=D, bias=bias)
    want = p.grads()
    with torch.autograd.graph.save_on_cpu():
        o = p.forward()
    assert same(p.grads(o), want)
    for change in (torch.clone, wide, shifted):
        with hooks(change):
            o = p.forward()
        assert same(p.grads(o), want), change
    mask = BA.materialize_bitfield_mask(p.bf)
    if not bias:
        want = torch.autograd.grad(A.flash_attn_func(*p.inputs, mask=mask), p.inputs, p.do)
        for change in (torch.clone, wide, shifted):
            with hooks(change):
                o = A.flash_attn_func(*p.inputs, mask=mask)
            assert same(torch.autograd.grad(o, p.inputs, p.do), want), change


def test_a_bias_that_comes_back_in_another_type_is_an_error_and_not_ignored():
    p = Problem(bias=True)
    with hooks(lambda t: t.double() if t.shape == p.bias.shape else t):
        o = p.forward()
    with pytest.raises(RuntimeError, match="bias"):
        p.grads(o)


# (tests of what else a hook may hand back, each refused on the host before anything is launched)
@pytest.mark.parametrize("which,change", [
    ("q", lambda t: t.float()), ("k", lambda t: t[:, :-1]), ("v", lambda t: t.cpu()), ("o", lambda t: t[..., :32]),
    ("lse", lambda t: t.half()), ("lse", lambda t: t[:, :, :-1]), ("mask", lambda t: t.int()), ("mask", lambda t: t[:, :-1]),
    ("flags", lambda t: t[:, :, :-1]), ("flags", lambda t: t.float()), ("bias", lambda t: t[..., :-1]), ("bias", lambda t: t.cpu()),
])
def test_a_tensor_that_comes_back_as_something_else_is_an_error(which, change):
    p = Problem(Hkv=4, bias=True)
    order = ["q", "k", "v", "lse", "bias", "mask", "flags", "o"]  # as the node packs them
    packed = []

    def pack(t):
        packed.append(t)
        return len(packed) - 1, t

    def unpack(x):
        n, t = x
        return change(t) if order[n] == which else t

    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        o = p.forward()
    assert len(packed) == len(order)
    with pytest.raises(_bam_hip.BamError, match=which):  # (the library's own error, also out of the engine)
        p.grads(o)


def test_a_python_error_inside_the_backward_reaches_the_caller_as_it_is(monkeypatch):
    def no_workspace(*args):
        raise KeyError("no workspace today")

    p = Problem(D=128)
    o = p.forward()
    monkeypatch.setattr(BA._TilePlan, "backward_workspace", no_workspace)
    with pytest.raises(KeyError, match="no workspace today"):
        p.grads(o)


def test_threads_that_run_the_backward_of_one_graph():
    p = Problem(D=128)
    o = p.forward()
    want = p.grads(o, retain_graph=True)
    got, go = {}, threading.Barrier(4)

    def work(n):
        go.wait()
        got[n] = [p.grads(o, retain_graph=True) for _ in range(5)]

    threads = [threading.Thread(target=work, args=(n,)) for n in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(same(x, want) for n in range(4) for x in got[n])


def test_threads_of_which_one_may_free_the_graph():
    # every backward either gives the gradients or says that the graph has been freed
    p = Problem(D=128)
    want = p.grads()
    for _ in range(20):
        o, go, got = p.forward(), threading.Barrier(4), {}

        def work(n):
            go.wait()
            try:
                got[n] = p.grads(o, retain_graph=n != 0)
            except RuntimeError as e:
                got[n] = e

        threads = [threading.Thread(target=work, args=(n,)) for n in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        for x in got.values():
            assert "second time" in str(x) if isinstance(x, RuntimeError) else same(x, want)


@pytest.mark.parametrize("reentrant", [False, True])
def test_activation_checkpointing(reentrant):
    p = Problem(D=128)
    want = p.grads()
    o = checkpoint(p.forward, *p.inputs, use_reentrant=reentrant)
    if reentrant:  # (its backward only runs through backward())
        o.backward(p.do)
        got = [x.grad for x in p.inputs]
    else:
        got = p.grads(o)
    assert same(got, want)


@pytest.mark.parametrize("D", [64, 128])
def test_a_graph_is_kept_or_freed(D):
    p = Problem(D=D)
    o = p.forward()
    first = p.grads(o, retain_graph=True)
    assert same(p.grads(o), first)
    with pytest.raises(RuntimeError, match="second time"):
        p.grads(o)
    # no second derivative: the gradients are constants
    assert not any(x.requires_grad for x in p.grads(create_graph=True))


def test_inputs_changed_after_the_forward_are_noticed():
    for name in ("q", "bf"):
        p = Problem()
        o = p.forward()
        with torch.no_grad():
            getattr(p, name).add_(0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            p.grads(o)


def test_gradients_of_some_inputs_only():
    p = Problem(D=128)
    want = p.grads()
    for n in range(3):
        inputs = [x if n == m else x.detach() for m, x in enumerate(p.inputs)]
        (got,) = torch.autograd.grad(p.forward(*inputs), (p.inputs[n],), p.do)
        assert torch.equal(got, want[n])
    # an input that is the output of other operations, and one tensor in two roles
    x = p.k.detach().clone().requires_grad_(True)
    (got,) = torch.autograd.grad(p.forward(p.q.detach(), x * 1.0, x), (x,), p.do)
    o = p.forward(p.q.detach(), p.k, p.k)
    (both,) = torch.autograd.grad(o, (p.k,), p.do)
    assert torch.equal(got, both)


def test_no_graph_without_gradients():
    p = Problem()
    want = p.forward().detach()
    with torch.no_grad():
        assert p.forward().grad_fn is None
    assert p.forward(*(x.detach() for x in p.inputs)).grad_fn is None


@pytest.mark.parametrize("masked", [False, True])
def test_inference_mode(masked):
    p = Problem()

    def forward(q, k, v, bf):
        return A.flash_attn_func(q, k, v, mask=BA.materialize_bitfield_mask(bf)) if masked else BA.bitfield_attn_func(q, k, v, bf)

    want = forward(*p.inputs, p.bf).detach()
    BA.BitfieldUtils.clear_cache()
    A._MaskPlan.forget()
    with torch.inference_mode():
        first = forward(*(x.detach() for x in p.inputs), p.bf)
        # inputs made in inference mode, a mask without a version counter among them
        copies = [x.detach().clone() for x in (*p.inputs, p.bf)]
        second = forward(*copies)
        copies[3].fill_(p.bf[0, 0])  # written to: nothing of the last call is left
        third = forward(*copies)
    assert first.is_inference() and torch.equal(first, want) and torch.equal(second, want)
    # what the first call left in the cache serves training as well
    got = torch.autograd.grad(forward(*p.inputs, p.bf), p.inputs, p.do)
    BA.BitfieldUtils.clear_cache()
    assert same(got, torch.autograd.grad(forward(*p.inputs, p.bf), p.inputs, p.do))
    assert torch.equal(third, forward(*p.inputs, torch.full_like(p.bf, int(p.bf[0, 0]))))
    BA.BitfieldUtils.clear_cache()


def test_tensor_subclasses():
    class Named(torch.Tensor):
        pass

    p = Problem()
    want = p.grads()
    named = [x.detach().as_subclass(Named).requires_grad_(True) for x in p.inputs]
    got = torch.autograd.grad(p.forward(*named), named, p.do)
    assert same(got, want)
    parameters = [torch.nn.Parameter(x.detach()) for x in p.inputs]
    assert same(torch.autograd.grad(p.forward(*parameters), parameters, p.do), want)


def test_transforms_without_a_rule_are_refused():
    p = Problem(Hkv=4)
    q, k, v = (x.detach() for x in p.inputs)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: p.forward(x, k, v).float().sum())(q)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: p.forward(x, k, v))(torch.stack((q, q)))
    with fwAD.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            p.forward(fwAD.make_dual(q, torch.ones_like(q)), k, v)
    o = p.forward()
    with pytest.raises(RuntimeError):
        torch.autograd.grad(o, p.inputs, torch.stack((p.do, p.do)), is_grads_batched=True)
