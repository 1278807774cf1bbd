"""Where the tiles of q, k, v and do are copied from: sequences that end inside a tile (the rows behind them belong to somebody
else), rows further apart than 32-bit tile offsets reach, and rows that overlap."""

import pytest
import torch

from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu


def _inputs(B, S, Hq, Hkv, D, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(torch.randn(B, S, H, D, generator=g, device="cuda") * 0.5).to(dtype) for H in (Hq, Hkv, Hkv, Hq)]


def _step(q, k, v, do, attend):
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    o = attend(q, k, v)
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))


@pytest.mark.parametrize("D", [32, 40, 64, 96, 128])
@pytest.mark.parametrize("S", [1, 31, 33, 63, 65, 95, 127, 129, 193])
def test_rows_behind_the_sequence_are_not_read(S, D):
    B, Hq, Hkv = 2, 4, 2
    plain = _inputs(B, S, Hq, Hkv, D, torch.bfloat16, S + D)
    # the same rows at the front of longer buffers that go on with NaN
    inside = []
    for t in plain:
        big = torch.full((B, S + 130, t.shape[2], D), float("nan"), dtype=t.dtype, device="cuda")
        big[:, :S] = t
        inside.append(big[:, :S])
    bf = random_bitfield(B, S, seed=S).cuda()
    wide = torch.full((B, S + 130), (1 << 62) - 1, dtype=torch.int64, device="cuda")  # bitfields that everybody sees
    wide[:, :S] = bf
    mask = BA.materialize_bitfield_mask(bf)
    bias = torch.full((1, 1, 1, S + 130), float("inf"), device="cuda")
    bias[..., :S] = torch.randn(S, device="cuda")
    ways = [
        (lambda q, k, v: BA.bitfield_attn_func(q, k, v, bf), lambda q, k, v: BA.bitfield_attn_func(q, k, v, wide[:, :S])),
        (lambda q, k, v: A.flash_attn_func(q, k, v, mask=mask),) * 2,
        (lambda q, k, v: BA.bitfield_attn_func(q, k, v, bf, bias[..., :S].clone()),
         lambda q, k, v: BA.bitfield_attn_func(q, k, v, wide[:, :S], bias[..., :S])),
    ]
    for attend, attend_inside in ways:
        for a, b in zip(_step(*plain, attend), _step(*inside, attend_inside)):
            assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("far", [0, 1, 2, 3], ids=["q", "k", "v", "do"])
def test_rows_two_gigabytes_apart(far, D):
    B, S, Hq, Hkv = 1, 135, 4, 2
    plain = _inputs(B, S, Hq, Hkv, D, torch.bfloat16, far + D)
    stride = (1 << 23) - 8  # the largest the entry points take: 134 rows of it are more than 2^31 bytes
    spread = list(plain)
    t = plain[far]
    store = torch.empty((S - 1) * stride + t.shape[2] * D, dtype=t.dtype, device="cuda")
    spread[far] = store.as_strided(t.shape, (stride, stride, D, 1))
    spread[far].copy_(t)
    bf = random_bitfield(B, S, seed=7).cuda()
    attend = lambda q, k, v: BA.bitfield_attn_func(q, k, v, bf)  # noqa: E731
    for a, b in zip(_step(*plain, attend), _step(*spread, attend)):
        # the other instantiation adds the same products in another order: the bar of the plan tests
        assert torch.isfinite(b).all() and rel_l2(b.float(), a.float()) <= 2e-3


@pytest.mark.parametrize("D", [8, 40, 64, 72, 120])
@pytest.mark.parametrize("far", [0, 1, 2, 3], ids=["q", "k", "v", "do"])
def test_rows_between_one_and_two_gigabytes_apart(far, D):
    # head dims between the compiled ones: the columns past them are zeros wherever in the tensor a tile starts
    B, S, Hq, Hkv = 1, 121, 4, 2
    plain = _inputs(B, S, Hq, Hkv, D, torch.bfloat16, far + D)
    stride = (1 << 23) - 8  # 120 rows of it are 2.01e9 bytes
    spread = list(plain)
    t = plain[far]
    store = torch.full(((S - 1) * stride + t.shape[2] * D,), float("inf"), dtype=t.dtype, device="cuda")
    spread[far] = store.as_strided(t.shape, (stride, stride, D, 1))
    spread[far].copy_(t)
    bf = random_bitfield(B, S, seed=7).cuda()
    attend = lambda q, k, v: BA.bitfield_attn_func(q, k, v, bf)  # noqa: E731
    for a, b in zip(_step(*plain, attend), _step(*spread, attend)):
        assert torch.isfinite(b).all() and torch.equal(a, b)
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("D", [40, 128])
@pytest.mark.parametrize("S", [70, 96])
def test_rows_that_overlap(S, D):
    # one row of keys for the whole sequence (a stride of 0): the same numbers as with that row written out
    q, k, v, do = _inputs(2, S, 4, 2, D, torch.float16, S + D)
    k, v = k[:, :1].expand(2, S, 2, D), v[:, :1].expand(2, S, 2, D)
    bf = random_bitfield(2, S, seed=S).cuda()
    flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf)
    got = BA._bitfield_attn_forward(q, k, v, bf, flags)
    want = BA._bitfield_attn_forward(q, k.contiguous(), v.contiguous(), bf, flags)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    grads = []
    for keys, values in ((k, v), (k.contiguous(), v.contiguous())):
        acc = [torch.zeros(t.shape, dtype=torch.float32, device="cuda") for t in (q, k, v)]
        BA._bitfield_attn_backward(do, q, keys, values, want[0], bf, flags, want[1], *acc, softmax_scale=want[2])
        grads.append(acc)
    for a, b in zip(*grads):
        assert torch.equal(a, b)
    BA.BitfieldUtils.clear_cache()
