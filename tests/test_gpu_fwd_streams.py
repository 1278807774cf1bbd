"""The forward and dQ with few workgroups walk two tiles at a time and merge two partial results per row.  Every sequence of a batch
that is large enough to go tile by tile, against the same sequence by itself."""

import pytest
import torch

from cornstarch_amd.kernel import bitfield_attention as BA
from tests.helpers import random_bitfield, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("D", [32, 40, 64, 96, 128])
@pytest.mark.parametrize("S", [1, 64, 65, 130, 200, 257])  # lists of 1 to 5 tiles, odd and even
def test_a_sequence_of_a_large_batch_equals_the_sequence_alone(S, D, biased):
    Hq, Hkv = 8, 2
    B = 1024 // (Hq * ((S + 127) // 128)) + 1  # more than 1024 workgroups
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v = ((torch.randn(B, S, H, D, generator=g, device="cuda")).bfloat16() for H in (Hq, Hkv, Hkv))
    bf = random_bitfield(B, S, seed=S, pad=S // 9).cuda()
    bias = torch.randn(1, Hq, 1, S, generator=g, device="cuda") if biased else None

    def forward(rows):
        BA.BitfieldUtils.clear_cache()
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf[rows])
        return BA._bitfield_attn_forward(q[rows], k[rows], v[rows], bf[rows], flags, bias=bias)[:2]

    o, lse = forward(slice(None))
    for b in (0, B // 2, B - 1):
        o1, lse1 = forward(slice(b, b + 1))
        # probabilities are rounded to bf16 against another running maximum: 2^-9 each, over at least one key; the sums of the
        # rounded ones (the lse) differ by no more than that
        assert rel_l2(o1[0].float(), o[b].float()) <= 2.0**-8
        live = torch.isfinite(lse[b])
        assert torch.equal(live, torch.isfinite(lse1[0])) and (lse1[0] - lse[b])[live].abs().max().item() <= 2.0**-8
        assert torch.isfinite(o1).all() and torch.equal(lse[b][~live], lse1[0][~live])
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("D", [32, 40, 64])
@pytest.mark.parametrize("S", [64, 65, 130, 200, 257])
def test_gradients_of_a_sequence_of_a_large_batch_equal_those_alone(S, D, biased):
    Hq, Hkv = 8, 2
    B = 1024 // (Hq * ((S + 127) // 128)) + 1
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v, do = ((torch.randn(B, S, H, D, generator=g, device="cuda")).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(B, S, seed=S, pad=S // 9).cuda()
    bias = torch.randn(1, Hq, 1, S, generator=g, device="cuda") if biased else None

    def gradients(rows):
        BA.BitfieldUtils.clear_cache()
        x = [t[rows].detach().requires_grad_(True) for t in (q, k, v)]
        return torch.autograd.grad(BA.bitfield_attn_func(*x, bf[rows], bias), x, do[rows])

    batch = gradients(slice(None))
    for b in (0, B // 2, B - 1):
        for one, all_ in zip(gradients(slice(b, b + 1)), batch):
            # o and the lse differ by a rounding of P to bf16 (2^-9 a term), which delta and P carry into the gradients
            assert torch.isfinite(one).all() and rel_l2(one[0].float(), all_[b].float()) <= 2.0**-7
    BA.BitfieldUtils.clear_cache()


# either side of the lines up to which two tiles are walked at a time: (few sequences: two, more of them: one)
@pytest.mark.parametrize("D,S,few,many", [(32, 2570, 3, 7), (64, 3100, 3, 4), (64, 5000, 2, 3), (96, 2005, 4, 5), (128, 1990, 3, 4), (128, 3100, 3, 4), (128, 8200, 1, 2)])
def test_long_lists_on_either_side_of_the_line(D, S, few, many):
    Hq, Hkv = 8, 2
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v, do = ((torch.randn(many, S, H, D, generator=g, device="cuda")).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(many, S, seed=S, pad=S // 9).cuda()

    def run(n):
        BA.BitfieldUtils.clear_cache()
        x = [t[:n].detach().requires_grad_(True) for t in (q, k, v)]
        o = BA.bitfield_attn_func(*x, bf[:n].contiguous())
        return o.detach(), *torch.autograd.grad(o, x, do[:n])

    for bound, one, two in zip((2.0**-8, 2.0**-7, 2.0**-7, 2.0**-7), run(many), run(few)):  # (as above)
        for b in range(few):
            assert torch.isfinite(two[b]).all() and rel_l2(two[b].float(), one[b].float()) <= bound
    BA.BitfieldUtils.clear_cache()


# dQ from the stored dS with 257 to 512 workgroups: long and short ones share a compute unit; with 258 and 270 of them the last ones
# are not whole runs of eight
@pytest.mark.parametrize("B,Hq,Hkv,S", [(3, 6, 3, 1900), (1, 6, 6, 43 * 128), (2, 16, 4, 2047), (8, 8, 8, 515)])
def test_dq_of_workgroups_taken_in_another_order(B, Hq, Hkv, S):
    D = 128
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v, do = ((torch.randn(B, S, H, D, generator=g, device="cuda")).bfloat16() for H in (Hq, Hkv, Hkv, Hq))
    bf = random_bitfield(B, S, seed=S, pad=S // 9).cuda()

    def dq(heads, kv):  # one kv head at a time: 43 to 64 workgroups, in the order of their lengths
        BA.BitfieldUtils.clear_cache()
        x = [t.detach().requires_grad_(True) for t in (q[:, :, heads], k[:, :, kv], v[:, :, kv])]
        return torch.autograd.grad(BA.bitfield_attn_func(*x, bf), x[0], do[:, :, heads])[0]

    whole, G = dq(slice(None), slice(None)), Hq // Hkv
    for h in range(Hkv):
        part = dq(slice(h * G, (h + 1) * G), slice(h, h + 1))
        # (another number of workgroups decides about the forward's streams: a rounding of P to bf16, as above)
        assert torch.isfinite(whole).all() and rel_l2(whole[:, :, h * G : (h + 1) * G].float(), part.float()) <= 2.0**-7
    BA.BitfieldUtils.clear_cache()
