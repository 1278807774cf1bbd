"""Forward tiles that every row of a slice sees as a whole or not at all: scores that jump by more than the running maximum may lag behind,
in either half of a tile and beyond what a 16-bit float (and, in two powers of the base, a bf16) holds, slices with rows of two kinds, and keys whose
scores are no numbers for rows that do not see them."""

import pytest
import torch

from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O

pytestmark = pytest.mark.gpu
TEXT = (1 << 62) | 1 | 2 | 4
ENTRIES = ["bits", "mask", "index"]


def _forward(q, k, v, bf, entry):
    d = torch.device("cuda:0")
    q, k, v, S = q.to(d), k.to(d), v.to(d), q.shape[1]
    BA.BitfieldUtils.clear_cache()
    if entry == "mask":
        o, lse, _ = A._flash_attn_forward(q, k, v, mask=O.materialize_mask(bf).to(d))
    else:
        flags = BA.BitfieldUtils.materialize_compressed_mask_from_bitfield_mask(bf.to(d))
        at = [torch.arange(S, device=d)] * 2 if entry == "index" else []
        o, lse, _ = BA._bitfield_attn_forward(q, k, v, bf.to(d), flags, *at)
    BA.BitfieldUtils.clear_cache()
    return o[:, :, :2].float().cpu(), lse[:, :2, :S].cpu()


def _check(got, q, k, v, bf, rows=slice(None)):
    """Probabilities and outputs are rounded to the type, each by a unit u at most: lse is off by u, O by twice u of the mean of |v| (and by what
    fp16 loses below 2^-14, 2^-25 a key); half as much again for everything in 32 bits."""
    u = 2.0**-9 if q.dtype == torch.bfloat16 else 2.0**-12
    want, lse = O.attention_forward(q, k, v, bf)
    most, _ = O.attention_forward(q, k, v.abs(), bf)
    o_err, lse_err = (got[0] - want).abs(), (got[1] - lse).abs()
    assert (o_err <= 3 * u * most + 5e-5)[:, rows].all(), (o_err - 3 * u * most)[:, rows].max().item()
    assert lse_err[..., rows].max().item() <= 1.5 * u + 1e-6 * lse.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 40, 64, 96, 128])
@pytest.mark.parametrize("heads", [2, 264])  # two streams of waves, and one
@pytest.mark.parametrize("key", [64 * 2 + 5, 64 * 3 + 40, 64 * 3 + 31, 319])
@pytest.mark.parametrize("jump", [7.0, 60.0, 100.0])  # of a score, in units of the exponential's base e
def test_a_score_that_jumps_in_a_full_tile(dtype, D, heads, key, jump):
    g = torch.Generator().manual_seed(key + D)
    S = 320
    q, k, v = (torch.randn(1, S, heads, D, generator=g) * 0.5 for _ in range(3))
    rows = torch.arange(S) % 3 == 0  # the others keep their maximum
    q[:, rows, :, 0], q[:, ~rows, :, 0] = 4.0, 0.0
    k[..., 0] = 0.0
    k[:, key, :, 0] = jump * D**0.5 / 4.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    bf = torch.full((1, S), 2, dtype=torch.int64)  # one modality: nothing is hidden
    few = [t[:, :, :2] for t in (q, k, v)]
    for entry in ENTRIES:
        _check(_forward(q, k, v, bf, entry), *few, bf)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("heads", [2, 264])
@pytest.mark.parametrize("column", [0.0, 1.0])  # of the queries where the keys are infinite: scores that are NaN, or infinite
@pytest.mark.parametrize("key", [64 * 2 + 5, 64 * 3 + 40])
def test_rows_of_two_kinds_in_a_slice(dtype, D, heads, column, key):
    # text rows see everything before them, rows of the second modality a segment far behind the keys of interest
    g = torch.Generator().manual_seed(D + key)
    S = 700
    q, k, v = (torch.randn(1, S, heads, D, generator=g) * 0.5 for _ in range(3))
    q[..., 3] = column
    k[..., 3] = 0.0
    bf = torch.full((1, S), TEXT, dtype=torch.int64)
    bf[:, 400:410] = 2
    bf[:, 421:650:3] = 4
    q, k, v = (t.to(dtype) for t in (q, k, v))
    few = [t[:, :, :2] for t in (q, k, v)]
    blind = ((bf != TEXT) | (torch.arange(S) < key))[0]  # rows that do not see the key
    for entry in ENTRIES:
        _check(_forward(q, k, v, bf, entry), *few, bf)
        bad = k.clone()
        bad[:, key, :, 3] = float("inf")
        got = _forward(q, bad, v, bf, entry)
        _check(got, *few, bf, rows=blind)
        seen = got[0][:, ~blind]
        assert not torch.isfinite(seen).any()  # as before: the infinity reaches the rows that see it, and only those
