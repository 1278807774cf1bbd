"""Forward tiles that take the short way -- every row of a slice sees all keys of the tile or none, and the running maximum is not looked
at: scores that jump by more than it may lag behind, in either half of a tile and beyond what a 16-bit float holds, slices with rows
of two kinds, and keys whose scores are no numbers for rows that do not see them."""

import pytest
import torch

from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA
from oracle import bam_oracle as O

pytestmark = pytest.mark.gpu
TEXT = (1 << 62) | 1 | 2 | 4


def _forward(q, k, v, bf, dense):
    d = torch.device("cuda:0")
    BA.BitfieldUtils.clear_cache()
    if dense:
        return A.flash_attn_func(q.to(d), k.to(d), v.to(d), mask=O.materialize_mask(bf).to(d))
    return BA.bitfield_attn_func(q.to(d), k.to(d), v.to(d), bf.to(d))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 40, 64, 96, 128])
@pytest.mark.parametrize("heads", [2, 264])  # two streams of waves, and one
@pytest.mark.parametrize("key", [64 * 2 + 5, 64 * 3 + 40, 64 * 3 + 31, 319])
@pytest.mark.parametrize("jump", [7.0, 60.0])  # of a score, in units of the exponential's base e
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
    few = slice(0, 2) if heads > 2 else slice(None)
    want, _ = O.attention_forward(q[:, :, few], k[:, :, few], v[:, :, few], bf)
    for dense in (False, True):
        got = _forward(q, k, v, bf, dense)[:, :, few].float().cpu()
        assert (got - want).abs().max().item() <= 2e-2
    BA.BitfieldUtils.clear_cache()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("column", [0.0, 1.0])  # of the queries where the keys are infinite: scores that are NaN, or infinite
@pytest.mark.parametrize("key", [64 * 2 + 5, 64 * 3 + 40])
def test_rows_of_two_kinds_in_a_slice(dtype, D, column, key):
    # text rows see everything before them, rows of the second modality a segment far behind the keys of interest
    g = torch.Generator().manual_seed(D + key)
    S, H = 700, 2
    q, k, v = (torch.randn(1, S, H, D, generator=g) * 0.5 for _ in range(3))
    q[..., 3] = column
    k[..., 3] = 0.0
    bf = torch.full((1, S), TEXT, dtype=torch.int64)
    bf[:, 400:410] = 2
    bf[:, 421:650:3] = 4
    q, k, v = (t.to(dtype) for t in (q, k, v))
    want, _ = O.attention_forward(q, k, v, bf)
    blind = (bf != TEXT) | (torch.arange(S) < key)  # rows that do not see the key
    for dense in (False, True):
        got = _forward(q, k, v, bf, dense).float().cpu()
        assert (got - want).abs().max().item() <= 2e-2
        bad = k.clone()
        bad[:, key, :, 3] = float("inf")
        got = _forward(q, bad, v, bf, dense).float().cpu()
        assert (got - want)[blind].abs().max().item() <= 2e-2
        seen = got[~blind]
        assert not torch.isfinite(seen).any()  # as before: the infinity reaches the rows that see it, and only those
    BA.BitfieldUtils.clear_cache()
