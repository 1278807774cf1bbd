"""Row sums of long rows: lse against the exact sum of probabilities that every type holds exactly."""

import math

import pytest
import torch

from cornstarch_amd.kernel import attention as A
from cornstarch_amd.kernel import bitfield_attention as BA

pytestmark = pytest.mark.gpu


# A row's probabilities are 2^0 .. 2^-12, drawn evenly, so that their sum S needs some 29 bits.  One rounding a tile of 64 keys, in
# either half of the lanes (as simulated in fp32): rms 6e-7 of S in one stream at 131072 keys, largest 1.6e-6; the lse adds its own roundings, at
# values near 9.9 three of 2^-21 / sqrt(12).  A rounding per product of four loses 2.4e-5 (3.7e-6 in two streams), all to one side.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("heads,S", [(2, 131072), (640, 131072), (2, 131072 + 640)])  # two streams, one, one and more than one list
def test_the_row_sum_rounds_once_a_tile(heads, S, D, dtype):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(D)
    k = torch.randint(-12, 1, (S, D), generator=g)
    k[0] = 0  # the maximum, in the first tile
    want = torch.exp2(k.double()).sum(0).log()  # of the row that is column c's unit vector
    q = torch.eye(D).repeat(-(-128 // D), 1)[:128].view(1, 128, 1, D).expand(1, 128, heads, D)
    k = k.view(1, S, 1, D)
    BA.BitfieldUtils.clear_cache()
    _, lse, _ = A._flash_attn_forward(q.to(dtype).to(dev), k.to(dtype).to(dev), torch.ones_like(k).to(dtype).to(dev), softmax_scale=math.log(2.0))
    err = lse[0, :2, :128].double().cpu() - want.repeat(-(-128 // D))[:128]
    assert err.square().mean().sqrt().item() <= 1.2e-6
    assert err.abs().max().item() <= 4e-6
    BA.BitfieldUtils.clear_cache()
