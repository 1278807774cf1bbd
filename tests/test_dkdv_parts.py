"""How many workgroups share the q heads of a kv head in dK/dV: the rule is host arithmetic, asked through ``bam_attn_bwd_parts``."""

import ctypes

import pytest

from cornstarch_amd.kernel import _bam_hip

DENSE = 2


def parts(B, S, Hq, Hkv, D, mode=0, pairs=0):
    a = _bam_hip.Attn()
    a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D, a.mode, a.pairs = B, S, S, Hq, Hkv, D, mode, pairs
    for name, heads in (("q", Hq), ("k", Hkv), ("v", Hkv), ("dout", Hq)):
        getattr(a, name).stride_s = heads * D
    n = ctypes.c_int64()
    _bam_hip.call("bam_attn_bwd_parts", ctypes.byref(a), ctypes.byref(n))
    assert n.value % (8 * B * S * Hkv * D) == 0
    return n.value // (8 * B * S * Hkv * D) or 1


# the shapes of the GPU tests, and the lines of the rule
@pytest.mark.parametrize("shape,want", [
    ((1, 129, 16, 1, 32), 16), ((1, 700, 32, 8, 40), 4), ((1, 2100, 6, 3, 56), 2), ((4, 400, 6, 1, 64), 6), ((3, 1000, 24, 4, 64), 3),
    ((1, 4100, 12, 3, 8), 4), ((1, 700, 32, 8, 128), 4), ((2, 900, 16, 4, 96), 4), ((1, 2003, 12, 4, 112), 3),
    ((2, 700, 16, 4, 96), 4), ((1, 1000, 72, 8, 80), 9),
    ((2, 283, 6, 2, 64), 1), ((4, 1537, 8, 4, 32), 1),
    ((1, 512, 8, 1, 64), 8),
    ((1, 300, 32, 8, 128), 1),   # 15 steps saved: 32 are asked for
    ((4, 1537, 32, 8, 128), 1),  # 416 workgroups
    ((1, 8192, 32, 8, 128), 1),
    ((1, 3001, 32, 32, 128), 1),  # nothing to deal
])
def test_causal_estimate(shape, want):
    assert parts(*shape) == want


def all_pairs(B, S):
    return B * ((S + 31) // 32) * ((S + 127) // 128)


# level lists: whole rounds of the 256 compute units count
@pytest.mark.parametrize("shape,causal,level", [
    ((1, 1024, 32, 8, 128), 4, 4), ((1, 2500, 32, 8, 128), 2, 1), ((1, 3001, 32, 8, 128), 2, 1), ((1, 4096, 32, 8, 128), 2, 1),
    ((2, 1537, 32, 8, 128), 2, 1), ((1, 5000, 32, 8, 128), 2, 4), ((1, 9000, 16, 4, 128), 4, 4), ((1, 2048, 16, 2, 64), 8, 8),
])
def test_masks_that_hide_nothing(shape, causal, level):
    B, S = shape[:2]
    assert parts(*shape) == causal
    assert parts(*shape, pairs=all_pairs(B, S)) == level
    assert parts(*shape, mode=DENSE) == level  # no mask
    # fewer pairs than a causal mask has: the estimate that was fitted to such masks
    assert parts(*shape, pairs=all_pairs(B, S) // 3) == causal
