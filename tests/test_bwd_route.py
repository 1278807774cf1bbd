"""Which backwards above head dim 64 hand dS over and which take one launch instead: the rule is host arithmetic, asked through
``bam_attn_bwd_takes_ds`` (no pointer is followed)."""

import ctypes

import pytest

from cornstarch_amd.kernel import _bam_hip

SOMEWHERE = 1 << 20


def takes_ds(B, Sq, Sk, Hq, Hkv, D, pairs=0, head_runs=1, workspace=False, bias=None, plan=True):
    a = _bam_hip.Attn()
    a.B, a.Sq, a.Sk, a.Hq, a.Hkv, a.D, a.dtype, a.pairs, a.head_runs, a.scale = B, Sq, Sk, Hq, Hkv, D, 1, pairs, head_runs, 1.0
    for name, S, H in (("q", Sq, Hq), ("k", Sk, Hkv), ("v", Sk, Hkv), ("o", Sq, Hq), ("dout", Sq, Hq), ("dq", Sq, Hq), ("dk", Sk, Hkv), ("dv", Sk, Hkv)):
        t = getattr(a, name)
        t.ptr, t.stride_b, t.stride_s, t.stride_h = SOMEWHERE, S * H * D, H * D, D
    a.lse = a.delta = a.bf = a.flags = SOMEWHERE
    a.bf_stride_b, a.flags_stride_m = Sk, -(-Sk // 32)
    a.flags_stride_b = a.flags_stride_m * -(-Sq // 128)
    p = _bam_hip.Plan()
    p.fine = p.order = p.group_order = p.ds_entry = p.ds_tile_base = SOMEWHERE
    p.fine_stride_s, p.B, p.Sq, p.Sk = -(-Sk // 512) * 16, B, Sq, Sk
    if Sq != Sk:
        view = _bam_hip.IndexView(SOMEWHERE, SOMEWHERE, SOMEWHERE, SOMEWHERE, Sq, Sk, Sq, Sk)
        a.mode, a.index = 1, ctypes.pointer(view)
    if plan:
        a.plan = ctypes.pointer(p)
    if bias is not None:
        a.bias = ctypes.pointer(_bam_hip.Bias(SOMEWHERE, 0, Sk, bias, 1))
    if workspace:
        a.ds_workspace, a.ds_capacity = SOMEWHERE, 1 << 16
    n = ctypes.c_int(-1)
    _bam_hip.call("bam_attn_bwd_takes_ds", ctypes.byref(a), ctypes.byref(n))
    return n.value


def all_pairs(B, Sq, Sk):
    return B * ((Sq + 31) // 32) * ((Sk + 127) // 128)


@pytest.mark.parametrize("shape,before,uneven,level", [
    ((1, 767, 767, 4, 4, 96), 1, 1, 1), ((1, 768, 768, 4, 4, 96), 0, 0, 0),            # from 768 keys on
    ((1, 2048, 2048, 8, 8, 128), 0, 0, 0), ((1, 2049, 2049, 8, 8, 128), 1, 0, 1),      # 256 and 272 workgroups
    ((1, 2048, 2048, 16, 16, 128), 1, 0, 1), ((1, 2049, 2049, 16, 16, 128), 1, 1, 1),  # 512 and 544
    ((1, 1024, 2048, 12, 12, 72), 1, 0, 1), ((1, 1024, 2048, 8, 8, 72), 0, 0, 0),      # index tensors: 96 + 192, 64 + 128
    ((1, 2048, 2048, 8, 2, 128), 0, 0, 0), ((1, 4096, 4096, 6, 1, 128), 1, 0, 1),      # parts of dK/dV count
    ((1, 2048, 2048, 8, 8, 64), 0, 0, 0), ((1, 131073, 131073, 1, 1, 128), 0, 0, 0),   # no hand-over at all
])
def test_sizes_and_the_count_decide(shape, before, uneven, level):
    B, Sq, Sk = shape[:3]
    total = all_pairs(B, Sq, Sk)
    assert [takes_ds(*shape), takes_ds(*shape, pairs=2 * total // 3), takes_ds(*shape, pairs=total)] == [before, uneven, level]


def test_what_keeps_two_launches():
    small = (1, 2048, 2048, 8, 8, 128)
    assert takes_ds(*small, head_runs=2) == 1 and takes_ds(*small, plan=False) == 0
    assert takes_ds(*small, workspace=True) == 0      # (what the call would need; a workspace that is given is used)
    assert takes_ds(*small, bias=0) == 0 and takes_ds(*small, bias=2048) == 1  # per key; a matrix
    assert takes_ds(1, 2047, 2047, 8, 8, 128, bias=0) == 1  # rows of the bias that no 16-byte load fits
