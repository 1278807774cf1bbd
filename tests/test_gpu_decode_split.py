"""How the decode step cuts its tiles over workgroups: units that divide the chip evenly and units that do not, parts that
hold one tile or none for some waves, merges by the last workgroup (counters, reused from call to call and per stream)
and by the second launch (bam_decode), head dims between the compiled ones."""

import math

import pytest
import torch

from cornstarch_amd.kernel import _bam_hip
from cornstarch_amd.kernel import bitfield_attention as BA
from cornstarch_amd.kernel import interface
from oracle import bam_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sk,D", [
    (10, 8, 8, 2100, 128),   # 80 units: 3 workgroups of four waves each
    (7, 6, 3, 517, 64), (3, 4, 1, 4001, 32), (1, 8, 2, 129, 96), (33, 16, 8, 97, 128), (2, 70, 2, 1025, 128),
    (300, 2, 1, 700, 128),   # more units than compute units: two workgroups of one wave each
    (2, 8, 2, 333, 8), (2, 8, 2, 1333, 40), (1, 6, 2, 2003, 80), (1, 4, 4, 65, 120),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_pieces_and_merges(B, Hq, Hkv, Sk, D, dtype):
    d = torch.device("cuda:0")
    g = torch.Generator().manual_seed(Sk + D)
    q, k, v = ((torch.randn(s, generator=g) * 0.5).to(dtype) for s in ((B, Hq, 1, D), (B, Hkv, Sk, D), (B, Hkv, Sk, D)))
    qd, kd, vd = (t.to(d) for t in (q, k, v))
    module = torch.nn.Module().eval()
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    for kw in ({}, {"sliding_window": Sk // 2 + 1, "softcap": 20.0}):
        want = O.decode_step(q, k, v, **kw)
        outs = []
        for n in range(4):  # counters are back at zero after every call, and each stream has its own
            with torch.cuda.stream(streams[n % 2]):
                outs.append(interface.bitfield_attention_forward(module, qd, kd, vd, None, **kw)[0])
        torch.cuda.synchronize()
        assert all(torch.equal(outs[0], x) for x in outs[1:])
        assert (outs[0].float().cpu() - want).abs().max().item() <= 2e-2
        if D in (32, 64, 128):  # the two-launch form
            lib, w, cap = _bam_hip.load(), kw.get("sliding_window", 0), kw.get("softcap", 0.0)
            need = lib.bam_decode_workspace_bytes(B, Sk, Hq, Hkv, D, w)
            ws = torch.empty((max(need, 1),), dtype=torch.uint8, device=d)
            out = torch.empty((B, 1, Hq, D), dtype=dtype, device=d)
            _bam_hip.call("bam_decode", qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), qd.stride(0), qd.stride(1),
                          kd.stride(0), kd.stride(2), kd.stride(1), vd.stride(0), vd.stride(2), vd.stride(1), Hq * D, D, B, Sk, Hq,
                          Hkv, D, 1.0 / math.sqrt(D), BA._dtype_code(dtype), w, cap, ws.data_ptr() if need else None, need,
                          BA._stream_ptr(d))
            torch.cuda.synchronize()
            assert (out.float().cpu() - want).abs().max().item() <= 2e-2


def test_the_stream_that_has_one_handle_for_all_threads():
    # hipStreamPerThread: no counters are kept for it, the second launch merges
    d = torch.device("cuda:0")
    g = torch.Generator().manual_seed(0)
    q, k, v = ((torch.randn(s, generator=g) * 0.5).bfloat16() for s in ((2, 8, 1, 64), (2, 2, 1999, 64), (2, 2, 1999, 64)))
    qd, kd, vd = (t.to(d) for t in (q, k, v))
    want = O.decode_step(q, k, v)
    before = _bam_hip.host.decode_counter_sets()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.ExternalStream(2)):
        out = interface.bitfield_attention_forward(torch.nn.Module().eval(), qd, kd, vd, None)[0]
    torch.cuda.synchronize()
    assert (out.float().cpu() - want).abs().max().item() <= 2e-2
    assert _bam_hip.host.decode_counter_sets() == before
