"""Kernels that take the layer-list decoders' large prompt steps, against the fp32 torch form of the same operator at the
sizes where their tiles, chunks and segments begin and end."""
import math

import pytest
import torch

from k8s_llm_monitor_amd.ops import hybrid as H

from test_hybrid_ops_gpu import _g, _i32, _paged, _r

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("dk,dv,Hq,G,new,ctx,window,kw", [
    (128, 128, 4, 1, [65, 1, 63], [0, 130, 1], 0, dict()),
    (128, 128, 2, 2, [257, 3], [0, 61], 0, dict(sinks=True)),
    (128, 128, 8, 1, [33, 95], [31, 0], 64, dict(sink=True)),
    (128, 128, 4, 2, [128, 129], [64, 500], 100, dict(gate=True)),
    (64, 64, 4, 1, [70, 200], [0, 7], 0, dict(cap=4.0)),
    (64, 128, 2, 1, [190, 64], [200, 0], 96, dict(chunked=True, cap=30.0)),
    (128, 64, 3, 1, [256, 40], [0, 90], 50, dict(keep=3)),
    (128, 128, 4, 1, [130], [300], 65, dict(keep=70, sinks=True, cap=20.0)),
    (128, 128, 8, 1, [64] * 70, [0] * 70, 17, dict(sink=True)),  # more segments than lanes
])
def test_window_flash(dk, dv, Hq, G, new, ctx, window, kw):
    """The LDS-staged prefill kernel (256 rows x heads per workgroup, 64-key tiles): rows and keys at and around tile
    edges, every mask, cap, sink and gate it takes.  bf16 weights and values: 2^-8 of the output's scale each."""
    g = _g(61)
    lens = [c + n for c, n in zip(ctx, new)]
    kc, vc, bt = _paged(g, BF, lens, Hq, G, dk, dv, nb=sum((n + 15) // 16 for n in lens) + 3)
    cu = _i32([0] + torch.tensor(new).cumsum(0).tolist())
    qkv = _r(g, sum(new), Hq * dk + 8, dt=BF)
    kw = dict(kw)
    sinks = _r(g, Hq) if kw.pop("sinks", False) else None
    gate = _r(g, sum(new), Hq + 8, dt=BF) if kw.pop("gate", False) else None
    a = (Hq, G, dk, dv, 1.0 / math.sqrt(dk), window, kw.pop("sink", False) or sinks is not None)
    want = H.window_attention_prefill(qkv, kc, vc, cu, _i32(ctx), bt, *a, sinks=sinks, gate=gate, g_col=8 if gate is not None else 0, **kw)
    dev = [x.cuda() for x in (qkv, kc, vc, cu, _i32(ctx), bt)]
    got = H.window_attention_prefill(*dev, *a, mfma=256, sinks=sinks.cuda() if sinks is not None else None,
                                     gate=gate.cuda() if gate is not None else None, g_col=8 if gate is not None else 0, **kw)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2e-2, atol=2e-2)
