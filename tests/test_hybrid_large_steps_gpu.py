"""Kernels that take the layer-list decoders' large prompt steps, against the fp32 torch form of the same operator at the
sizes where their tiles, chunks and segments begin and end."""
import math

import pytest
import torch
import torch.nn.functional as F

from k8s_llm_monitor_amd.ops import hybrid as hops

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
    want = hops.window_attention_prefill(qkv, kc, vc, cu, _i32(ctx), bt, *a, sinks=sinks, gate=gate, g_col=8 if gate is not None else 0, **kw)
    dev = [x.cuda() for x in (qkv, kc, vc, cu, _i32(ctx), bt)]
    got = hops.window_attention_prefill(*dev, *a, mfma=256, sinks=sinks.cuda() if sinks is not None else None,
                                     gate=gate.cuda() if gate is not None else None, g_col=8 if gate is not None else 0, **kw)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("H,R,dn,dr,dv,pages", [(4, 128, 96, 32, 128, 1), (3, 256, 32, 32, 64, 9), (2, 256, 96, 32, 128, 17), (2, 48, 12, 4, 20, 5)])
def test_latent_expand_and_rotate_heads(H, R, dn, dr, dv, pages):
    """Temporary pages from listed latent pages (in and out of order, a list that does not fill the last workgroup; the
    last case: matrix products).  Sums of R bf16 products in fp32, one rounding: 2^-8 of the value."""
    g = _g(62)
    pitch = (R + dr + 31) // 32 * 32
    kc = torch.cat([_r(g, 40, 16, R + dr, dt=BF), torch.zeros(40, 16, pitch - R - dr, dtype=BF)], -1)
    wk, wv = _r(g, H * dn, R, s=R ** -0.5, dt=BF), _r(g, H * dv, R, s=R ** -0.5, dt=BF)
    pl = torch.randperm(40, generator=g)[:pages].to(torch.int32)
    kt, vt = hops.latent_expand(kc, pl, wk, wv, H, R, dr)
    kg, vg = hops.latent_expand(kc.cuda(), pl.cuda(), wk.cuda(), wv.cuda(), H, R, dr)
    torch.testing.assert_close(kg.cpu().float(), kt.float(), rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(vg.cpu().float(), vt.float(), rtol=1e-2, atol=1e-2)
    for pairs in (False, True):
        x, pos = _r(g, 7, H * (dn + dr) + 8, dt=BF), torch.randint(0, 3000, (7,), generator=g, dtype=torch.int32)
        freq = hops.rotary_freq(1e4, dr, "cpu")
        a, b = x.clone(), x.clone().cuda()
        hops.rotate_heads(a, H, dn + dr, pos, freq, pairs, dn)
        hops.rotate_heads(b, H, dn + dr, pos.cuda(), freq.cuda(), pairs, dn)
        torch.testing.assert_close(b.cpu().float(), a.float(), rtol=1e-2, atol=1e-2)


def test_latent_portions_in_the_expanded_form(monkeypatch):
    """Portions of prompts beside a decode row, their keys expanded from cached and new latents, a layer that reads
    another's pages; against whole-sequence float64 results and the form over the latent cache."""
    import bitonex_oracle as O
    import test_bitonex_model as B
    from k8s_llm_monitor_amd.models.hybrid import LatentAttention

    cfg = B.make_cfg([B.lat(4, 32, 32, 64, 48, 128, 0.12, 1e4, mlp=B.dense(64)), B.lat(2, 96, 32, 128, 40, 128, 0.09, 1e4, kv_from=0)],
                     width=128, vocab=211, mult=0.35)
    w = O.random_weights(cfg, 9)
    t, u = B.toks(200, cfg["vocab"], 4), B.toks(120, cfg["vocab"], 5)
    calls = []
    real = LatentAttention._forward_expanded
    monkeypatch.setattr(LatentAttention, "_forward_expanded", lambda self, *a: calls.append(1) or real(self, *a))

    def run(min_rows, most=None):
        monkeypatch.setattr(LatentAttention, "EXPAND_MIN_ROWS", min_rows)
        rig = B.rig_for(cfg, w=w, device="cuda", dtype=BF, num_blocks=48)
        for m in rig.model.mixers:
            m.most_pages = most or m.most_pages
        a = rig.step([("a", t[:90]), ("b", u[:119])])
        b = rig.step([("a", t[90:161]), ("b", u[119:])], end=["b"])  # a portion behind 90 cached tokens, a decode row
        c = rig.step([("a", t[161:])], end=["a"])
        return torch.cat([a["a"], b["a"], c["a"]]), torch.cat([a["b"], b["b"]])

    ga, gb = run(32)
    assert len(calls) == 6
    ca, cb = run(32, 13)  # the first step's 6 and 8 pages in two groups; the cached sequence has 11, then 13
    assert len(calls) == 12
    assert torch.equal(ca, ga) and torch.equal(cb, gb)
    ha, hb = run(1 << 30)
    for got, form, ref in ((ga, ha, O.forward(cfg, w, t)), (gb, hb, O.forward(cfg, w, u))):
        B.close_most(got, ref, 0.05, frac=1.0)
        B.close_most(got, form.double(), 0.02, frac=1.0)


def _segments(lens, ctx, slot):
    return _i32([0] + torch.tensor(lens).cumsum(0).tolist()), _i32(ctx), _i32(slot)


def test_chunked_linear_attention_negative_decay():
    g = _g(64)
    cu, ctx, slot = _segments([70, 129], [0, 2], [1, 0])
    vkq, decay, state = _r(g, 199, 2 * (32 + 64), s=0.7, dt=BF), torch.tensor([-0.9, -1.0]), _r(g, 2, 2, 32, 32)
    want_s, got_s = state.clone(), state.cuda()
    want = hops.linear_attention(vkq, decay, want_s, cu, ctx, slot, 2, 32, 32)
    got = hops.linear_attention(vkq.cuda(), decay.cuda(), got_s, cu.cuda(), ctx.cuda(), slot.cuda(), 2, 32, 32, mode=3)
    for a, b in ((got.cpu(), want), (got_s.cpu(), want_s)):
        torch.testing.assert_close(a, b, rtol=2e-5, atol=2e-5 * float(b.abs().max()))
    scan = hops.linear_attention(vkq.cuda(), decay.cuda(), state.cuda(), cu.cuda(), ctx.cuda(), slot.cuda(), 2, 32, 32, mode=2)
    assert not torch.equal(got, scan)  # it was the chunked kernel


def test_forms_that_are_asked_for_run_or_raise():
    """A forced kernel that is not one for the call's sizes, form or alignment raises instead of leaving the call to another one."""
    g = _g(87)
    cu, ctx, slot = (v.cuda() for v in _segments([70], [0], [0]))

    def decay(mode, dk=32, per_head=True, shift=0, **kw):
        qkv, z = _r(g, 70, 3 * dk + shift, dt=BF).cuda()[:, shift:], _r(g, 70, 1 if per_head else dk, dt=BF).cuda()
        zb, st = _r(g, z.shape[1]).cuda(), torch.zeros(1, 1, dk, dk).cuda()
        if per_head:
            kw = dict(kw, beta=_r(g, 70, 1, dt=BF).cuda())
        return hops.decay_scan(qkv, 0, dk, 2 * dk, z, zb, st, cu, ctx, slot, 1, 1, dk, dk, 1.0, tau=2.0, mode=mode, **kw)

    for kw in (dict(mode=3), dict(mode=3, per_head=False), dict(mode=4, per_head=False)):
        decay(**kw)
    for kw in (dict(mode=4), dict(mode=3, dk=24), dict(mode=3, shift=1), dict(mode=3, per_head=False, unit=True), dict(mode=4, per_head=False, dk=160)):
        with pytest.raises(RuntimeError):
            decay(**kw)
    kc, vc, bt = (v.cuda() for v in _paged(g, BF, [20], 2, 1, 96, 64))
    q = _r(g, 20, 2 * 96, dt=BF).cuda()
    a = (_i32([0, 20]).cuda(), _i32([0]).cuda(), bt, 2, 1, 96, 64, 0.1, 0, False)
    hops.window_attention_prefill(q, kc, vc, *a)
    for x in ((q, kc, vc), (q.float(), kc.float(), vc.float())):
        with pytest.raises(RuntimeError):
            hops.window_attention_prefill(*x, *a, mfma=256)


@pytest.mark.parametrize("H,Gk,dk,dv", [(4, 2, 128, 128), (2, 2, 32, 16), (3, 1, 64, 48), (2, 1, 96, 32)])
@pytest.mark.parametrize("kind", ["slow", "fast", "root", "plain_keys"])
def test_chunked_delta_rule(H, Gk, dk, dv, kind):
    """The delta rule with one decay per head in chunks of 64 tokens: segments around the chunk size, continued ones, a padding
    one, decays near one and down to zero, keys that repeat (the triangular solve's worst case) and keys that are no unit
    vectors.  fp32 sums in another order through a recurrence of a few hundred tokens: 5e-5 of the result's scale."""
    g = _g(65)
    lens = [1, 63, 64, 65, 200, 7, 130, 128]
    cu, ctx, slot = _segments(lens, [0, 5, 0, 64, 0, 3, 9, 1], [0, 1, 2, 3, 4, -1, 5, 6])
    T = sum(lens)
    qkv = _r(g, T, 2 * Gk * dk + H * dv, dt=BF)
    qkv[100:160, Gk * dk:2 * Gk * dk] = qkv[100, Gk * dk:2 * Gk * dk]  # equal keys in a row
    kw = dict(unit=True, a_log=_r(g, H, s=0.5))
    if kind == "plain_keys":
        kw["unit"] = False
        qkv[:, :2 * Gk * dk] *= 0.7 * dk ** -0.5
    if kind == "root":
        kw = dict(unit=True, tau=4.0)
    z, zb = _r(g, T, H + 3, s=4.0 if kind == "fast" else 1.0, dt=BF), _r(g, H) - (4.0 if kind != "fast" else -1.0) * (1 if kind != "root" else -1)
    beta, state = _r(g, T, H + 2, dt=BF), _r(g, 7, H, dv, dk)
    want_s, got_s = state.clone(), state.cuda()
    a = (0, Gk * dk, 2 * Gk * dk)
    want = hops.decay_scan(qkv, *a, z, zb, want_s, cu, ctx, slot, H, Gk, dk, dv, dk ** -0.5, beta=beta, beta_col=2, z_col=3, **kw)
    dev = {k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in kw.items()}
    got = hops.decay_scan(qkv.cuda(), *a, z.cuda(), zb.cuda(), got_s, cu.cuda(), ctx.cuda(), slot.cuda(), H, Gk, dk, dv, dk ** -0.5,
                          beta=beta.cuda(), beta_col=2, z_col=3, mode=3, **dev)
    for x, y in ((got.cpu(), want), (got_s.cpu(), want_s)):
        torch.testing.assert_close(x, y, rtol=5e-5, atol=5e-5 * float(y.abs().max()))


@pytest.mark.parametrize("H,Gk,dk,dv", [(4, 4, 64, 64), (2, 2, 32, 16), (3, 3, 128, 48), (2, 2, 96, 32), (4, 2, 64, 128)])
@pytest.mark.parametrize("kind", ["bonus", "bonus_fast", "root", "softplus_fast"])
def test_chunked_channel_decays(H, Gk, dk, dv, kind):
    """Decays per key channel in chunks of 64 tokens, plain and with a bonus: segments around the chunk size and its sub-blocks
    of 16, continued ones, a padding one, channels that keep hundreds of tokens beside channels that forget at once (their
    sums leave the fp32 range of 2^x).  fp32 sums of a few hundred terms in another order: 2e-5 of the result's scale."""
    if kind.startswith("bonus") and Gk != H:
        pytest.skip("a bonus goes with a key head per head")
    g = _g(66)
    lens = [1, 63, 64, 65, 200, 7, 130, 128, 16, 17, 48]
    cu, ctx, slot = _segments(lens, [0, 5, 0, 64, 0, 3, 9, 1, 0, 2, 0], [0, 1, 2, 3, 4, -1, 5, 6, 7, 8, 9])
    T = sum(lens)
    qkv = _r(g, T, 2 * Gk * dk + H * dv, dt=BF)
    z, zb, state = _r(g, T, H * dk, s=2.0, dt=BF), _r(g, H * dk, s=2.0), _r(g, 10, H, dv, dk)
    kw = dict(decay="exp_exp", bonus=_r(g, H, dk)) if kind.startswith("bonus") else dict(tau=3.0) if kind == "root" else dict(a_log=_r(g, H) + 2.0)
    zb += {"bonus": -3.0, "bonus_fast": 2.0, "root": 3.0, "softplus_fast": 1.0}[kind]
    want_s, got_s = state.clone(), state.cuda()
    a = (0, Gk * dk, 2 * Gk * dk)
    want = hops.decay_scan(qkv, *a, z, zb, want_s, cu, ctx, slot, H, Gk, dk, dv, dk ** -0.5, **kw)
    dev = {k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in kw.items()}
    got = hops.decay_scan(qkv.cuda(), *a, z.cuda(), zb.cuda(), got_s, cu.cuda(), ctx.cuda(), slot.cuda(), H, Gk, dk, dv, dk ** -0.5, mode=3, **dev)
    for x, y in ((got.cpu(), want), (got_s.cpu(), want_s)):
        torch.testing.assert_close(x, y, rtol=2e-5, atol=2e-5 * float(y.abs().max()))


@pytest.mark.parametrize("C,N,long", [(40, 3, 700), (70, 16, 513), (33, 20, 300), (129, 64, 260), (20, 7, 384), (17, 130, 257), (1030, 66, 3700)])
def test_selective_scan_in_spans(C, N, long):
    """The selective recurrence with long segments cut into spans: segments around the spans' lengths (128; in the last case 256),
    continued ones, a padding one, a long one, odd channel and state counts, steps from near zero to such that forget at once.
    The CPU form rounds every product of decays as well: fp32 noise of a recurrence of hundreds of tokens, 2e-5 of the scale."""
    g = _g(67)
    lens = [1, 127, 128, 129, long, 7, 256, 255, 257]
    cu, ctx, slot = _segments(lens, [0, 5, 0, 64, 9, 3, 0, 1, 2], [0, 1, 2, 3, 4, -1, 5, 6, 7])
    T = sum(lens)
    xc, q, dt, pr = _r(g, T, C), _r(g, T, 2 * N + 3), _r(g, T, C, s=3.0), _r(g, T, C + 5)
    db, al, D, state = _r(g, C) - 2.0, _r(g, C, N), _r(g, C), _r(g, 8, C, N)
    want_s, got_s = state.clone(), state.cuda()
    want = hops.selective_scan(xc, q, 3, 3 + N, dt, db, al, D, pr, 5, want_s, cu, ctx, slot)
    dev = [v.cuda() for v in (xc, q, dt, db, al, D, pr, cu, ctx, slot)]
    got = hops.selective_scan(dev[0], dev[1], 3, 3 + N, *dev[2:7], 5, got_s, *dev[7:], longest=max(lens), mode=2)
    for x, y in ((got.cpu(), want), (got_s.cpu(), want_s)):
        torch.testing.assert_close(x, y, rtol=2e-5, atol=2e-5 * float(y.abs().max()))


@pytest.mark.parametrize("nh,P,N,G", [(4, 64, 128, 1), (3, 24, 40, 1), (2, 20, 64, 2), (2, 64, 256, 2), (2, 40, 136, 1), (8, 32, 72, 4)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("fixed", [False, True])
def test_state_scan_products_on_the_matrix_cores(nh, P, N, G, dt, fixed):
    """The long-segment scan with its products on the matrix cores gives the bits of the other long-segment mapping (which an
    input that is not 16-byte aligned takes), and the oracle's values within fp32 noise: segments around the tile of 32 tokens
    and the 256 tokens whose step sizes are computed at once, continued ones, a padding one."""
    g = _g(68)
    lens = [1, 31, 32, 33, 300, 7, 257, 64]
    cu, ctx, slot = _segments(lens, [0, 5, 0, 64, 9, 3, 0, 1], [0, 1, 2, 3, 4, -1, 5, 6])
    T, W = sum(lens), nh * P + 2 * G * N
    xbc, proj, state = _r(g, T, W, dt=dt), _r(g, T, nh + 3, dt=dt), _r(g, 7, nh, N, P)
    db, al, D = _r(g, nh) - 2.0, _r(g, nh, s=0.5), _r(g, nh)
    decay = torch.sigmoid(_r(g, nh) + 3.0) if fixed else None
    par = (None, 0, None, None, None) if fixed else (proj, 3, db, al, D)
    want_s = state.clone()
    want = hops.ssm_scan(xbc, *par, want_s, cu, ctx, slot, nh, P, N, G, decay=decay)
    dev = [v.cuda() if isinstance(v, torch.Tensor) else v for v in par]
    odd = torch.empty(T * W + 2, dtype=dt, device="cuda")[2:].view(T, W).copy_(xbc)
    assert odd.data_ptr() % 16 != 0
    res = []
    for x in (xbc.cuda(), odd):
        st = state.cuda()
        y = hops.ssm_scan(x, *dev, st, cu.cuda(), ctx.cuda(), slot.cuda(), nh, P, N, G, mode=2, decay=None if decay is None else decay.cuda())
        res.append((y.cpu(), st.cpu()))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    for a, b in zip(res[0], (want, want_s)):
        torch.testing.assert_close(a, b.view_as(a), rtol=2e-5, atol=2e-5 * float(b.abs().max()))


@pytest.mark.parametrize("C,col0,pad", [(2056, 8, 16), (64, 0, 0)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_conv_rows_of_large_steps(C, col0, pad, dt):
    """The convolution of a step whose threads take four rows each: segments that start anywhere in a group of four, of one row and of
    many, continued ones and a padding one, gives the bits of the same segments in steps too small for it."""
    g = _g(69)
    lens = [1, 2, 3, 4, 5, 130, 7, 200, 1, 1, 203]
    ctxs, slots = [0, 5, 0, 64, 9, 3, 0, 1, 0, 8, 2], [0, 1, 2, 3, 4, -1, 5, 6, 7, 8, 9]
    T = sum(lens)
    assert T >= 512
    proj, cw, cb, state = _r(g, T, col0 + C + pad, dt=dt).cuda(), _r(g, C, 4).cuda(), _r(g, C).cuda(), _r(g, 10, 3, C, dt=dt)
    sa, sb = state.cuda(), state.cuda()
    got = hops.conv_silu(proj, col0, C, cw, cb, sa, *(v.cuda() for v in _segments(lens, ctxs, slots)))
    r = 0
    for n, c, sl in zip(lens, ctxs, slots):
        want = hops.conv_silu(proj[r:r + n], col0, C, cw, cb, sb, *(v.cuda() for v in _segments([n], [c], [sl])))
        assert torch.equal(got[r:r + n], want)
        r += n
    assert torch.equal(sa, sb)


@pytest.mark.parametrize("rows,N,Kd", [(1, 64, 32), (63, 65, 64), (64, 128, 1024), (300, 200, 96), (65, 1, 160)])
@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
def test_fp32_grouped_gemm(rows, N, Kd, act):
    """Grouped fp32 products on the matrix cores: rows and columns around the 64 x 64 tile, an expert without rows, every activation,
    gathered and plain rows.  fp32 sums of Kd products of unit variance: 1e-6 sqrt(Kd) before the activation, which at most
    doubles it times the other factor."""
    g = _g(70)
    E, gated = 4, act in (1, 3)
    off = [0, rows // 3, rows // 3, rows - rows // 4, rows]
    a, w = _r(g, rows, Kd), _r(g, E, N * (2 if gated else 1), Kd)
    idx = torch.randperm(rows, generator=g).int()
    ext = hops.native()
    for sorted_idx in (None, idx):
        y = torch.empty(rows, N, device="cuda")
        ext.grouped_gemm(y, a.cuda(), w.cuda(), _i32(off).cuda(), None if sorted_idx is None else sorted_idx.cuda(), 1, act, False, True,
                         7.0 if act == 3 else 0.0)
        x = (a if sorted_idx is None else a[sorted_idx.long()]).double()
        z = torch.cat([x[off[e]:off[e + 1]] @ w[e].double().t() for e in range(E)])
        u, z = (z[:, N:], z[:, :N]) if gated else (z, z)
        lim = 7.0
        want = {0: lambda: z, 1: lambda: z * torch.sigmoid(z) * u, 2: lambda: torch.nn.functional.gelu(z), 4: lambda: z.clamp(min=0) ** 2,
                3: lambda: z.clamp(max=lim) * torch.sigmoid(1.702 * z.clamp(max=lim)) * (u.clamp(-lim, lim) + 1)}[act]()
        tol = 1e-6 * Kd ** 0.5 * 4 * (1 + z.abs().max() + u.abs().max())
        assert float((y.cpu().double() - want).abs().max()) <= float(tol)


@pytest.mark.parametrize("rows,N", [(70, 72), (700, 3000)])  # 64 and 128 columns a workgroup
def test_fp32_grouped_gemm_what_is_no_number(rows, N):
    """Infinities, NaN, values that a bf16 rounding takes to infinity and sums that overflow come out of the fp32 products as the CPU's
    fp32 has them, and nothing else is touched: within a unit in the last place of the largest sum for each of three steps of 32
    products and the last addition."""
    g, K, inf, nan = _g(90), 96, float("inf"), float("nan")
    a, w = _r(g, rows, K), _r(g, 1, N, K)
    a[0, 3], a[1, 40], a[2, 95], a[3, 7], a[4] = inf, nan, -inf, 3.4e38, 1e38
    w[0, 5, 3], w[0, 6, 3], w[0, 7, 50], w[0, 8, 9] = 0.0, -1.0, inf, 3.39e38
    w[0, 9] = 8.0
    got = torch.empty(rows, N, device="cuda")
    hops.native().grouped_gemm(got, a.cuda(), w.cuda(), _i32([0, rows]).cuda(), None, 1, 0, False, True, 0.0)
    want, z = a @ w[0].t(), a.double() @ w[0].double().t()
    got = got.cpu()
    assert got[4, 9] == inf  # elsewhere in this row the order of the sums decides what overflows
    got[4], want[4], z[4] = 0.0, 0.0, 0.0
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
    plain = torch.ones(rows, N, dtype=torch.bool)
    plain[:5], plain[:, 5:10] = False, False
    assert float((got.double() - z)[plain].abs().max()) <= 4 * 2 ** -23 * float(z[plain].abs().max())


@pytest.mark.parametrize("dk,dv,Hq,G", [(128, 128, 8, 2), (64, 128, 3, 1), (128, 64, 2, 2), (64, 64, 16, 2)])
@pytest.mark.parametrize("kw", [dict(window=0, sink=False), dict(window=5, sink=True), dict(window=40, sink=False, keep=3),
                                dict(window=33, sink=True, keep=20, cap=2.0), dict(window=32, sink=False, chunked=True)])
def test_fp32_window_attention(dk, dv, Hq, G, kw):
    """fp32 windowed attention on the matrix cores: chunks around the 16-row tile with and without a past, kept tokens before, inside
    and past the window, caps, sinks, gates, a padding row; the pages' unused ends hold NaN.  fp32 softmax sums: 2e-5."""
    g = _g(71)
    kw = dict(kw)
    new, ctx = [1, 15, 16, 17, 50, 3], [0, 37, 0, 130, 16, 250]
    lens = [a + b for a, b in zip(ctx, new)]
    W = max((n + 15) // 16 for n in lens)
    bt = torch.randperm(len(lens) * W, generator=g).int().view(-1, W)
    kc, vc = _r(g, bt.numel(), 16, G * dk), _r(g, bt.numel(), G, dv, 16)
    for row, n in zip(bt, lens):
        for j in range(n, W * 16):
            vc[row[j // 16].item(), :, :, j % 16] = float("nan")
            kc[row[j // 16].item(), j % 16] = float("nan")
    cu = _i32([0] + torch.tensor(new).cumsum(0).tolist())
    qkv, gate = _r(g, sum(new), Hq * dk + G * (dk + dv)), _r(g, sum(new), Hq)
    a = (Hq, G, dk, dv, dk ** -0.5, kw.pop("window"), kw.pop("sink"))
    want = hops.window_attention_prefill(qkv, kc, vc, cu, _i32(ctx), bt, *a, gate=gate, **kw)
    got = hops.window_attention_prefill(qkv.cuda(), kc.cuda(), vc.cuda(), cu.cuda(), _i32(ctx).cuda(), bt.cuda(), *a, gate=gate.cuda(), **kw)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-5, atol=2e-5)
    q1, bt1, sl = qkv[:7], torch.cat([bt, bt[:1]]), _i32(lens + [0])
    want = hops.window_attention_decode(q1, kc, vc, bt1, sl, *a, gate=gate[:7], **kw)
    got = hops.window_attention_decode(q1.cuda(), kc.cuda(), vc.cuda(), bt1.cuda(), sl.cuda(), *a, gate=gate[:7].cuda(), **kw)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("rows", [17, 40, 90])  # a mean of 8.5, 20, 45 rows an expert: 32, 32 and 64 rows a wave
@pytest.mark.parametrize("N,Kd", [(40, 32), (64, 288), (16, 1024)])
@pytest.mark.parametrize("act", [0, 1, 3])
def test_grouped_gemm_rows_per_wave(rows, N, Kd, act):
    """The bf16 weight-streaming products give the same bits however many rows of an expert a wave takes (experts without rows lower
    the mean that decides it), at K of less than one batch of loads, of a batch and a rest, and of several batches; and the
    oracle's values within the rounding of the bf16 result."""
    g = _g(72)
    gated = act in (1, 3)
    a, w = _r(g, rows, Kd, dt=BF), _r(g, 2, N * (2 if gated else 1), Kd, s=Kd ** -0.5, dt=BF)
    off = [0, rows // 3, rows]
    ext, res = hops.native(), []
    for E in (2, rows):
        y = torch.empty(rows, N, dtype=BF, device="cuda")
        wide = torch.cat([w, torch.zeros(E - 2, *w.shape[1:], dtype=BF)])
        ext.grouped_gemm(y, a.cuda(), wide.cuda(), _i32(off + [rows] * (E - 2)).cuda(), None, 1, act, False, True, 7.0 if act == 3 else 0.0)
        res.append(y.cpu())
    assert torch.equal(res[0], res[1])
    z = torch.cat([a[off[e]:off[e + 1]].float() @ w[e].float().t() for e in range(2)]).to(BF).float()
    u, z = (z[:, N:], z[:, :N]) if gated else (z, z)
    want = {0: lambda: z, 1: lambda: z * torch.sigmoid(z) * u,
            3: lambda: z.clamp(max=7) * torch.sigmoid(1.702 * z.clamp(max=7)) * (u.clamp(-7, 7) + 1)}[act]()
    torch.testing.assert_close(res[0].float(), want, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("rows,N", [(3, 40), (3, 8200), (33, 72), (33, 8200), (130, 136)])  # 16 rows by 2 and 4 waves, 32 by 2 and 4, 64 by 4
@pytest.mark.parametrize("Kd", [32, 256, 288, 1056])  # one step, a whole chunk of 8, a chunk and a rest, four chunks and a rest
@pytest.mark.parametrize("act,il", [(0, False), (1, False), (1, True)])
def test_grouped_gemm_tiles_keep_the_bits(rows, N, Kd, act, il):
    """Experts' products, rows gathered by index, give the same bits by every tile (one chain of products in the order of k): against the
    same rows beside an expert of 520 more, which brings the mean to 64 rows a tile; and the values of fp64 products within the
    roundings of gate, up and result."""
    if il:
        N = N // 64 * 64 or 64
    g = _g(75)
    more = 520
    a = _r(g, rows + more, Kd, dt=BF).cuda()
    w = _r(g, 3, N * (2 if act else 1), Kd, s=Kd ** -0.5, dt=BF).cuda()
    perm = torch.cat([torch.randperm(rows, generator=g), torch.arange(rows, rows + more)]).int().cuda()
    ext, off = hops.native(), [0, rows // 3, rows]
    few, many = (torch.empty(n, N, dtype=BF, device="cuda") for n in (rows, rows + more))
    ext.grouped_gemm(few, a[:rows], w[:2].contiguous(), _i32(off).cuda(), perm[:rows].contiguous(), 1, act, il, True, 0.0)
    ext.grouped_gemm(many, a, w, _i32(off + [rows + more]).cuda(), perm, 1, act, il, True, 0.0)
    assert torch.equal(few, many[:rows])
    z = torch.cat([a[perm[off[e]:off[e + 1]].long()].double() @ w[e].double().t() for e in range(2)])
    if act:
        z = z.view(rows, -1, 2, 64) if il else z.view(rows, 2, N)
        p, u = (z[:, :, i].reshape(rows, N) if il else z[:, i] for i in (0, 1))
        z = F.silu(p) * u
    torch.testing.assert_close(few.double(), z, rtol=2e-2, atol=1e-2)  # three roundings of 2^-9, gate and up of up to 4


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17])
@pytest.mark.parametrize("N,K", [(16, 32), (1, 96), (200, 512), (72, 2080), (1024, 4096), (24, 4128)])
def test_linear_of_few_rows(M, N, K):
    """Projections of a few rows against 64 bits: fewer steps of 32 k than waves, a rest, whole batches, columns around the tile of
    16, a slice of wider rows, and 32 k more than the kernel takes beside more than 4 rows.  fp32 sums, one bf16 rounding: 2^-8 of the
    value and 1e-6 sqrt(K) of what cancels."""
    g = _g(73)
    x, w = _r(g, M, K + 24, dt=BF).cuda()[:, 16:16 + K], _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    got, want = hops.linear(x, w).double(), x.double() @ w.double().t()
    assert got.shape == want.shape
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("T", [1, 5, 4099])  # one token a workgroup; up to 8 rows of weights in registers, four tokens a round with a rest
@pytest.mark.parametrize("E,K,shared", [(8, 2, 0), (7, 3, 1), (16, 4, 1), (70, 16, 0)])
def test_router_ranks(T, E, K, shared):
    """Routers: the K largest logits in order, the lower number first among equal ones (whole rows of ties), weights and the shared
    expert's gate.  Logits are fp32 sums: 1e-5."""
    g = _g(74)
    d = 136
    h, wr, bias = _r(g, T, d, dt=BF), _r(g, E + shared, d, s=d ** -0.5), _r(g, E)
    h[::3] = 0  # the bias alone decides there
    bias[1:4] = bias.max() + 1
    got = hops.moe_router(h.cuda(), wr.cuda(), bias.cuda(), E, K)
    want = torch.sort(bias, descending=True, stable=True).indices[:K]
    assert want[:3].tolist() == [1, 2, 3][:min(K, 3)] and bool((got[0][::3].cpu() == want).all())
    lg = h.float() @ wr[:E].t() + bias
    chosen = lg.gather(1, got[0].cpu().long())
    assert bool((chosen[:, :-1] >= chosen[:, 1:] - 1e-5).all()) and all(len(set(r)) == K for r in got[0].tolist())
    torch.testing.assert_close(chosen, lg.sort(1, descending=True).values[:, :K], rtol=0, atol=1e-5)
    torch.testing.assert_close(got[1].cpu(), chosen.softmax(1), rtol=1e-5, atol=1e-5)
    if shared:
        torch.testing.assert_close(got[2].cpu().view(-1), torch.sigmoid(h.float() @ wr[E]), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("over_all", [False, True])
def test_router_logits_that_are_no_numbers(over_all):
    """An expert whose logit is NaN is chosen first and the token's weights are NaN, as in the torch form: a fault in a router's weights
    does not pass unseen.  Infinite logits keep their place."""
    g = _g(88)
    E, K = 9, 2
    h, wr = _r(g, 5, 64, dt=BF), _r(g, E, 64, s=0.1)
    for e, bad in ((0, float("nan")), (4, float("nan")), (8, float("nan")), (4, float("-inf"))):
        bias = _r(g, E)
        bias[e] = bad
        want = hops.moe_router(h, wr, bias, E, K, over_all)
        got = hops.moe_router(h.cuda(), wr.cuda(), bias.cuda(), E, K, over_all)
        assert torch.equal(got[0].cpu(), want[0]) and torch.equal(got[1].cpu().isnan(), want[1].isnan())


@pytest.mark.parametrize("n,E", [(1, 1), (63, 8), (128, 8), (1000, 64), (1024, 5), (1025, 8), (700, 65)])
def test_expert_sort(n, E):
    """The counting sort of (token, expert) pairs around the limits of its one-pass form: stable, every pair once."""
    ids = torch.randint(0, E, (n, 1), generator=_g(75)).int()
    off, srt, inv = (torch.full((k,), -1, dtype=torch.int32, device="cuda") for k in (E + 1, n, n))
    hops.native().moe_align(ids.cuda(), E, off, srt, inv)
    want = torch.sort(ids.view(-1), stable=True).indices
    assert torch.equal(srt.cpu().long(), want) and torch.equal(inv.cpu().long(), torch.sort(want).indices)
    assert off.tolist() == [0] + torch.bincount(ids.view(-1).long(), minlength=E).cumsum(0).tolist()


@pytest.mark.parametrize("longest", [0, 300])
def test_scans_of_a_long_prompt_beside_single_tokens(longest):
    """One prompt of 300 rows after 40 single tokens, where a known longest segment brings the chunks to linear attention, the delta
    rule and decays per channel: both routes against the oracle.  Tolerances as for the chunks above: 2e-5, the delta rule 5e-5."""
    g = _g(76)
    lens = [1] * 40 + [300]
    cu, ctx, slot = _segments(lens, [3 + i for i in range(40)] + [0], list(range(41)))
    T, H, d = sum(lens), 2, 32
    dev = [v.cuda() for v in (cu, ctx, slot)]

    def check(f, state, tol):
        a, b = state.clone(), state.cuda()
        want, got = f(lambda v: v, a, cu, ctx, slot), f(lambda v: v.cuda(), b, *dev)
        for x, y in ((got.cpu(), want), (b.cpu(), a)):
            torch.testing.assert_close(x, y, rtol=tol, atol=tol * float(y.abs().max()))

    qkv, z, zb, beta, bonus = _r(g, T, 3 * H * d, dt=BF), _r(g, T, H * d, dt=BF), _r(g, H * d) - 3.0, _r(g, T, H, dt=BF), _r(g, H, d)
    lam, al = torch.sigmoid(_r(g, H) + 3.0), _r(g, H)
    check(lambda c, s, *seg: hops.linear_attention(c(qkv), c(lam), s, *seg, H, d, d, longest=longest), _r(g, 41, H, d, d), 2e-5)
    a = (0, H * d, 2 * H * d)
    check(lambda c, s, *seg: hops.decay_scan(c(qkv), *a, c(z[:, :H].contiguous()), c(zb[:H]), s, *seg, H, H, d, d, d ** -0.5, a_log=c(al), beta=c(beta),
                                             unit=True, longest=longest), _r(g, 41, H, d, d), 5e-5)
    check(lambda c, s, *seg: hops.decay_scan(c(qkv), *a, c(z), c(zb), s, *seg, H, H, d, d, 1.0, decay="exp_exp", bonus=c(bonus),
                                             longest=longest), _r(g, 41, H, d, d), 2e-5)


@pytest.mark.parametrize("dk,dv", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("Hq,G", [(3, 3), (4, 2), (4, 1), (16, 2)])  # 1, 2, 4, 8 heads per kv head
def test_decode_attention_row_broadcasts(dk, dv, Hq, G):
    """bf16 decode attention whose multiply-adds pick queries and weights from their 16-lane row: lengths around pages, tiles of 64 and
    a round of all waves, windows, kept tokens, caps, sinks.  bf16 rounding of the result: 2e-2; fp32 inside, so against the
    oracle on the same bf16 values half a unit in the last place and a few more."""
    g = _g(77)
    lens = [1, 15, 16, 17, 63, 64, 65, 500, 600, 0]
    W = max((n + 15) // 16 for n in lens)
    bt = torch.randperm(len(lens) * W, generator=g).int().view(-1, W)
    kc, vc = _r(g, bt.numel(), 16, G * dk, dt=BF), _r(g, bt.numel(), G, dv, 16, dt=BF)
    q, gate, sl = _r(g, len(lens), Hq * dk + G * (dk + dv), dt=BF), _r(g, len(lens), Hq, dt=BF), _i32(lens)
    for window, sink, kw in ((0, False, {}), (70, True, dict(keep=20)), (64, False, dict(chunked=True, cap=2.0))):
        a = (Hq, G, dk, dv, dk ** -0.5, window, sink)
        want = hops.window_attention_decode(q, kc, vc, bt, sl, *a, gate=gate, **kw)
        got = hops.window_attention_decode(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(), sl.cuda(), *a, gate=gate.cuda(), **kw)
        torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1e-2, atol=2e-3)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])  # one, two and four row tiles
@pytest.mark.parametrize("f,rest,K", [(16, 0, 32), (48, 40, 96), (112, 24, 288), (32, 200, 2080)])
@pytest.mark.parametrize("shared", [False, True])
def test_few_rows_forms(M, f, rest, K, shared):
    """Both forms of a few rows' projection, plain, with a unit at its end and as capped fp32 logits, against 64 bits: fewer steps
    of 32 k than waves, a chunk of 8 and a rest, columns around the tile, a slice of wider rows.  fp32 sums, one bf16 rounding: 2^-8 of
    the value and 1e-6 sqrt(K) of what cancels; what a unit makes of two rounded products of up to 4: 2e-2."""
    g = _g(76)
    x, w = _r(g, M, K + 24, dt=BF).cuda()[:, 16:16 + K], _r(g, 2 * f + rest, K, s=K ** -0.5, dt=BF).cuda()
    N, z, ext = 2 * f + rest, x.double() @ w.double().t(), hops.native()

    def out(n, dt=BF):
        return torch.full((M, n), float("nan"), dtype=dt, device="cuda")

    y = out(N)
    ext.few_rows(y, None, x, w, -1, 0.0, shared)
    assert bool(((y.double() - z).abs() <= 2 ** -8 * z.abs() + 1e-6 * K ** 0.5).all())
    for cap in (0.0, 3.0):
        q = out(N, torch.float32)
        ext.few_rows(q, None, x, w, -1, cap, shared)
        torch.testing.assert_close(q, cap * torch.tanh(y.float() / cap) if cap else y.float(), rtol=1e-6, atol=1e-6)
    for kind in ("relu_sq", "tanh"):
        q = out(N)
        ext.few_rows(q, None, x, w, 16 + hops.ACTS[kind], 0.0, shared)
        assert torch.equal(q, hops.activation(y, kind))
    for kind in ("gelu_tanh", "silu", "relu"):
        a, q = out(f), out(rest)
        ext.few_rows(q, a, x, w, hops.ACTS[kind], 0.0, shared)
        assert torch.equal(a, hops.glu(y, 0, f, kind)) and torch.equal(q, y[:, 2 * f:])


@pytest.mark.parametrize("K", [64, 160, 512, 544, 1088, 8192])  # lines of 64 k: one, two and a half, a wave's last one half, chunks of four and a rest
@pytest.mark.parametrize("M", [3, 24, 50])
def test_few_rows_and_experts_in_lines(M, K):
    """Both forms and the experts' kernel, which read weights in lines of 64 k, against 64 bits; rows and weights end where their
    allocations do.  fp32 sums, one bf16 rounding: 2^-8 of the value and 1e-6 sqrt(K) of what cancels."""
    g = _g(77)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, 88, K, s=K ** -0.5, dt=BF).cuda()
    z, ext = x.double() @ w.double().t(), hops.native()
    y = torch.full((3, M, 88), float("nan"), dtype=BF, device="cuda")
    for shared in (False, True):
        ext.few_rows(y[int(shared)], None, x, w, -1, 0.0, shared)
    ext.grouped_gemm(y[2], x, w.view(1, 88, K), torch.tensor([0, M], dtype=torch.int32, device="cuda"), None, 1, 0, False, True, 0.0)
    assert bool(((y.double() - z).abs() <= 2 ** -8 * z.abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("M,K", [(5, 448), (30, 448), (64, 448), (30, 480)])
@pytest.mark.parametrize("shared", [False, True])
def test_few_rows_of_weights_read_once(M, K, shared):
    """Weights of more than 8 MB, which are loaded non-temporal where their rows begin at cache lines, and the same in halves, which are not: the
    same bits, and near 64 bits as above."""
    g = _g(98)
    N = 10304
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    assert 2 * w.numel() > 8 << 20 > w.numel()
    y = torch.full((2, M, N), float("nan"), dtype=BF, device="cuda")
    hops.native().few_rows(y[0], None, x, w, -1, 0.0, shared)
    for a in (0, N // 2):
        h = torch.empty(M, N // 2, dtype=BF, device="cuda")
        hops.native().few_rows(h, None, x, w[a:a + N // 2], -1, 0.0, shared)
        y[1, :, a:a + N // 2] = h
    z = x.double() @ w.double().t()
    assert torch.equal(y[0], y[1]) and bool(((y[0].double() - z).abs() <= 2 ** -8 * z.abs() + 1e-6 * K ** 0.5).all())


def _singles(g, n):
    """Segments, cached tokens and slots of a decode step: a fresh sequence, a padding row and, at last, no token beside two of one sequence."""
    ctx = torch.randint(1, 900, (n,), generator=g)
    slot = torch.randperm(n + 2, generator=g)[:n]
    ctx[0], slot[1] = 0, -1
    cu = torch.arange(n + 1)
    cu[n - 2 + 1] = cu[n - 2]
    return _i32(cu.tolist()).cuda(), _i32(ctx.tolist()).cuda(), _i32(slot.tolist()).cuda()


def _same_step(f, state):
    """The step kernel (mode 0) and the scan (mode 1): the same results and states, whatever a slot held that starts fresh."""
    state[:] = torch.where(torch.rand(state.shape[0], device="cuda").view(-1, *[1] * (state.dim() - 1)) < 0.2, float("nan"), state)
    a, b = state.clone(), state.clone()
    ya, yb = f(a, 0), f(b, 1)
    torch.testing.assert_close(ya, yb, rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("n", [3, 66])
@pytest.mark.parametrize("nh,P,N,G", [(4, 64, 128, 1), (2, 100, 16, 2), (6, 4, 36, 3), (2, 128, 256, 1), (3, 72, 100, 3), (256, 64, 128, 1)])
def test_one_token_a_segment_ssm(n, nh, P, N, G, dt):
    """Decode steps of the Mamba-2 recurrence: values and states around the workgroup's 64 and the groups of four, every sum as in the scan."""
    if nh * n > 1000 and dt == torch.float32:
        pytest.skip("the largest states once")
    g = _g(78)
    cu, ctx, slot = _singles(g, n)
    C = nh * P + 2 * G * N
    x, proj, par = _r(g, n, C, dt=dt).cuda(), _r(g, n, nh + 3, dt=dt).cuda(), [_r(g, nh).cuda() for _ in range(3)]
    state = _r(g, n + 2, nh, N, P).cuda()
    _same_step(lambda s, mode: hops.ssm_scan(x, proj, 3, *par, s, cu, ctx, slot, nh, P, N, G, mode=mode), state)
    if G == nh or G == 1:
        xx = _r(g, n, nh * P + 2 * nh * N, dt=dt).cuda()
        dec = torch.rand(nh, generator=g).cuda()
        _same_step(lambda s, mode: hops.linear_attention(xx, dec, s, cu, ctx, slot, nh, N, P, mode=mode), state)


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("n,H,Gk,dk,dv", [(3, 4, 2, 128, 128), (40, 16, 16, 64, 64), (24, 40, 20, 128, 128), (5, 2, 1, 96, 20), (30, 32, 32, 8, 300),
                                          (9, 16, 16, 256, 72), (130, 32, 32, 64, 64), (6, 32, 16, 128, 128)])
def test_one_token_a_segment_decay(n, H, Gk, dk, dv, dt):
    """Decode steps of the recurrences with decays, one and four rows of the state a lane: the delta rule with decays per channel and per
    head, plain, with a bonus; every sum as in the scan."""
    g = _g(79)
    cu, ctx, slot = _singles(g, n)
    cols = 2 * Gk * dk + H * dv
    x, z, beta = _r(g, n, cols + 8, dt=dt).cuda(), _r(g, n, H * dk, dt=dt).cuda(), _r(g, n, H, dt=dt).cuda()
    zb, al, state = _r(g, H * dk).cuda(), _r(g, H).cuda(), _r(g, n + 2, H, dv, dk).cuda()
    args = (x, 0, Gk * dk, 2 * Gk * dk)

    def run(zz, bias, **kw):
        _same_step(lambda s, mode: hops.decay_scan(*args, zz, bias, s, cu, ctx, slot, H, Gk, dk, dv, dk ** -0.5, mode=mode, **kw), state)

    run(z, zb, a_log=al, beta=beta, unit=True)
    run(z[:, :H].contiguous(), zb[:H].contiguous(), a_log=al, beta=beta, unit=True)
    run(z, zb, tau=16.0)
    if Gk == H:
        run(z, zb, decay="exp_exp", bonus=_r(g, H, dk).cuda())


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("n,C,N", [(3, 70, 16), (24, 1000, 16), (5, 33, 4), (4, 65, 8), (6, 100, 24), (5, 40, 64), (3, 20, 256), (70, 8192, 16)])
def test_one_token_a_segment_selective(n, C, N, dt):
    g = _g(80)
    cu, ctx, slot = _singles(g, n)
    xc, q, d, proj = (_r(g, n, w, dt=dt).cuda() for w in (C, 2 * N + 5, C, 2 * C))
    par = (_r(g, C).cuda(), _r(g, C, N).cuda(), _r(g, C).cuda())
    _same_step(lambda s, mode: hops.selective_scan(xc, q, 5, 5 + N, d, *par, proj, C, s, cu, ctx, slot, mode=mode), _r(g, n + 2, C, N).cuda())


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("n,C,bias", [(3, 8, True), (24, 2056, False), (66, 4352, True)])
def test_one_token_a_segment_conv(n, C, bias, dt):
    """The decode steps' convolution with its history, against the launches of steps with a longer segment (here of five rows behind
    the others): the same bits in rows and slots; a fresh sequence, a padding row, no row beside two of one sequence."""
    g = _g(81)
    cu, ctx, slot = _singles(g, n)
    proj, w, b = _r(g, n + 5, C + 24, dt=dt).cuda(), _r(g, C, 4).cuda(), _r(g, C).cuda() if bias else None
    a = _r(g, n + 3, 3, C, dt=dt).cuda()
    b2 = a.clone()
    got = hops.conv_silu(proj[:n], 16, C, w, b, a, cu, ctx, slot)

    def more(t, v):
        return torch.cat([t, torch.tensor([v], dtype=torch.int32, device="cuda")])

    want = hops.conv_silu(proj, 16, C, w, b, b2, more(cu, n + 5), more(ctx, 0), more(slot, n + 2))
    a[n + 2] = b2[n + 2]
    assert torch.equal(got, want[:n]) and torch.equal(a, b2)


@pytest.mark.parametrize("n,d", [(1, 1024), (30, 4096), (7, 2052), (255, 3000), (256, 2048)])
def test_token_mix_of_few_rows(n, d):
    """Rows over one or several workgroups: fp32 products of the torch form (a difference, a product and a sum: 3e-7 of values up to 10)."""
    g = _g(82)
    cu, ctx, slot = _i32(list(range(n + 1))), torch.randint(0, 3, (n,), generator=g).int(), torch.randperm(n, generator=g).int()
    h, mu, st = _r(g, n, d), _r(g, 5, d), _r(g, n, d)
    sg = st.clone().cuda()
    want = hops.token_mix(h, mu, st, cu, ctx, slot, torch.float32)
    got = hops.token_mix(h.cuda(), mu.cuda(), sg, cu.cuda(), ctx.cuda(), slot.cuda(), torch.float32)
    torch.testing.assert_close(got.cpu(), want, rtol=1e-6, atol=3e-6)
    assert torch.equal(sg.cpu(), st)


@pytest.mark.parametrize("M", [1, 257, 600])
@pytest.mark.parametrize("f,rest,K", [(128, 0, 192), (144, 48, 256), (400, 272, 320), (16, 256, 192)])  # tiles of 128 features and 256 columns
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "relu"])
def test_gated_unit_in_the_tile_gemm(M, f, rest, K, kind):
    """The tile GEMM's gated unit and the rows behind it against 64 bits: whole and partial tiles of both.  Two rounded factors and a
    rounded product: 2^-7 of it, and 2^-8 of each factor's unit scale where the other is small."""
    from k8s_llm_monitor_amd import ops

    g = _g(91)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, 2 * f + rest, K, s=K ** -0.5, dt=BF).cuda()
    a, y = (torch.full((M, n), float("nan"), dtype=BF, device="cuda") for n in (f, rest))
    ops.native().gemm_tile_unit(a, y, x, w, hops.TILE_UNITS[kind])
    z = x.double() @ w.double().t()
    p, u = z[:, :f], z[:, f:2 * f]
    t = {"gelu_tanh": lambda v: F.gelu(v, approximate="tanh"), "silu": F.silu, "relu": F.relu}[kind](p)
    assert bool(((a.double() - t * u).abs() <= 2 ** -7 * (t * u).abs() + 2 ** -8 * (t.abs() + 1.2 * p.abs() * u.abs()) + 1e-5).all())
    assert bool(((y.double() - z[:, 2 * f:]).abs() <= 2 ** -8 * z[:, 2 * f:].abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "relu"])
def test_tile_gemm_units_of_large_factors(kind):
    """Gates far below zero beside ups whose product with them has no fp32, large gates, infinities and NaN: what the unit's own launch
    makes of the same products (one nonzero term each, exact), to the rounding of the result."""
    from k8s_llm_monitor_amd import ops

    f, K, inf, nan = 16, 192, float("inf"), float("nan")
    gate = torch.tensor([-1e20, -3e38, -100.0, -1e20, 1e20, 3e38, 0.0, -0.0, inf, -inf, nan, 2.0, -1e20, 50.0, -50.0, 1.0])
    up = torch.tensor([1e20, 1e10, 1e38, -3e38, 1e10, 0.5, inf, 3e38, 2.0, 2.0, 1.0, nan, inf, -3e38, 3e38, 0.0])
    w = torch.zeros(2 * f, K)
    w[:, 0] = torch.cat([gate, up])
    w, x = w.to(BF).cuda(), torch.zeros(3, K, dtype=BF, device="cuda")
    x[:, 0] = 1.0
    a, y = torch.empty(3, f, dtype=BF, device="cuda"), torch.empty(3, 0, dtype=BF, device="cuda")
    ops.native().gemm_tile_unit(a, y, x, w, hops.TILE_UNITS[kind])
    want = hops.glu((x.double() @ w.double().t()).to(BF), 0, f, kind)
    torch.testing.assert_close(a, want, rtol=2 ** -7, atol=1e-30, equal_nan=True)


@pytest.mark.parametrize("M,N,K", [(1, 16, 192), (300, 272, 256), (256, 512, 320)])
def test_squared_relu_in_the_tile_gemm(M, N, K):
    from k8s_llm_monitor_amd import ops

    g = _g(92)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    y = torch.empty(M, N, dtype=BF, device="cuda")
    ops.native().gemm_tile_unit(y, None, x, w, hops.TILE_UNITS["relu_sq"])
    z = torch.relu(x.double() @ w.double().t())
    assert bool(((y.double() - z ** 2).abs() <= 3 * 2 ** -8 * z ** 2 + 1e-5).all())  # twice the rounding of z, once that of its square


@pytest.mark.parametrize("M", [4, 17, 64])
def test_gradients_of_few_rows_products(M):
    """A product or logits that a backward is wanted of stay the library's, which has one: gradients of a sum against the operands."""
    g = _g(96)
    x, w = _r(g, M, 64, dt=BF).cuda(), _r(g, 48, 64, dt=BF).cuda()
    for f in (hops.linear, hops.logits):
        xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
        f(xg, wg).float().sum().backward()
        torch.testing.assert_close(xg.grad.float(), w.float().sum(0).expand(M, 64), rtol=1e-2, atol=1e-2)
        torch.testing.assert_close(wg.grad.float(), x.float().sum(0).expand(48, 64), rtol=1e-2, atol=1e-2)
        with torch.no_grad():
            assert not f(xg, wg).requires_grad


@pytest.mark.parametrize("lens", [[130, 0, 64, 5, 5, 257, 1], [70] * 5, [9 * (i % 8) for i in range(64)], [9 * (i % 8) for i in range(65)], [300]])
def test_segments_in_turn(lens):
    """Prompts of all lengths (equal and empty ones, a table of 64 entries and one more), which the scans take longest and shortest in turn: each is
    taken once.  A prompt alone in its step has the same bits."""
    g = _g(79)
    S, H, d, C, N = len(lens), 5, 64, 640, 16
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    ctx, slot, T = _i32([0] * S).cuda(), _i32(list(range(S))).cuda(), sum(lens)
    vkq, dec = _r(g, T, 3 * H * d, dt=BF).cuda(), torch.rand(H, generator=g).cuda()
    x, q, dt, z = (_r(g, T, n, s=0.3, dt=BF).cuda() for n in (C, 2 * N, C, C))
    bias, a_log, D = _r(g, C, s=0.3).cuda(), _r(g, C, N, s=0.3).cuda(), _r(g, C).cuda()

    def run(a, b, s0, s1):
        seg = ((cu[s0:s1 + 1] - cu[s0]).contiguous(), ctx[s0:s1], slot[s0:s1])
        st1, st2 = torch.zeros(S, H, d, d, device="cuda"), torch.zeros(S, C, N, device="cuda")
        o1 = hops.linear_attention(vkq[a:b], dec, st1, *seg, H, d, d, mode=3, col_tiles=1)
        o2 = hops.selective_scan(x[a:b], q[a:b], 0, N, dt[a:b], bias, a_log, D, z[a:b], 0, st2, *seg, mode=1)
        return o1, o2, st1[s0:s1], st2[s0:s1]

    whole = run(0, T, 0, S)
    for s, n in enumerate(lens):
        if n and (s < 8 or s > S - 3):
            a = int(cu[s])
            for got, want in zip(run(a, a + n, s, s + 1), whole):
                assert torch.equal(got, want[a:a + n] if got.shape[0] == n and want.shape[0] == T else want[s:s + 1])


@pytest.mark.parametrize("lens", [[130, 0, 64, 5, 5, 257, 1, 90, 65, 3, 700], [70] * 12, [9 * (i % 8) for i in range(42)], [(i * 37) % 150 for i in range(43)],
                                  [4200 if i == 5 else (i * 53) % 120 for i in range(20)]])
def test_segments_in_turn_over_rounds(lens):
    """More workgroups (24 a segment) than units, up to four rounds of them and one segment more: linear attention, the delta rule, decays per channel with
    a bonus and, of 20 workgroups a segment, the selective scan.  A prompt alone in its step, which no choice is made for, has the same bits."""
    g = _g(80)
    S, H, dk, dv, C, N = len(lens), 24, 32, 16, 1280, 16
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    ctx, slot, T = _i32([0] * S).cuda(), _i32([i if i != 4 else -1 for i in range(S)]).cuda(), sum(lens)  # the fifth is padding
    qkv, z, beta = _r(g, T, H * (2 * dk + dv), dt=BF).cuda(), _r(g, T, H * dk, dt=BF).cuda(), _r(g, T, H, dt=BF).cuda()
    dec, zb, al, u = torch.rand(H, generator=g).cuda(), _r(g, H * dk).cuda(), _r(g, H).cuda(), _r(g, H, dk).cuda()
    x, q, dt, gate = (_r(g, T, n, s=0.3, dt=BF).cuda() for n in (C, 2 * N, C, C))
    bias, a_log, D = _r(g, C, s=0.3).cuda(), _r(g, C, N, s=0.3).cuda(), _r(g, C).cuda()

    def run(s0, s1):
        a, b = int(cu[s0]), int(cu[s1])
        seg, at = ((cu[s0:s1 + 1] - cu[s0]).contiguous(), ctx[s0:s1], slot[s0:s1]), (0, H * dk, 2 * H * dk)
        st = [torch.zeros(S, H, *n, device="cuda") for n in ((dk, dv), (dv, dk), (dv, dk))] + [torch.zeros(S, C, N, device="cuda")]
        out = [hops.linear_attention(qkv[a:b], dec, st[0], *seg, H, dk, dv, mode=3),
               hops.decay_scan(qkv[a:b], *at, z[a:b, :H].contiguous(), zb[:H].contiguous(), st[1], *seg, H, H, dk, dv, dk ** -0.5, a_log=al, beta=beta[a:b],
                               unit=True, mode=3),
               hops.decay_scan(qkv[a:b], *at, z[a:b], zb, st[2], *seg, H, H, dk, dv, 1.0, decay="exp_exp", bonus=u, mode=3),
               hops.selective_scan(x[a:b], q[a:b], 0, N, dt[a:b], bias, a_log, D, gate[a:b], 0, st[3], *seg, mode=1)]
        return out, [t[s0:s1] for t in st]

    whole, states = run(0, S)
    for s, n in enumerate(lens):
        if n and (s < 8 or s > S - 3):
            a = int(cu[s])
            out, st = run(s, s + 1)
            for got, want in zip(out + st, [w[a:a + n] for w in whole] + [w[s:s + 1] for w in states]):
                assert torch.equal(got, want)


@pytest.mark.parametrize("M", [1, 24, 64])
@pytest.mark.parametrize("N,K,shared", [(2056, 2048, True), (1544, 4096, True), (520, 8192, False), (264, 16384, False), (1100, 16384, True),  # below 128
                                        (8136, 2048, True), (8120, 2048, True), (8200, 6144, True), (2040, 8192, False), (2024, 8192, False), (2056, 16384, False)])
def test_few_rows_from_a_k_of_their_own(M, N, K, shared):
    """Weights above 8 MB with rows of whole 4 KB: each workgroup begins at another k where there are 128 and more.  Against 64 bits, fp32 sums of K products
    and one rounding; the columns' workgroups are more than the pieces of K and end inside a tile."""
    g = _g(75)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    y = torch.empty(M, N, dtype=BF, device="cuda")
    hops.native().few_rows(y, None, x, w, -1, 0.0, shared)
    want = x.double() @ w.double().t()
    assert bool(((y.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("M,N,K", [(4, 72, 6144), (5, 72, 6144), (2, 72, 6176), (3, 4096, 4128), (3, 4104, 4128), (16, 8200, 1056), (17, 8184, 1056),
                                   (32, 72, 4096), (33, 72, 4096), (33, 2048, 2048), (33, 2064, 2048), (64, 1024, 96), (65, 1024, 96),
                                   (16, 8192, 4096), (16, 10240, 4096), (64, 16384, 64), (64, 16400, 64)])
def test_linear_at_the_limits_of_its_kernels(M, N, K):
    """Products on both sides of each limit of the rule of few rows, against 64 bits, as above."""
    g = _g(77)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    got, want = hops.linear(x, w).double(), x.double() @ w.double().t()
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("M,N,K", [(1, 40, 96), (64, 8200, 288), (65, 8200, 288), (16, 40, 40), (512, 25616, 192), (511, 25616, 192), (300, 25616, 192)])
@pytest.mark.parametrize("kind", ["relu_sq", "tanh"])
def test_linear_act(M, N, K, kind):
    """A product with an activation behind it, by a few-row kernel, the tile GEMM with partial tiles of rows and columns, and the library, against 64 bits:
    the product's rounding through the activation, 2^-8 of its slope, and the result's."""
    g = _g(79)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=K ** -0.5, dt=BF).cuda()
    z = x.double() @ w.double().t()
    want, slope = (torch.relu(z) ** 2, 2 * torch.relu(z)) if kind == "relu_sq" else (torch.tanh(z), 1 - torch.tanh(z) ** 2)
    tol = 1.1 * 2 ** -8 * (want.abs() + slope * z.abs()) + 1e-4
    assert bool(((hops.linear_act(x, w, kind).double() - want).abs() <= tol).all())


@pytest.mark.parametrize("M,f,rest", [(1, 4112, 24), (33, 4112, 24), (64, 208, 0), (65, 208, 24), (512, 12816, 48), (450, 12816, 48), (300, 12816, 48)])
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "relu"])
def test_linear_glu_by_every_kernel(M, f, rest, kind):
    """Gated units through ``linear_glu`` on both sides of its rules, the large ones with partial tiles of rows, features and the rest, against 64
    bits: two rounded factors and a rounded product (as in test_gated_unit_in_the_tile_gemm)."""
    g, K = _g(80), 192
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, 2 * f + rest, K, s=K ** -0.5, dt=BF).cuda()
    a, y, col = hops.linear_glu(x, w, f, kind)
    z = x.double() @ w.double().t()
    p, u = z[:, :f], z[:, f:2 * f]
    t = {"gelu_tanh": lambda v: F.gelu(v, approximate="tanh"), "silu": F.silu, "relu": F.relu}[kind](p)
    assert bool(((a.double() - t * u).abs() <= 2 ** -7 * (t * u).abs() + 2 ** -8 * (t.abs() + 1.2 * p.abs() * u.abs()) + 1e-5).all())
    r = z[:, 2 * f:]
    assert bool(((y[:, col:col + rest].double() - r).abs() <= 2 ** -8 * r.abs() + 1e-6 * K ** 0.5).all())


@pytest.mark.parametrize("M,N", [(1, 200), (3, 8200), (64, 8200), (65, 8200)])
@pytest.mark.parametrize("scale,cap", [(1.0, 0.0), (1.0, 3.0), (0.25, 0.0), (0.25, 3.0)])
def test_logits(M, N, scale, cap):
    """fp32 logits of the rounded product, scaled and capped, in one launch and in several: exact but for the product's rounding, 2^-8 of it, and
    1e-6 of the cap's tanh."""
    g, K = _g(100), 288
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, s=2 * K ** -0.5, dt=BF).cuda()
    z = scale * (x.double() @ w.double().t())
    got = hops.logits(x, w, scale, cap)
    assert got.dtype == torch.float32
    want = cap * torch.tanh(z / cap) if cap else z
    assert bool(((got.double() - want).abs() <= 2 ** -8 * z.abs() + 1e-5).all())


@pytest.mark.parametrize("M", [1, 17, 40, 65, 512])
def test_gated_units_that_no_projection_ends_with(M):
    """What is no gated unit of ``glu`` is refused as ``glu`` refuses it, whatever kernel the step's size would choose."""
    g = _g(93)
    f = 96 if M < 512 else 12800  # 512 rows: 200 tiles
    x, w = _r(g, M, 192, dt=BF).cuda(), _r(g, 2 * f, 192, s=192 ** -0.5, dt=BF).cuda()
    for kind in ("clamped_swish", "relu_sq", "tanh"):
        with pytest.raises(RuntimeError, match="glu: columns / kind"):
            hops.linear_glu(x, w, f, kind)


def test_linear_of_nothing():
    """Empty sums, no columns, no rows and no gated unit are what the library makes of them."""
    g = _g(89)
    for M, N, K in ((3, 8, 0), (3, 0, 64), (0, 8, 64)):
        x, w = _r(g, M, K, dt=BF).cuda(), _r(g, N, K, dt=BF).cuda()
        assert torch.equal(hops.linear(x, w), torch.nn.functional.linear(x, w))
    x, w = _r(g, 2, 64, dt=BF).cuda(), _r(g, 24, 64, dt=BF).cuda()
    a, y, col = hops.linear_glu(x, w, 0, "silu")
    assert a.shape == (2, 0) and torch.equal(y[:, col:], hops.linear(x, w))


@pytest.mark.parametrize("E", [64, 65, 128, 129, 200])  # one after another; 64 at a time, whole and broken
@pytest.mark.parametrize("rows", [1, 70, 700, 4000])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_experts_by_their_number(E, rows, dt):
    """Every row tile finds its expert, with none, one and many rows in the others, the last and the first: against the rows' own products in
    64 bits, to the rounding of the result (bf16) or 2e-7 of sums of 32 products of order one (1e-5)."""
    g = _g(98)
    a, w = _r(g, rows, 32, dt=dt), _r(g, E, 16, 32, dt=dt)
    for pick in (torch.randint(0, E, (rows,), generator=g), torch.full((rows,), E - 1), torch.zeros(rows, dtype=torch.int64),
                 torch.where(torch.rand(rows, generator=g) < 0.9, E // 2, torch.randint(0, E, (rows,), generator=g))):
        e = pick.sort().values
        off = torch.cat([torch.zeros(1, dtype=torch.int64), torch.bincount(e, minlength=E).cumsum(0)]).int()
        y = torch.full((rows, 16), float("nan"), dtype=dt, device="cuda")
        hops.native().grouped_gemm(y, a.cuda(), w.cuda(), off.cuda(), None, 1, 0, False, True, 0.0)
        want = torch.einsum("rk,rnk->rn", a.double(), w.double()[e])
        torch.testing.assert_close(y.cpu().double(), want, rtol=2 ** -8, atol=1e-5) if dt == BF else torch.testing.assert_close(y.cpu().double(), want, rtol=0, atol=1e-5)


def test_experts_of_very_many_rows():
    """More row tiles than a grid's second dimension holds (65535 of 64 rows): the bits of the same rows in smaller calls."""
    g, rows, K, N = _g(97), 64 * 65600, 32, 32
    a, w = _r(g, 4096, K, dt=BF).cuda(), _r(g, 2, N, K, dt=BF).cuda()
    idx = torch.randint(0, 4096, (rows,), generator=g, dtype=torch.int32).cuda()
    a = a[idx.long()]
    y, few = torch.empty(rows, N, dtype=BF, device="cuda"), torch.empty(1000, N, dtype=BF, device="cuda")
    off = [0, rows - 1000, rows]
    hops.native().grouped_gemm(y, a, w, _i32(off).cuda(), None, 1, 0, False, True, 0.0)
    for e, i in ((0, 0), (0, rows // 2), (0, rows - 2000), (1, rows - 1000)):
        hops.native().grouped_gemm(few, a[i:i + 1000].contiguous(), w[e:e + 1].contiguous(), _i32([0, 1000]).cuda(), None, 1, 0, False, True, 0.0)
        assert torch.equal(y[i:i + 1000], few)


@pytest.mark.parametrize("rows", [1, 40, 700])
@pytest.mark.parametrize("act", [0, 1, 3, 4])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_experts_of_empty_sums(rows, act, dt):
    """Products over no k are zero, and so is what every unit makes of them."""
    a, w = torch.empty(rows, 0, dtype=dt, device="cuda"), torch.empty(2, 48, 0, dtype=dt, device="cuda")
    y = torch.full((rows, 24 if act in (1, 3) else 48), float("nan"), dtype=dt, device="cuda")
    hops.native().grouped_gemm(y, a, w, _i32([0, rows // 3, rows]).cuda(), None, 1, act, False, True, 7.0 if act == 3 else 0.0)
    assert not bool(y.any()) and not bool(y.isnan().any())


@pytest.mark.parametrize("M,f,rest,K", [(1, 16, 0, 32), (3, 48, 40, 1024), (16, 176, 16, 160), (17, 32, 8, 64), (2, 24, 8, 64)])
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "relu"])
def test_gated_unit_in_the_projection(M, f, rest, K, kind):
    """The gated unit at the end of a few rows' projection gives the bits of the projection and the unit as two launches, and so do
    the rows of the weights behind the unit's (an f that is no multiple of 16: two launches)."""
    g = _g(78)
    x, w = _r(g, M, K, dt=BF).cuda(), _r(g, 2 * f + rest, K, s=K ** -0.5, dt=BF).cuda()
    a, y, col = hops.linear_glu(x, w, f, kind)
    proj = hops.linear(x, w)
    assert torch.equal(a, hops.glu(proj, 0, f, kind)) and torch.equal(y[:, col:col + rest], proj[:, 2 * f:])


@pytest.mark.parametrize("H,dk,dv", [(4, 64, 64), (2, 32, 48), (2, 128, 32)])
@pytest.mark.parametrize("kind", ["bonus", "root"])
def test_chunked_channel_decays_in_spans(H, dk, dv, kind):
    """Decays per key channel with segments cut into spans of chunks (256 tokens here): segments around the span and the chunk,
    continued ones, a padding one, one of several spans beside single rows.  Tolerance as for whole segments: 2e-5."""
    g = _g(79)
    lens = [1, 256, 257, 700, 300, 64, 512, 1]
    cu, ctx, slot = _segments(lens, [4, 5, 0, 64, 3, 0, 9, 1], [0, 1, 2, 3, -1, 4, 5, 6])
    T = sum(lens)
    qkv, z, zb, state = _r(g, T, 2 * H * dk + H * dv, dt=BF), _r(g, T, H * dk, s=2.0, dt=BF), _r(g, H * dk, s=2.0), _r(g, 7, H, dv, dk)
    kw = dict(decay="exp_exp", bonus=_r(g, H, dk)) if kind == "bonus" else dict(tau=3.0)
    zb += -3.0 if kind == "bonus" else 3.0
    want_s, got_s = state.clone(), state.cuda()
    a = (0, H * dk, 2 * H * dk)
    want = hops.decay_scan(qkv, *a, z, zb, want_s, cu, ctx, slot, H, H, dk, dv, dk ** -0.5, **kw)
    dev = {k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in kw.items()}
    got = hops.decay_scan(qkv.cuda(), *a, z.cuda(), zb.cuda(), got_s, cu.cuda(), ctx.cuda(), slot.cuda(), H, H, dk, dv, dk ** -0.5, mode=4, **dev)
    for x, y in ((got.cpu(), want), (got_s.cpu(), want_s)):
        torch.testing.assert_close(x, y, rtol=2e-5, atol=2e-5 * float(y.abs().max()))


@pytest.mark.parametrize("n,groups", [(1, 1), (255, 1), (257, 1), (1024, 1), (1025, 1), (2048, 1), (4096, 2), (4097, 1), (3072, 3)])
@pytest.mark.parametrize("after,gate", [(False, "silu"), (True, "sigmoid"), (True, "silu")])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_gated_group_norm_sizes(n, groups, after, gate, dt):
    """Groups around what the kernel keeps in registers (4, 8 and 16 values a thread, more than that from memory).  fp32 inside: 1e-5 of
    the value, and the rounding of a bf16 result."""
    g = _g(80)
    y, z, w = _r(g, 3, n), _r(g, 3, n + 5, dt=dt), _r(g, n)
    want = hops.gated_group_norm(y, z, 5, w, 1e-5, groups, dt, after=after, gate=gate)
    got = hops.gated_group_norm(y.cuda(), z.cuda(), 5, w.cuda(), 1e-5, groups, dt, after=after, gate=gate)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2 ** -7 if dt == BF else 1e-5, atol=1e-5)


@pytest.mark.parametrize("rows,groups,gs", [(1, 2, 64), (3, 3, 64), (5, 33, 64), (1, 2, 128), (7, 5, 128), (1, 2, 256), (3, 9, 256)])
@pytest.mark.parametrize("col", [0, 8, 5])
@pytest.mark.parametrize("gate", ["silu", "sigmoid"])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_head_norm_sizes(rows, groups, gs, col, gate, dt):
    """Per-head norms of 64, 128 and 256 values, eight a lane, around whole workgroups (256 lanes), and a column where the gate's rows are not
    aligned (a wave a group).  fp32 inside: 1e-5 of the value, and the rounding of a bf16 result."""
    g = _g(81)
    n = groups * gs
    y, z, w = _r(g, rows, n), _r(g, rows, n + 8, dt=dt), _r(g, n)
    want = hops.gated_group_norm(y, z, col, w, 1e-5, groups, dt, after=True, gate=gate)
    got = hops.gated_group_norm(y.cuda(), z.cuda(), col, w.cuda(), 1e-5, groups, dt, after=True, gate=gate)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2 ** -7 if dt == BF else 1e-5, atol=1e-5)


@pytest.mark.parametrize("gs", [64, 128, 256])
@pytest.mark.parametrize("gate", ["silu", "sigmoid"])
def test_head_norm_of_large_values_and_small_gates(gs, gate):
    """Values of 1e18 with gates of e^-80: the norm, of order one, meets the gate, and nothing underflows on the way.  fp32 inside: 1e-5 of
    the value, and e^-80 to its own 80 2^-24."""
    g = _g(87)
    y, z, w = _r(g, 3, 2 * gs, s=1e18), torch.full((3, 2 * gs), -80.0), _r(g, 2 * gs)
    want = hops.gated_group_norm(y.double(), z.double(), 0, w.double(), 1e-5, 2, torch.float64, after=True, gate=gate)
    got = hops.gated_group_norm(y.cuda(), z.cuda(), 0, w.cuda(), 1e-5, 2, torch.float32, after=True, gate=gate)
    assert float(got.abs().max()) > 1e-35
    torch.testing.assert_close(got.cpu().double(), want, rtol=2e-5, atol=1e-41)


@pytest.mark.parametrize("T,d,E,K,shared", [(1000, 2048, 8, 2, False), (1003, 8, 3, 1, True), (4100, 1000, 7, 7, True), (2049, 2056, 8, 8, False),
                                            (2050, 4096, 5, 2, True)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_router_long_steps(T, d, E, K, shared, dt):
    """The router that keeps its weights in registers, around a round of four tokens and 2048 columns: the same bits as of short steps."""
    g = _g(84)
    h, wr, bias = _r(g, T, d, dt=dt).cuda(), _r(g, E + shared, d, s=0.3).cuda(), _r(g, E, s=0.3).cuda()
    h[5, d // 2] = math.nan
    h[T - 1] = 0.0  # ties, but for the bias
    got = hops.moe_router(h, wr, bias, E, K)
    parts = [hops.moe_router(h[i:i + 200], wr, bias, E, K) for i in range(0, T, 200)]
    for x, *ys in zip(got, *parts):
        if x is not None:
            y = torch.cat(ys)
            assert torch.equal(torch.nan_to_num(x, nan=-1.0) if x.is_floating_point() else x, torch.nan_to_num(y, nan=-1.0) if y.is_floating_point() else y)


@pytest.mark.parametrize("d", [4104, 1003])  # wider than the registers hold; no multiple of 8
@pytest.mark.parametrize("E,K,shared", [(8, 2, False), (7, 3, True)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_router_two_tokens_a_workgroup(d, E, K, shared, dt):
    """Long steps that the registers' router does not take, two tokens a workgroup and one left over: the bits of short steps."""
    g, T = _g(101), 4099
    h, wr, bias = _r(g, T, d, dt=dt).cuda(), _r(g, E + shared, d, s=d ** -0.5).cuda(), _r(g, E, s=0.3).cuda()
    got = hops.moe_router(h, wr, bias, E, K)
    parts = [hops.moe_router(h[i:i + 500], wr, bias, E, K) for i in range(0, T, 500)]
    for x, *ys in zip(got, *parts):
        assert x is None or torch.equal(x, torch.cat(ys))


@pytest.mark.parametrize("T", [300, 4100])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_router_of_empty_sums(T, dt):
    """Rows of no columns leave the bias's choice: logits that are its values exactly, softmax to rounding."""
    bias = _r(_g(85), 4)
    h, wr = torch.empty(T, 0, dtype=dt), torch.empty(4, 0)
    want = hops.moe_router(h, wr, bias, 4, 2)
    ids, wts, _ = hops.moe_router(h.cuda(), wr.cuda(), bias.cuda(), 4, 2)
    assert torch.equal(ids.cpu(), want[0])
    torch.testing.assert_close(wts.cpu(), want[1], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("Hq,G,dk,dv,window", [(4, 1, 64, 64, 0), (8, 1, 128, 128, 40), (8, 4, 128, 64, 0), (16, 2, 64, 128, 100), (4, 1, 128, 128, 64)])
def test_window_decode_heads(Hq, G, dk, dv, window):
    """Fewer query heads a workgroup than share a kv head: the same bits as all of them together, sinks and head gates included."""
    g = _g(82)
    lens = [1, 64, 65, 700, 17]
    kc, vc, bt = _paged(g, BF, lens, Hq, G, dk, dv, nb=80)
    q, gate, sinks = _r(g, len(lens) + 1, Hq * dk + 8, dt=BF), _r(g, len(lens) + 1, Hq + 8, dt=BF), _r(g, Hq)
    bt = torch.cat([bt, torch.zeros(1, bt.shape[1], dtype=torch.int32)])
    dev = [t.cuda() for t in (q, kc, vc, bt, _i32(lens + [0]))]
    a = (Hq, G, dk, dv, 1.0 / math.sqrt(dk), window, True)
    for kw in (dict(), dict(sinks=sinks.cuda(), gate=gate.cuda(), g_col=3, cap=9.0)):
        want = hops.window_attention_decode(*dev, *a, **kw, heads=Hq // G)
        for heads in (0, 2, 1):
            if heads == 0 or (Hq // G) % heads == 0:
                assert torch.equal(hops.window_attention_decode(*dev, *a, **kw, heads=heads), want)
    with pytest.raises(RuntimeError):
        hops.window_attention_decode(*dev, *a, heads=3)


@pytest.mark.parametrize("B", [256, 257])  # one workgroup for each compute unit, and more
@pytest.mark.parametrize("window", [0, 50])
def test_window_decode_two_workgroups_a_unit(B, window):
    """Heads of 64, four a workgroup: the form that leaves room for two gives the bits of two heads a workgroup, and the torch form's values
    within the rounding of the bf16 weights and result."""
    g = _g(95)
    lens = [int(n) for n in torch.randint(1, 300, (B,), generator=g)]
    lens[:4] = [1, 64, 65, 0]
    kc, vc = _r(g, 40, 16, 64, dt=BF), _r(g, 40, 1, 64, 16, dt=BF)
    bt = torch.randint(0, 40, (B, 19), generator=g, dtype=torch.int32)
    q = _r(g, B, 4 * 64, dt=BF)
    a = (4, 1, 64, 64, 0.125, window, True)
    dev = [t.cuda() for t in (q, kc, vc, bt, _i32(lens))]
    got = hops.window_attention_decode(*dev, *a)
    assert torch.equal(got, hops.window_attention_decode(*dev, *a, heads=2)) and torch.equal(got, hops.window_attention_decode(*dev, *a, heads=4))
    want = hops.window_attention_decode(q, kc, vc, bt, _i32(lens), *a)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1e-2, atol=2e-3)


@pytest.mark.parametrize("Hq,G,dk,dv,vec,dt", [(8, 2, 96, 128, True, BF), (8, 2, 128, 96, True, BF), (8, 2, 128, 128, False, BF), (6, 2, 64, 64, True, BF),
                                               (8, 2, 128, 128, True, torch.float32)])
def test_window_decode_heads_elsewhere(Hq, G, dk, dv, vec, dt):
    """A forced number of query heads raises where the kernels that take one do not apply; without one the call runs."""
    g = _g(83)
    lens = [1, 40]
    kc, vc, bt = _paged(g, dt, lens, Hq, G, dk, dv, nb=8)
    a = [t.cuda() for t in (_r(g, 2, Hq * dk, dt=dt), kc, vc, bt, _i32(lens))] + [Hq, G, dk, dv, 1.0 / math.sqrt(dk), 0, True]
    assert bool(hops.window_attention_decode(*a, vec=vec).isfinite().all())
    with pytest.raises(RuntimeError):
        hops.window_attention_decode(*a, vec=vec, heads=1)


@pytest.mark.parametrize("Hq,G,dk,dv", [(1, 1, 1, 1), (2, 1, 128, 64), (16, 4, 128, 128), (17, 1, 128, 8), (32, 8, 128, 16), (33, 3, 128, 8)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_qk_norm_sizes(Hq, G, dk, dv, dt):
    """Whole-projection norms around what the kernel keeps in registers (8 and 16 columns a thread, more from memory), rows without a
    slot.  fp32 inside: 1e-5 of the value, and the rounding of bf16 results."""
    g = _g(81)
    qkv, qw, kw = _r(g, 5, Hq * dk + G * (dk + dv), dt=dt), _r(g, Hq * dk), _r(g, G * dk)
    kc, vc, slots = torch.zeros(3, 16, G * dk, dtype=dt), torch.zeros(3, G, dv, 16, dtype=dt), _i32([17, -1, 3, 40, 0])
    dev = [v.cuda() for v in (qkv, qw, kw, kc, vc, slots)]
    hops.qk_norm_cache(qkv, qw, kw, 1e-5, Hq, G, dk, dv, kc, vc, slots)
    hops.qk_norm_cache(dev[0], dev[1], dev[2], 1e-5, Hq, G, dk, dv, dev[3], dev[4], dev[5])
    for a, b in zip((dev[0], dev[3], dev[4]), (qkv, kc, vc)):
        torch.testing.assert_close(a.cpu().float(), b.float(), rtol=2 ** -7 if dt == BF else 1e-5, atol=1e-5)


@pytest.mark.parametrize("dk,dv,Hq,G", [(128, 128, 4, 1), (64, 128, 3, 3), (128, 64, 2, 1), (128, 8, 2, 1)])
def test_page_ends_that_hold_no_numbers(dk, dv, Hq, G):
    """NaN behind the last token in a sequence's last page - what an earlier owner of the page may leave - reaches no result of the
    bf16 kernels: staged and register prefill, decode by row broadcasts and (the last case) by LDS broadcasts."""
    g = _g(82)
    new, ctx = [1, 40, 130, 16], [0, 9, 60, 0]
    lens = [a + b for a, b in zip(ctx, new)]
    kc, vc, bt = _paged(g, BF, lens, Hq, G, dk, dv)
    for row, n in zip(bt, lens):
        for j in range(n, (n + 15) // 16 * 16):
            vc[row[j // 16].item(), :, :, j % 16] = float("nan")
            kc[row[j // 16].item(), j % 16] = float("nan")
    cu = _i32([0] + torch.tensor(new).cumsum(0).tolist())
    qkv = _r(g, sum(new), Hq * dk + 8, dt=BF)
    for window, sink, kw in ((0, False, {}), (37, True, dict(keep=3)), (32, False, dict(chunked=True, cap=5.0))):
        a = (Hq, G, dk, dv, dk ** -0.5, window, sink)
        want = hops.window_attention_prefill(qkv, kc, vc, cu, _i32(ctx), bt, *a, **kw)
        for mfma in (256, 16, 32) if dv >= 64 else ():
            got = hops.window_attention_prefill(*(x.cuda() for x in (qkv, kc, vc, cu, _i32(ctx), bt)), *a, mfma=mfma, **kw)
            torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2e-2, atol=2e-2)
        want = hops.window_attention_decode(qkv[:4], kc, vc, bt, _i32(lens), *a, **kw)
        got = hops.window_attention_decode(*(x.cuda() for x in (qkv[:4].contiguous(), kc, vc, bt, _i32(lens))), *a, **kw)
        torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("t", [20, 35, 36, 59])
@pytest.mark.parametrize("kw", [dict(window=0, sink=False), dict(window=9, sink=True), dict(window=10, sink=False, keep=24),
                                dict(window=16, sink=False, chunked=True)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_fp32_values_that_are_no_numbers(t, kw, bad):
    """fp32 attention: a value of one head that is no number reaches the rows that see its token, in its column, and no others; all
    other results are those of the same step without it, bit for bit."""
    g = _g(83)
    kw = dict(kw)
    G, dk, dv, n, ctx = 2, 64, 64, 40, 20
    kc, vc, bt = _paged(g, torch.float32, [n + ctx], 4, G, dk, dv)
    a = (4, G, dk, dv, dk ** -0.5, kw.pop("window"), kw.pop("sink"))
    q = _r(g, n, 4 * dk).cuda()
    dev = (_i32([0, n]).cuda(), _i32([ctx]).cuda(), bt.cuda())
    v2 = vc.clone()
    v2[bt[0, t // 16].item(), 1, 5, t % 16] = bad
    p = torch.arange(ctx, ctx + n)
    lo = p - p % a[5] if kw.get("chunked") else (p - a[5] + 1 if a[5] else 0 * p)
    seen = (t <= p) & ((t >= lo) | (t < kw.get("keep", 0)))
    hit = torch.zeros(n, 4, dv, dtype=torch.bool)
    hit[seen, 2:, 5] = True
    want = hops.window_attention_prefill(q, kc.cuda(), vc.cuda(), *dev, *a, **kw).cpu().view(n, 4, dv)
    got = hops.window_attention_prefill(q, kc.cuda(), v2.cuda(), *dev, *a, **kw).cpu().view(n, 4, dv)
    assert torch.equal(got[~hit], want[~hit]) and not bool(torch.isfinite(got[hit]).any())
    for i in (0, 15, 16, 39):  # each row as a decode step
        sl = _i32([ctx + i + 1]).cuda()
        want = hops.window_attention_decode(q[i:i + 1], kc.cuda(), vc.cuda(), dev[2], sl, *a, **kw).cpu().view(4, dv)
        got = hops.window_attention_decode(q[i:i + 1], kc.cuda(), v2.cuda(), dev[2], sl, *a, **kw).cpu().view(4, dv)
        assert torch.equal(got[~hit[i]], want[~hit[i]]) and not bool(torch.isfinite(got[hit[i]]).any())


@pytest.mark.parametrize("where", ["v", "k", "q", "z", "beta"])
@pytest.mark.parametrize("t", [0, 63, 70, 149, 402])
@pytest.mark.parametrize("kind", ["linear", "delta", "delta_plain", "bonus", "root", "root_spans"])
def test_chunks_keep_later_tokens_out_of_earlier_ones(kind, where, t):
    """A NaN or an infinity in a token's value, key, query, decay or beta leaves the outputs in front of it as they are, and the same
    outputs and states are no numbers as token by token (the scan): at the first and last token of a segment and of a chunk, and
    inside one.  Tolerances as for the chunks above."""
    if where == "z" and kind == "linear" or where == "beta" and not kind.startswith("delta"):
        pytest.skip("not an input of this form")
    g = _g(84)
    H, d = 2, 32
    cu, ctx, slot = _segments([150, 300, 40], [0, 7, 3], [1, 0, 2])
    T = 490
    qkv, beta, state = _r(g, T, 3 * H * d, s=0.5, dt=BF), _r(g, T, H, dt=BF), _r(g, 3, H, d, d)
    per_head = kind.startswith("delta")
    z, zb = _r(g, T, H if per_head else H * d, dt=BF), _r(g, H if per_head else H * d) + (3.0 if kind.startswith("root") else -3.0)
    cols = {"q": 0, "k": H * d, "v": 2 * H * d}
    if kind == "linear":  # rows are [v | k | q] there
        cols = {"v": 0, "k": H * d, "q": 2 * H * d}
    for bad in (float("nan"),) if where in ("z", "beta") else (float("nan"), float("inf")):
        a = [qkv.clone(), z.clone(), beta.clone()]
        if where in cols:
            a[0][t, cols[where] + d + 3] = bad
        else:
            a[1 if where == "z" else 2][t, -1] = bad
        dev = [x.cuda() for x in a]

        def run(chunks):
            s = state.cuda()
            seg = (s, cu.cuda(), ctx.cuda(), slot.cuda())
            if kind == "linear":
                o = hops.linear_attention(dev[0], torch.tensor([0.9, 0.99]).cuda(), *seg, H, d, d, mode=3 if chunks else 2)
            else:
                kw = dict(a_log=_r(_g(85), H).cuda(), beta=dev[2], unit=kind == "delta") if per_head else \
                    dict(decay="exp_exp", bonus=_r(_g(85), H, d).cuda()) if kind == "bonus" else dict(tau=3.0)
                o = hops.decay_scan(dev[0], 0, H * d, 2 * H * d, dev[1], zb.cuda(), *seg, H, H, d, d, 0.2,
                                    mode=(4 if kind == "root_spans" else 3) if chunks else 2, **kw)
            return o.cpu(), s.cpu()

        for x, y in zip(run(True), run(False)):
            fin = torch.isfinite(y)
            assert torch.equal(torch.isfinite(x), fin)
            if x.shape[0] == T:
                assert bool(fin[:t].all()) and (kind == "bonus" and where == "z" or not bool(fin[t].all()))  # (a bonus token reads the state before its own decay)
            torch.testing.assert_close(x[fin], y[fin], rtol=5e-5, atol=5e-5 * float(y[fin].abs().max()))


@pytest.mark.parametrize("kind", ["linear", "delta", "bonus", "root"])
@pytest.mark.parametrize("prompts", [[300], [290, 1, 70], [256, 513]])
def test_single_tokens_beside_prompts_keep_their_bits(kind, prompts):
    """Running sequences' next tokens in front of prompts that go in chunks: outputs and states have the bits of the same tokens in a
    step of their own, and the prompts' those of a step without them."""
    g = _g(86)
    H, d, nd = 2, 32, 40
    lens = [1] * nd + prompts
    S, T = len(lens), nd + sum(prompts)
    cu, ctx, slot = (v.cuda() for v in _segments(lens, [9] * nd + [0, 3, 0][:len(prompts)], list(range(S))))
    qkv, state = _r(g, T, 3 * H * d, s=0.5, dt=BF).cuda(), _r(g, S, H, d, d).cuda()
    per_head = kind == "delta"
    z, zb = _r(g, T, H if per_head else H * d, dt=BF).cuda(), (_r(g, H if per_head else H * d) - 1.0).cuda()
    beta, al, bonus, lam = _r(g, T, H, dt=BF).cuda(), _r(g, H).cuda(), _r(g, H, d).cuda(), torch.tensor([0.9, 0.99]).cuda()
    longest = max(prompts)
    assert T < 32 * S  # (longer segments: test_single_tokens_beside_long_prompts)

    def run(a, b, s0, s1, **kw):  # rows [a, b), segments [s0, s1)
        s = state.clone()
        seg = (s, cu[s0:s1 + 1] - cu[s0], ctx[s0:s1], slot[s0:s1])
        if kind == "linear":
            return hops.linear_attention(qkv[a:b], lam, *seg, H, d, d, **kw), s
        form = dict(a_log=al, beta=beta[a:b], unit=True) if per_head else dict(decay="exp_exp", bonus=bonus) if kind == "bonus" else dict(tau=3.0)
        return hops.decay_scan(qkv[a:b], 0, H * d, 2 * H * d, z[a:b], zb, *seg, H, H, d, d, 0.2, **form, **kw), s

    o, s = run(0, T, 0, S, longest=longest, singles=nd)
    od, sd = run(0, nd, 0, nd, longest=1)
    assert torch.equal(o[:nd], od) and torch.equal(s[:nd], sd[:nd])
    op, sp = run(nd, T, nd, S, longest=longest)
    assert torch.equal(o[nd:], op) and torch.equal(s[nd:], sp[nd:])


@pytest.mark.parametrize("prompts", [[1500, 700], [1100, 1, 64]])
def test_single_tokens_beside_long_prompts(prompts):
    """Linear attention with a mean of 32 rows a segment and more: running sequences' tokens in front have the bits of a step of their own, and
    the prompts' those of a step without them."""
    g, nd, H, d = _g(102), 20, 2, 32
    lens = [1] * nd + prompts
    S, T = len(lens), nd + sum(prompts)
    assert T >= 32 * S
    cu, ctx, slot = (v.cuda() for v in _segments(lens, [9] * nd + [0, 3, 0][:len(prompts)], list(range(S))))
    vkq, state, lam = _r(g, T, 3 * H * d, s=0.5, dt=BF).cuda(), _r(g, S, H, d, d).cuda(), torch.tensor([0.9, 0.99]).cuda()

    def run(a, b, s0, s1, **kw):
        s = state.clone()
        return hops.linear_attention(vkq[a:b], lam, s, cu[s0:s1 + 1] - cu[s0], ctx[s0:s1], slot[s0:s1], H, d, d, **kw), s

    (o, s), (od, sd) = run(0, T, 0, S, longest=max(prompts), singles=nd), run(0, nd, 0, nd, longest=1)
    op, sp = run(nd, T, nd, S, longest=max(prompts))
    assert torch.equal(o[:nd], od) and torch.equal(s[:nd], sd[:nd])
    assert torch.equal(o[nd:], op) and torch.equal(s[nd:], sp[nd:])


@pytest.mark.parametrize("Hq,G", [(8, 2), (8, 1), (4, 4)])  # four heads that share their keys, twice; none
@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 128), (128, 64)])
@pytest.mark.parametrize("window,kw", [(0, {}), (40, dict(keep=5)), (64, dict(chunked=True)), (33, dict(cap=20.0)), (0, dict(cap=80.0, sink=True))])
def test_window_prefill_heads_that_share_their_keys(Hq, G, dk, dv, window, kw):
    """Query rows 32 at a time, with the keys through LDS where four heads share them, have the bits of 16 at a time with keys of
    their own: segments of one row and of whole and broken tiles, an odd and an even number of key tiles, ends inside a page."""
    g = _g(91)
    kw = dict(kw)
    sink = kw.pop("sink", False)
    lens, ctx = [1, 16, 32, 33, 47, 100], [0, 5, 16, 96, 31, 0]
    T, S = sum(lens), len(lens)
    W = max((a + b + 15) // 16 for a, b in zip(lens, ctx))
    bt = torch.randperm(S * W, generator=g).int().view(S, W).cuda()
    qkv = _r(g, T, Hq * dk + G * (dk + dv), dt=BF).cuda()
    kc, vc = _r(g, S * W, 16, G * dk, dt=BF).cuda(), _r(g, S * W, G, dv, 16, dt=BF).cuda()
    cu = _i32([0] + torch.tensor(lens).cumsum(0).tolist()).cuda()
    run = lambda rows: hops.window_attention_prefill(qkv, kc, vc, cu, _i32(ctx).cuda(), bt, Hq, G, dk, dv, dk ** -0.5, window, sink, mfma=rows, **kw)
    assert torch.equal(run(32), run(16))


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (300, 2, 3), (517, 3, 5)])
@pytest.mark.parametrize("d,swiglu", [(64, False), (192, True), (320, False)])
def test_grouped_tiles_sort_their_rows_as_they_read(T, K, E, d, swiglu):
    """The grouped tile GEMM over rows in their own order has the bits of the sorted copy's: an expert without rows, tiles that end
    inside an expert, every k-tile count of the ring's head."""
    from k8s_llm_monitor_amd import ops

    g = _g(92)
    ids = torch.randint(0, max(E - 1, 1), (T, K), generator=g, dtype=torch.int32).cuda()
    off, idx, _ = ops.moe_align(ids, E)
    x, w = _r(g, T, d, dt=BF).cuda(), _r(g, E, 256, d, s=0.1, dt=BF).cuda()
    want = ops.moe_grouped_gemm(ops.gather_rows(x, idx, K), w, off, swiglu=swiglu)
    assert torch.equal(ops.moe_grouped_gemm(x, w, off, swiglu=swiglu, rows=idx, div=K), want)
    cpu = ops.moe_grouped_gemm(x.cpu(), w.cpu(), off.cpu(), swiglu=swiglu, rows=idx.cpu(), div=K)
    torch.testing.assert_close(want.cpu().float(), cpu.float(), rtol=2e-2, atol=2e-2 * float(cpu.float().abs().max()))


@pytest.mark.parametrize("at", [1, 4, 8])
def test_grouped_tiles_of_rows_at_any_address(at):
    """Rows in their own order that do not start on 16 bytes (the first two) are sorted by a copy: the bits of an aligned clone.  The tile
    kernel itself refuses them."""
    from k8s_llm_monitor_amd import ops

    g = _g(94)
    T, K, E, d = 300, 2, 3, 192
    off, idx, _ = ops.moe_align(torch.randint(0, E, (T, K), generator=g, dtype=torch.int32).cuda(), E)
    x, w = _r(g, T * d + at, dt=BF).cuda()[at:].view(T, d), _r(g, E, 256, d, s=0.1, dt=BF).cuda()
    want = ops.moe_grouped_gemm(x.clone(), w, off, rows=idx, div=K)
    assert torch.equal(ops.moe_grouped_gemm(x, w, off, rows=idx, div=K), want)
    if at != 8:
        with pytest.raises(RuntimeError, match="alignment"):
            ops.native().gemm_tile_rows(want, x, w, off, idx, K, False, 0)


@pytest.mark.parametrize("T,Hq,G,dk,dv,nf,extra,pairs,dt", [
    (255, 4, 2, 64, 64, 32, 8, False, BF),        # the last size whose values go row by row
    (256, 4, 2, 64, 72, 24, 8, True, BF),         # entries that pass; values not a multiple of a group's columns
    (1023, 3, 1, 128, 640, 64, 0, False, BF),     # two groups of value columns
    (1025, 3, 1, 128, 40, 64, 16, True, BF),      # several rows a workgroup, the last with one
    (1030, 2, 2, 48, 32, 8, 0, False, BF),
    (300, 2, 1, 36, 34, 18, 2, False, BF),        # neither eight neighbours nor 16-byte rows
    (270, 2, 1, 36, 33, 18, 0, True, BF),         # odd rows: values row by row
    (1040, 2, 1, 2048, 16, 1024, 0, False, BF),   # more frequencies than a workgroup holds
    (1025, 2, 2, 64, 64, 32, 0, True, torch.float32),
])
def test_values_to_pages_in_runs(T, Hq, G, dk, dv, nf, extra, pairs, dt):
    """rotary_cache and qk_norm_cache of large steps: decode rows, then sequences that begin and end inside pages, rows that are not
    written, pages in any order.  Values are copies: equal to the bit; turned and normed entries as the fp32 form up to one rounding."""
    g = _g(90)
    nv, bs = G * dv, 16
    lens = [1, 1, 1, 37, 5, T - 45]
    starts = [15, 0, 7, 11, 16, 3]
    nb = sum((a + n + 15) // 16 for a, n in zip(starts, lens)) + 2
    pages, slots, at = torch.randperm(nb, generator=g), [], 0
    for a, n in zip(starts, lens):
        p = torch.arange(a, a + n)
        slots.append(pages[at + p // 16] * 16 + p % 16)
        at += (a + n + 15) // 16
    slots = torch.cat(slots).to(torch.int32)
    slots[[20, 60, T - 1]] = -1
    pos = torch.randint(0, 4000, (T,), generator=g, dtype=torch.int32)
    freq = hops.rotary_freq(1e4, nf)
    temp = torch.rand(Hq, generator=g) + 0.5
    x = _r(g, T, (Hq + G) * dk + nv + extra, dt=dt)
    tol = dict(rtol=2 ** -7, atol=2 ** -7) if dt == BF else dict(rtol=1e-5, atol=1e-5)  # one rounding; some units of fp32

    def run(device, norm):
        y = (x[:, :(Hq + G) * dk + nv] if norm else x).to(device, copy=True).contiguous()
        kc = torch.zeros(nb, bs, G * dk, dtype=dt, device=device)
        vc = torch.zeros(nb, G, dv, bs, dtype=dt, device=device)
        s = slots.to(device)
        if norm:
            w = torch.linspace(0.5, 1.5, Hq * dk, device=device)
            hops.qk_norm_cache(y, w, w[:G * dk].contiguous(), 1e-5, Hq, G, dk, dv, kc, vc, s)
        else:
            hops.rotary_cache(y, Hq, G, dk, dv, pos.to(device), freq.to(device), pairs, temp.to(device), kc, vc, s)
        return y.cpu(), kc.cpu(), vc.cpu()

    for norm in (False, True):
        want, got = run("cpu", norm), run("cuda", norm)
        assert torch.equal(got[2], want[2])
        assert torch.equal(got[0][:, (Hq + G) * dk:], want[0][:, (Hq + G) * dk:])
        torch.testing.assert_close(got[0].float(), want[0].float(), **tol)
        torch.testing.assert_close(got[1].float(), want[1].float(), **tol)


@pytest.mark.parametrize("T,d,E,K,at,shared,dt", [
    (1, 8, 3, 1, 0, False, BF), (3, 264, 8, 2, 1, True, BF), (64, 2048, 8, 2, 1, False, BF), (255, 2056, 7, 5, 2, True, BF),
    (256, 4104, 8, 8, 1, True, BF), (300, 1024, 5, 3, 1, False, BF), (37, 1000, 8, 2, 1, True, torch.float32), (64, 4096, 9, 2, 0, False, torch.float32),
    (5, 24, 12, 2, 1, True, BF),  # more weight rows than the norm's launch takes
])
def test_experts_sum_and_router_with_the_norm(T, d, E, K, at, shared, dt):
    """add_norm that forms the experts' sum and routes its rows, against the launches it replaces: the same bits; and against the fp32 form
    (a bf16 row's rounding)."""
    g = _g(91)
    x = _r(g, T, d)
    ys, wts = _r(g, T * K, d, dt=dt), torch.rand(T, K, generator=g)
    sh, gate = (_r(g, T, d, dt=dt), torch.rand(T, generator=g)) if shared else (None, None)
    inv = torch.randperm(T * K, generator=g).to(torch.int32)
    adds = [_r(g, T, d, dt=dt), _r(g, T, d)]
    w, vec = torch.rand(d, generator=g), _r(g, d)
    wr, bias = _r(g, E + int(shared), d, s=d ** -0.5), _r(g, E)
    dev = lambda t: t.cuda() if t is not None else None
    ex = hops.ExpertSum(*map(dev, (ys, inv, wts, sh, gate)))
    route = (wr.cuda(), bias.cuda(), E, K)
    cadds = [a.cuda() for a in adds]
    x1, x2, x3 = (x.cuda() for _ in range(3))
    h1 = hops.add_norm(x1, tuple(cadds[:at] + [ex.rows()] + cadds[at:]), vec.cuda(), w.cuda(), 1e-5, True, dt)
    r1 = hops.moe_router(h1, *route)
    fused = tuple(cadds[:at] + [ex] + cadds[at:])
    h2, r2 = hops.add_norm(x2, fused, vec.cuda(), w.cuda(), 1e-5, True, dt, route=route)
    h3 = hops.add_norm(x3, fused, vec.cuda(), w.cuda(), 1e-5, True, dt)
    for a, b in ((x1, x2), (x1, x3), (h1, h2), (h1, h3), *((a, b) for a, b in zip(r1, r2) if a is not None)):
        assert torch.equal(a, b)
    s = (wts.unsqueeze(-1) * ys.float()[inv.long()].view(T, K, d)).sum(1)
    if shared:
        s += gate.unsqueeze(-1) * sh.float()
    want = hops.add_norm(x, tuple(adds[:at] + [s] + adds[at:]), vec, w, 1e-5, True, dt)
    tol = 2 ** -7 if dt == BF else 1e-5
    torch.testing.assert_close(h2.cpu().float(), want.float(), rtol=tol, atol=tol)


@pytest.mark.parametrize("T,H,dn,dr,dv,R,pitch,nf,pairs,sliced", [
    (1, 8, 96, 32, 128, 256, 288, 16, False, False), (16, 3, 8, 8, 16, 8, 16, 4, True, False), (17, 5, 40, 8, 24, 72, 96, 2, False, False),
    (33, 2, 128, 64, 40, 136, 224, 32, True, False), (70, 4, 64, 32, 65, 128, 160, 0, False, False), (2048, 1, 32, 8, 16, 128, 160, 4, True, False),
    (2049, 1, 32, 8, 16, 128, 160, 4, False, False), (256, 2, 24, 8, 7, 264, 288, 4, False, False), (257, 2, 24, 8, 7, 264, 288, 4, False, False),
    (9, 2, 20, 6, 12, 36, 42, 3, True, False),  # not in 16-byte pieces
    (5, 2, 32, 32, 32, 64, 96, 16, False, True),  # rows inside wider ones (two heads of 64)
])
def test_latent_heads(T, H, dn, dr, dv, R, pitch, nf, pairs, sliced):
    """Per-head products around latent attention at and around tiles of 16 rows and 128 columns and the sizes that leave them.  fp32 sums of
    bf16 products, one rounding: 2^-8 of the value; the turned part the same; copies and zeros equal."""
    g = _g(92)
    q = _r(g, T, H * (dn + dr) * (2 if sliced else 1), dt=BF)
    wk, wv, o = _r(g, H * dn, R, s=R ** -0.5, dt=BF), _r(g, H * dv, R, s=R ** -0.5, dt=BF), _r(g, T, H * R, dt=BF)
    pos, freq = torch.randint(0, 4000, (T,), generator=g, dtype=torch.int32), hops.rotary_freq(1e4, nf)
    cut = lambda t: t[:, :H * (dn + dr)]
    lat = torch.bmm(cut(q).reshape(T, H, dn + dr)[:, :, :dn].transpose(0, 1).float().contiguous(), wk.view(H, dn, R).float()).to(BF)
    want = hops.latent_queries(cut(q).contiguous(), lat, H, dn, dr, pos, freq, pitch, pairs).view(T, H, pitch)
    gq = cut(q.cuda())
    got = hops.latent_head_queries(gq, wk.cuda(), H, dn, dr, pos.cuda(), freq.cuda(), pitch, pairs).cpu().view(T, H, pitch)
    torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -7)
    assert torch.equal(got[..., R + 2 * nf:], want[..., R + 2 * nf:])
    v = torch.bmm(o.view(T, H, R).transpose(0, 1).float().contiguous(), wv.view(H, dv, R).transpose(1, 2).float().contiguous())
    got = hops.latent_head_values(o.cuda(), wv.cuda(), H).cpu().view(T, H, dv)
    torch.testing.assert_close(got.float(), v.transpose(0, 1), rtol=2 ** -7, atol=2 ** -7)


@pytest.mark.parametrize("mfma,vec,dk,dv,Hq,G,off,dt", [
    (256, True, 128, 128, 8, 2, 8, BF), (256, True, 64, 128, 3, 3, 0, BF), (2, True, 128, 64, 4, 1, 16, BF), (2, True, 64, 64, 2, 2, 8, BF),
    (1, True, 128, 128, 4, 1, 4, BF),  # logits not in 16-byte pieces: gated in a pass of its own, as the kernels below do
    (0, False, 128, 128, 4, 2, 8, BF), (1, True, 48, 40, 4, 2, 8, BF), (1, True, 64, 64, 4, 2, 0, torch.float32),
])
def test_gate_by_value(mfma, vec, dk, dv, Hq, G, off, dt):
    """The output gate in the attention kernels, rows written into a given buffer: the bits of the ungated rows and sigmoid_gate, for chunks
    around a tile's end and decode rows beside a padding row."""
    g = _g(93)
    new, ctx = [65, 1, 130], [0, 40, 17]
    lens = [c + n for c, n in zip(ctx, new)]
    kc, vc, bt = _paged(g, dt, lens, Hq, G, dk, dv, nb=sum((n + 15) // 16 for n in lens) + 3)
    T = sum(new)
    qkv, z = _r(g, T, Hq * dk + 8, dt=dt).cuda(), _r(g, T, Hq * dv + 24, s=2.0, dt=dt).cuda()
    dev = [x.cuda() for x in (kc, vc, _i32([0, 65, 66, 196]), _i32(ctx), bt)]
    a = (Hq, G, dk, dv, dk ** -0.5, 50, True)
    want = hops.sigmoid_gate(hops.window_attention_prefill(qkv, *dev, *a, mfma=mfma), z, off)
    rows = torch.full((T + 2, Hq * dv), 7.0, dtype=dt, device="cuda")
    got = hops.window_attention_prefill(qkv, *dev, *a, mfma=mfma, gate=z, g_col=off, by_value=True, out=rows[1:-1])
    assert torch.equal(got, want) and torch.equal(rows[1:-1], want) and bool((rows[[0, -1]] == 7).all())
    n = _i32(lens[:2] + [0]).cuda()
    want = hops.sigmoid_gate(hops.window_attention_decode(qkv[:3], dev[0], dev[1], bt.cuda(), n, *a, vec=vec), z[:3], off)
    got = hops.window_attention_decode(qkv[:3], dev[0], dev[1], bt.cuda(), n, *a, vec=vec, gate=z, g_col=off, by_value=True, out=rows[1:4])
    assert torch.equal(got, want) and bool((rows[0] == 7).all())
    cpu = hops.window_attention_decode(*(x.cpu() for x in (qkv[:3], dev[0], dev[1], bt, n)), *a, gate=z.cpu(), g_col=off, by_value=True)
    torch.testing.assert_close(got.cpu().float(), cpu.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("T,d,E,pos,prev,shift,dt", [
    (1, 8, 0, True, True, False, BF), (64, 2048, 8, True, False, True, BF), (255, 2056, 7, False, True, True, BF), (256, 264, 8, True, False, False, BF),
    (300, 4104, 0, False, False, False, BF), (37, 1000, 8, True, True, True, torch.float32),
    (5, 20, 4, True, False, True, BF),  # rows not in 16-byte pieces
])
def test_embedding_with_the_norm(T, d, E, pos, prev, shift, dt):
    """embed_norm against embed_pos, add_norm and moe_router: the same bits, tokens and positions outside the tables included."""
    g = _g(94)
    emb, pt = _r(g, 50, d, dt=dt).cuda(), _r(g, 40, d, dt=dt).cuda() if pos else None
    ids, p = (torch.randint(-2, 55, (T,), generator=g, dtype=torch.int32).cuda() for _ in range(2))
    src = (torch.arange(T, dtype=torch.int32) % 5 - 1).cuda() if prev else None
    pv = torch.randint(0, 50, (4,), generator=g, dtype=torch.int32).cuda() if prev else None
    vec, w = _r(g, d).cuda() if shift else None, torch.rand(d, generator=g).cuda()
    route = (_r(g, E + 1, d, s=d ** -0.5).cuda(), _r(g, E).cuda(), E, 2) if E else None
    x = hops.embed_pos(ids, p, emb, pt, src, pv, scale=1.7)
    h = hops.add_norm(x, (), vec, w, 1e-5, True, dt)
    gx, gh = hops.embed_norm(ids, p, emb, pt, src, pv, 1.7, vec, w, 1e-5, True, route)
    if E:
        gh, r = gh
        assert all(torch.equal(a, b) for a, b in zip(r, hops.moe_router(h, *route)))
    assert torch.equal(gx, x) and torch.equal(gh, h)


@pytest.mark.parametrize("T", [1, 3, 300])
def test_add_norm_of_width_0(T):
    """Nothing is read or written."""
    x, w = torch.empty(T, 0, device="cuda"), torch.empty(0, device="cuda")
    for dt in (BF, torch.float32):
        assert hops.add_norm(x, (), w, w, 1e-5, True, dt).shape == (T, 0)
        x2, h = hops.embed_norm(_i32([0] * T).cuda(), _i32([0] * T).cuda(), torch.empty(4, 0, dtype=dt, device="cuda"), None, None, None, 1.0, None,
                                w, 1e-5, True)
        assert x2.shape == h.shape == (T, 0)


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("fixed", [False, True])
def test_one_token_a_segment_without_states(fixed, dt):
    """A recurrence of no states is its skip term (with a fixed decay: zero)."""
    g = _g(97)
    n, nh, P = 5, 2, 64
    x, z = _r(g, n, nh * P, dt=dt), _r(g, n, nh, dt=dt)
    dtb, al, dk = (_r(g, nh) for _ in range(3))
    seg = (_i32(list(range(n + 1))), _i32([3] * n), _i32([0, 1, -1, 2, 3]))
    a = (x, None if fixed else z, 0, *((None,) * 3 if fixed else (dtb, al, dk)), torch.zeros(4, nh, 0, P), *seg)
    d = torch.rand(nh, generator=g).cuda() if fixed else None
    got = hops.ssm_scan(*(t.cuda() if isinstance(t, torch.Tensor) else t for t in a), nh, P, 0, 1, decay=d)
    want = x.float().view(n, nh, P) * (0.0 if fixed else dk[:, None])
    want[2] = 0.0  # a padding row
    torch.testing.assert_close(got.cpu(), want.view(n, nh * P), rtol=1e-6, atol=0)  # one product


@pytest.mark.parametrize("T,H,singles", [
    (3, 2, True), (256, 4, True), (1025, 2, True),   # up to 512 turning pairs a row
    (511, 13, False), (512, 13, False), (300, 14, False),  # those without and with runs of values; more pairs
    (300, 14, True), (1030, 20, True),
])
def test_values_of_rows_by_themselves(T, H, singles):
    """Rows whose slots do not follow one another, as a large decode step's, with a few pairs that happen to, inside a page and over two: the values
    of every row, once.  Copies: equal to the bit."""
    g, G, dk = _g(91), 3, 64
    nb = (T + 15) // 16 + 8
    slots = torch.randperm(nb * 16, generator=g)[:T].to(torch.int32)
    left = torch.ones(nb * 16, dtype=torch.bool)
    left[slots.long()] = False
    for a in (0, 15, 16, T - 3) if T > 16 else ():  # pairs in the first and last rows, over a workgroup's last row
        p = int((left[:-1] & left[1:]).nonzero()[a % 3])
        slots[a], slots[a + 1] = p, p + 1
        left[p:p + 2] = False
    x = _r(g, T, (H + 2 * G) * dk, dt=BF)
    freq, pos, w = hops.rotary_freq(1e4, 64), torch.arange(T, dtype=torch.int32), torch.ones(H * dk)
    for norm in (False, True):
        out = []
        for dev in ("cpu", "cuda"):
            y, kc, vc = x.to(dev, copy=True), torch.zeros(nb, 16, G * dk, dtype=BF, device=dev), torch.zeros(nb, G, dk, 16, dtype=BF, device=dev)
            if norm:
                hops.qk_norm_cache(y, w.to(dev), torch.ones(G * dk, device=dev), 1e-5, H, G, dk, dk, kc, vc, slots.to(dev), singles=singles)
            else:
                hops.rotary_cache(y, H, G, dk, dk, pos.to(dev), freq.to(dev), False, None, kc, vc, slots.to(dev), singles=singles)
            out.append((y.cpu(), kc.cpu(), vc.cpu()))
        assert torch.equal(out[0][2], out[1][2])
        for a, b in zip(out[0][:2], out[1][:2]):  # turned and normed entries up to one rounding
            torch.testing.assert_close(a.float(), b.float(), rtol=2 ** -7, atol=2 ** -7)
