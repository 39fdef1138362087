"""Operators of the layer-list (hybrid) decoders: fp32 residual stream with one-plus RMSNorm,
windowed attention with a softmax sink over a paged cache, the Mamba-2 recurrence with its short
convolution and per-sequence state slots, and routed experts with a biased fp32 router and a
gated shared expert; and, for the sequential-block designs, the token-shifted norm, the depth
average of layer results, latent (low-rank compressed) attention with rotary positions and learned
per-head sinks, and ungated experts with a softmax-over-all router; and the gated residual
(a sublayer's result times the sigmoid of a projection of its input, scaled, then the norm),
rotary grouped-query attention with per-head temperatures, the fixed-decay linear-attention
recurrence, gated linear units and the logit soft cap; and layer norms before and after a sublayer,
token-shift mixes, attention within position chunks with capped scores, the selective scan (a decay per
channel and state), linear attention with a current-token bonus and the delta rule with a decay per head;
and several residual streams with learned read / mix / write weights, windows that keep the first tokens
visible, per-head output gates, and routers with a choice correction and identity experts.

GPU tensors run the gfx950 kernels of ``_k8sllm_hybrid`` (``ops/csrc/hybrid``; built by
``python -m k8s_llm_monitor_amd.ops.build --only hybrid``) for bfloat16 and float32 activations
alike; CPU tensors run the torch forms below (the same arithmetic in fp32).  A GPU tensor never
falls back: without the extension the call raises.

Conventions.  ``T`` rows are the step's tokens, all sequences concatenated; a *segment* is one
sequence's rows of this step (a decode token is a segment of one row).  ``seg_cu`` [R+1] are the
segments' row offsets, ``seg_ctx`` [R] the tokens each sequence already holds in its cache /
state (0 = the sequence starts here, its state is taken as zero), ``seg_slot`` [R] its state slot
(< 0: a padding row, skipped).  Paged caches: keys ``[blocks, block_size, heads * dim]`` (a token's
keys contiguous), values ``[blocks, heads, vdim, block_size]`` (a value dim's tokens contiguous - the
direction the PV products read along).
"""
from __future__ import annotations

import importlib
import math
from typing import NamedTuple, Optional

import torch
import torch.nn.functional as F

_EXT = None
_EXT_ERR: Optional[BaseException] = None


def native():
    """The compiled ``_k8sllm_hybrid`` module (raises with the build hint if unavailable)."""
    global _EXT, _EXT_ERR
    if _EXT is None and _EXT_ERR is None:
        try:
            _EXT = importlib.import_module("k8s_llm_monitor_amd.ops._k8sllm_hybrid")
        except BaseException as e:  # noqa: BLE001 - remembered, re-raised on GPU use
            _EXT_ERR = e
    if _EXT is None:
        raise RuntimeError("gfx950 kernels (_k8sllm_hybrid) are not built/loadable; run "
                           "`python -m k8s_llm_monitor_amd.ops.build --only hybrid` (cause: %r)" % (_EXT_ERR,))
    return _EXT


def native_available() -> bool:
    try:
        native()
        return True
    except RuntimeError:
        return False


def _silu(z: torch.Tensor) -> torch.Tensor:
    return z * torch.sigmoid(z)


# ---------------------------------------------------------------- residual stream / norms

def embed_pos(ids: torch.Tensor, positions: torch.Tensor, embed: torch.Tensor, pos: Optional[torch.Tensor],
              src: Optional[torch.Tensor] = None, prev: Optional[torch.Tensor] = None,
              out: Optional[torch.Tensor] = None, scale: float = 1.0) -> torch.Tensor:
    """fp32 rows ``embed[id] * scale + pos[position]`` (``pos`` None: no learned positions).  ``src`` /
    ``prev`` (pipelined decode): row i takes token ``prev[src[i]]`` where ``src[i] >= 0``.
    ``out``: a contiguous fp32 [T, d] buffer to fill."""
    if not embed.is_cuda:
        if src is not None:
            ids = torch.where(src >= 0, prev.index_select(0, src.clamp(min=0).long()), ids)
        x = embed[ids.long()].float()
        if scale != 1.0:
            x = x * scale
        x = x + pos[positions.long()].float() if pos is not None else x
        if out is not None:
            out.copy_(x)
            return out
        return x
    if out is None:
        out = torch.empty(ids.numel(), embed.shape[1], dtype=torch.float32, device=embed.device)
    native().embed_pos(out, ids, positions, embed, pos, src, prev, float(scale))
    return out


class ExpertSum(NamedTuple):
    """What moe_experts(join=True) returns on the GPU: the chosen experts' rows, not yet summed.  add_norm takes it as an addend;
    ``rows()`` is the sum itself (fp32 [T, d])."""
    ys: torch.Tensor
    inv: torch.Tensor
    wts: torch.Tensor
    shared: Optional[torch.Tensor]
    gate: Optional[torch.Tensor]

    def rows(self) -> torch.Tensor:
        out = torch.empty(self.wts.shape[0], self.ys.shape[1], dtype=torch.float32, device=self.ys.device)
        native().moe_combine(out, self.ys, self.inv, self.wts, self.shared, self.gate, None, None, 0)
        return out


def add_norm(residual: torch.Tensor, addends: tuple, vec: Optional[torch.Tensor], w: torch.Tensor, eps: float,
             one_plus: bool, out_dtype: torch.dtype, route: Optional[tuple] = None):
    """``residual`` (fp32 [T, d], updated in place) += sum of ``addends`` ([T, d] each, any float
    dtype, at most three) + ``vec`` ([d], broadcast over the rows); returns the RMSNorm of the new
    residual times ``w`` (``one_plus``: times ``1 + w``) in ``out_dtype``.  The sum and the norm
    are fp32.  An addend may be an ExpertSum of rows of ``out_dtype`` (``d`` a multiple of 8).  ``route`` (wr, bias, E, K): returns
    (rows, moe_router's results for them), in one launch for the steps that ``route_with_norm`` names."""
    if route is not None and not (residual.is_cuda and route_with_norm(*residual.shape, route[0].shape[0])):
        h = add_norm(residual, addends, vec, w, eps, one_plus, out_dtype)
        return h, moe_router(h, *route)
    if not residual.is_cuda:
        for a in addends:
            residual += a.float()
        if vec is not None:
            residual += vec.float()
        y = residual * torch.rsqrt(residual.pow(2).mean(-1, keepdim=True) + eps)
        wf = w.float()
        return (y * (1.0 + wf if one_plus else wf)).to(out_dtype)
    assert len(addends) <= 3
    out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
    a = list(addends) + [None] * (3 - len(addends))
    at = next((i for i, x in enumerate(a) if isinstance(x, ExpertSum)), -1)
    if at < 0 and route is None:
        native().add_norm(out, residual, a[0], a[1], a[2], vec, w, float(eps), bool(one_plus))
        return out
    ex: tuple = (None,) * 5
    if at >= 0:
        ex, a[at] = a[at], None
    wr, bias, E, K = route or (None, None, 0, 0)
    routed = _route_out(residual, route)
    native().add_norm_experts(out, residual, a[0], a[1], a[2], vec, w, float(eps), bool(one_plus), at, *ex, *routed, wr, bias, E, K, False)
    return out if route is None else (out, routed)


def _route_out(residual: torch.Tensor, route: Optional[tuple]) -> tuple:
    if route is None:
        return None, None, None
    (wr, _, E, K), T, dev = route, residual.shape[0], residual.device
    return (torch.empty(T, K, dtype=torch.int32, device=dev), torch.empty(T, K, dtype=torch.float32, device=dev),
            torch.empty(T, dtype=torch.float32, device=dev) if wr.shape[0] == E + 1 else None)


def embed_norm(ids: torch.Tensor, positions: torch.Tensor, embed: torch.Tensor, pos: Optional[torch.Tensor], src: Optional[torch.Tensor],
               prev: Optional[torch.Tensor], scale: float, vec: Optional[torch.Tensor], w: torch.Tensor, eps: float, one_plus: bool,
               route: Optional[tuple] = None) -> tuple:
    """(embed_pos's rows + ``vec``, add_norm's result for them - with ``route`` a pair, as there), in one launch on the GPU where
    rows are in 16-byte pieces; ``embed``'s dtype is the result's."""
    d = embed.shape[1]
    one = route is None or (embed.is_cuda and route_with_norm(ids.numel(), d, route[0].shape[0]))
    if not (embed.is_cuda and one and d % 8 == 0 and embed.data_ptr() % 16 == 0 and (pos is None or pos.data_ptr() % 16 == 0)):
        x = embed_pos(ids, positions, embed, pos, src, prev, scale=scale)
        return x, add_norm(x, (), vec, w, eps, one_plus, embed.dtype, route=route)
    x = torch.empty(ids.numel(), d, dtype=torch.float32, device=embed.device)
    out = torch.empty(x.shape, dtype=embed.dtype, device=embed.device)
    wr, bias, E, K = route or (None, None, 0, 0)
    routed = _route_out(x, route)
    native().embed_norm(out, x, ids, positions, embed, pos, src, prev, float(scale), vec, w, float(eps), bool(one_plus), *routed, wr, bias, E, K)
    return x, (out if route is None else (out, routed))


def route_with_norm(T: int, d: int, rows_w: int) -> bool:
    """Steps whose router runs in the norm's launch: few rows, for a row reads all router weights (hy_router_walk_kernel keeps them for many)."""
    return T < 256 and d % 8 == 0 and d > 0 and rows_w <= 9


def sum_norm(residual: torch.Tensor, addends: tuple, normed: Optional[tuple], w: Optional[torch.Tensor], eps: float,
             center: bool, one_plus: bool, out_dtype: torch.dtype) -> torch.Tensor:
    """``residual`` (fp32 [T, d], updated in place) += sum of ``scale * a`` over ``addends`` (at most
    two (a [T, d] of any float dtype, scale) pairs) + ``y / sqrt(mean(y^2) + eps) * wy`` for ``normed``
    = (y [T, d], wy [d] fp32) - a branch that joins the stream through an RMS norm of its own.  Returns
    the norm of the new residual times ``w`` (``one_plus``: ``1 + w``) in ``out_dtype``: ``center`` False
    the RMS norm, True the layer norm ``(x - mean) / sqrt(mean((x - mean)^2) + eps)``.  ``w`` None: no
    norm, the new residual itself in ``out_dtype``.  Sums and norms are fp32."""
    if not residual.is_cuda:
        for a, sc in addends:
            residual += a.float() * sc if sc != 1.0 else a.float()
        if normed is not None:
            y = normed[0].float()
            residual += y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + eps) * normed[1].float()
        if w is None:
            return residual.to(out_dtype)
        x = residual - residual.mean(-1, keepdim=True) if center else residual
        h = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
        wf = w.float()
        return (h * (1.0 + wf if one_plus else wf)).to(out_dtype)
    assert len(addends) <= 2
    out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
    a = list(addends) + [(None, 1.0)] * (2 - len(addends))
    yn, wy = normed if normed is not None else (None, None)
    native().sum_norm(out, residual, a[0][0], float(a[0][1]), a[1][0], float(a[1][1]), yn, wy, w, float(eps), bool(center),
                      bool(one_plus))
    return out


def join_norm(residual: torch.Tensor, branch: tuple, post: Optional[tuple], pre: Optional[tuple], eps: float,
              out_dtype: torch.dtype, branch_w: Optional[tuple] = None, mix: float = 1.0) -> Optional[torch.Tensor]:
    """A sublayer's result through a layer norm of its own into the stream, then the next sublayer's norm.
    ``branch``: () (nothing joins), (y,) or (y0, y1) ([T, d] of any float dtype); two results are first
    RMS-normed each and combined, ``b = mix * (y0 / rms(y0) * w0 + y1 / rms(y1) * w1)`` with ``branch_w`` =
    (w0, w1).  ``residual`` (fp32 [T, d], updated in place) += ``LN(b) * post[0] + post[1]``; returns
    ``LN(residual) * pre[0] + pre[1]`` in ``out_dtype`` (``pre`` None: nothing).  LN(x) = (x - mean) /
    sqrt(mean((x - mean)^2) + eps).  Norms and sums are fp32."""
    if not residual.is_cuda:
        def ln(x, wb):
            x = x - x.mean(-1, keepdim=True)
            return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * wb[0].float() + wb[1].float()

        if branch:
            b = branch[0].float()
            if len(branch) == 2:
                ys = [y.float() for y in branch]
                ys = [y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + eps) * w.float() for y, w in zip(ys, branch_w)]
                b = mix * (ys[0] + ys[1])
            residual += ln(b, post)
        return ln(residual, pre).to(out_dtype) if pre is not None else None
    out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device) if pre is not None else None
    y = list(branch) + [None] * (2 - len(branch))
    w0, w1 = branch_w if len(branch) == 2 else (None, None)
    pw, pb = post if branch else (None, None)
    nw, nb = pre if pre is not None else (None, None)
    native().join_norm(out, residual, y[0], y[1], w0, w1, float(mix), pw, pb, nw, nb, float(eps))
    return out


def stream_norm(src: torch.Tensor, y: Optional[torch.Tensor], write: Optional[tuple], read: Optional[torch.Tensor],
                w: torch.Tensor, eps: float, out_dtype: torch.dtype, S: int) -> tuple:
    """Several residual streams per token.  ``src`` [T, S, d] fp32, or [T, 1, d] for S equal streams (the
    model's start).  ``y`` [T, d] (any float dtype; None: nothing is written) with ``write`` = (mix [S, S],
    out [S]) fp32: every stream t becomes ``sum_s mix[s, t] x_s + out[t] y`` of the streams before.
    Then with ``read`` [S] fp32 (None: all ones) ``u = sum_t read[t] x_t``.  Returns (the RMSNorm of u times
    ``w`` in ``out_dtype`` [T, d], the new streams [T, S, d] - ``src`` itself, updated in place, where it holds
    all of them).  Sums and norm are fp32."""
    T, n, d = src.shape
    if not src.is_cuda:
        x = src
        if y is not None:
            x = torch.einsum("nsd,st->ntd", src.expand(T, S, d), write[0].float()) + write[1].float().view(1, S, 1) * y.float().unsqueeze(1)
            if n == S:
                src.copy_(x)
                x = src
        u = x.expand(T, S, d).sum(1) if read is None else torch.einsum("nsd,s->nd", x.expand(T, S, d), read.float())
        return (u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + eps) * w.float()).to(out_dtype), x
    out = torch.empty(T, d, dtype=out_dtype, device=src.device)
    dst = None
    if y is not None:
        dst = src if n == S else torch.empty(T, S, d, dtype=torch.float32, device=src.device)
    mix, wo = write if y is not None else (None, None)
    native().stream_norm(out, dst, src, int(S), y, mix, wo, read, w, float(eps))
    return out, (dst if dst is not None else src)


def token_mix(h: torch.Tensor, mu: torch.Tensor, state: torch.Tensor, seg_cu: torch.Tensor, seg_ctx: torch.Tensor,
              seg_slot: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """Token-shift mixes of normed rows ``h`` (fp32 [T, d]): [T, n, d] in ``out_dtype`` with
    ``h[t] + (h[t-1] - h[t]) * mu[j]`` for the ``n`` rows of ``mu`` (fp32, up to 8).  The row before a
    segment's first comes from ``state[slot]`` ([slots, d] fp32; zeros where seg_ctx is 0), which then
    takes the segment's last row."""
    T, d = h.shape
    n = mu.shape[0]
    if not h.is_cuda:
        prev = torch.zeros_like(h)
        prev[1:] = h[:-1]
        cul = seg_cu.tolist()
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if b <= a:
                continue
            prev[a] = state[slot] if (c0 > 0 and slot >= 0) else 0.0
            if slot >= 0:
                state[slot] = h[b - 1]
        return (h[:, None] + (prev - h)[:, None] * mu[None]).to(out_dtype)
    out = torch.empty(T, n, d, dtype=out_dtype, device=h.device)
    native().token_mix(out, h, mu, state, seg_cu, seg_ctx, seg_slot)
    return out


def gated_lookup(gate: torch.Tensor, table: torch.Tensor, ids: torch.Tensor, col: int,
                 src: Optional[torch.Tensor] = None, prev: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``gelu_tanh(gate) * table[id, col : col + n]`` for ``gate`` [T, n]: a per-token table slice gated
    by a projection of the stream (fp32 arithmetic, result in the gate's dtype).  ``src`` / ``prev``: as
    in embed_pos."""
    n = gate.shape[1]
    if not gate.is_cuda:
        if src is not None:
            ids = torch.where(src >= 0, prev.index_select(0, src.clamp(min=0).long()), ids)
        e = table[ids.long(), col:col + n].float()
        return (F.gelu(gate.float(), approximate="tanh") * e).to(gate.dtype)
    out = torch.empty_like(gate)
    native().gated_lookup(out, gate, table, ids, int(col), src, prev)
    return out


def gated_add_norm(residual: torch.Tensor, y: torch.Tensor, proj: torch.Tensor, g_col: int, bias: torch.Tensor,
                   mult: float, w: torch.Tensor, eps: float, one_plus: bool, out_dtype: torch.dtype) -> torch.Tensor:
    """Gated residual: ``residual`` (fp32 [T, d], updated in place) += ``mult * y * sigmoid(g + bias)``
    with the gate logits ``g = proj[:, g_col : g_col + d]`` (a column range of a wider projection of
    the sublayer's input, activation dtype) and ``bias`` [d] fp32; returns the RMSNorm of the new
    residual times ``w`` (``one_plus``: ``1 + w``) in ``out_dtype``.  ``y`` [T, d]: any float dtype.
    Sigmoid, product, sum and norm are fp32."""
    d = residual.shape[1]
    if not residual.is_cuda:
        g = proj[:, g_col:g_col + d].float() + bias.float()
        residual += mult * y.float() * torch.sigmoid(g)
        h = residual * torch.rsqrt(residual.pow(2).mean(-1, keepdim=True) + eps)
        wf = w.float()
        return (h * (1.0 + wf if one_plus else wf)).to(out_dtype)
    out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
    native().gated_add_norm(out, residual, y.contiguous(), proj, int(g_col), bias, float(mult), w, float(eps), bool(one_plus))
    return out


class GatedRows:
    """The rows that ``gated_add_norm`` would make, not made yet: the first ``linear`` or ``linear_glu`` of them has the sum and the norm as its
    prologue (few_rows.hip) where there are few enough; anything else makes them first.  ``residual`` is the new residual behind that."""

    def __init__(self, residual, y, proj, g_col, bias, mult, w, eps, one_plus, dtype):
        self.args = (residual, y, proj, g_col, bias, mult, w, eps, one_plus)
        self.dtype, self.shape, self.is_cuda, self.rows = dtype, residual.shape, True, None

    @staticmethod
    def take(residual: torch.Tensor, y: torch.Tensor, proj: torch.Tensor, g_col: int, *rest) -> bool:
        """Whether the prologue is this sum's and norm's: bf16 on the device, everything in 16-byte pieces, no gradients."""
        M, d = residual.shape
        return (residual.is_cuda and 0 < M <= (GATED_ROWS if d <= 1024 else 2) and d <= 2048 and d % 32 == 0 and y.dtype == proj.dtype == torch.bfloat16
                and residual.dtype == torch.float32 and residual.is_contiguous() and y.is_contiguous() and y.shape == residual.shape
                and proj.dim() == 2 and proj.stride(1) == 1 and proj.stride(0) % 8 == 0 and g_col % 8 == 0
                and all(t.data_ptr() % 16 == 0 for t in (residual, y, proj, rest[0], rest[2]))
                and not (torch.is_grad_enabled() and any(t.requires_grad for t in (residual, y, proj, rest[0], rest[2]))))

    @property
    def residual(self) -> torch.Tensor:
        if self.rows is None and not self.done:
            self.tensor()
        return self.new

    done, new = False, None

    def tensor(self) -> torch.Tensor:
        """The rows as a tensor (the residual is updated in place if no product has made a new one)."""
        if self.rows is None:
            if self.done:
                self.rows = add_norm(self.new, (), None, self.args[6], self.args[7], self.args[8], self.dtype)
            else:
                self.rows, self.new = gated_add_norm(*self.args, self.dtype), self.args[0]
        return self.rows

    def product(self, w: torch.Tensor, f: int = 0, kind: str = "") -> Optional[tuple]:
        """(unit or None, product of the other rows of w) with the rows made on the way; None: this product is not the prologue's."""
        x, y, proj, g_col, bias, mult, nw, eps, one_plus = self.args
        M = x.shape[0]
        if (self.done or self.rows is not None or w.dtype != torch.bfloat16 or w.dim() != 2 or not w.is_contiguous() or w.data_ptr() % 16
                or w.shape[1] != x.shape[1] or (torch.is_grad_enabled() and w.requires_grad)
                or _rows_form(M, w.shape[0], w.shape[1], "glu" if f else "") is None or w.shape[0] > GATED_COLUMNS):
            return None
        a = torch.empty(M, f, dtype=self.dtype, device=x.device) if f else None
        z = torch.empty(M, w.shape[0] - 2 * f, dtype=self.dtype, device=x.device)
        self.new, self.done = torch.empty_like(x), True
        native().few_rows_gated(z, a, x, self.new, y, proj, int(g_col), bias, float(mult), nw, float(eps), bool(one_plus), w,
                                ACTS[kind] if f else -1)
        return a, z


GATED_ROWS, GATED_COLUMNS = 4, 16384  # the most that its prologue takes


def gated_rows(residual: torch.Tensor, y: torch.Tensor, proj: torch.Tensor, g_col: int, bias: torch.Tensor, mult: float, w: torch.Tensor,
               eps: float, one_plus: bool, out_dtype: torch.dtype):
    """``gated_add_norm``, or the GatedRows of it where a product can make them."""
    args = (residual, y, proj, g_col, bias, mult, w, eps, one_plus)
    if out_dtype == torch.bfloat16 and GatedRows.take(*args):
        return GatedRows(*args, out_dtype)
    return gated_add_norm(*args, out_dtype)


def norm_shift(residual: torch.Tensor, addends: tuple, w: torch.Tensor, eps: float, one_plus: bool,
               mu: torch.Tensor, state: torch.Tensor, seg_cu: torch.Tensor, seg_ctx: torch.Tensor,
               seg_slot: torch.Tensor, out_dtype: torch.dtype, advance: bool = True,
               multi: bool = True) -> torch.Tensor:
    """Token-shifted norm.  ``residual`` (fp32 [T, d], updated in place) += ``addends``; with
    ``h[t]`` the RMSNorm of row t times ``w`` (fp32), returns ``h[t] + (h[t-1] - h[t]) * mu`` in
    ``out_dtype``, where the row before a segment's first comes from ``state[slot]`` ([slots, d]
    fp32; zeros where seg_ctx is 0).  ``advance``: ``state[slot]`` then takes the segment's last
    ``h`` (unshifted).  GPU: the state of segments longer than one row is advanced by a second
    small launch, after every row has read the old state (``multi`` False: the caller knows every
    segment is one row, as in a decode step, and that launch is left out)."""
    if not residual.is_cuda:
        for a in addends:
            residual += a.float()
        h = residual * torch.rsqrt(residual.pow(2).mean(-1, keepdim=True) + eps)
        wf = w.float()
        h = h * (1.0 + wf if one_plus else wf)
        prev = torch.zeros_like(h)
        prev[1:] = h[:-1]
        cul = seg_cu.tolist()
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if b <= a:
                continue
            prev[a] = state[slot] if (c0 > 0 and slot >= 0) else 0.0
            if advance and slot >= 0:
                state[slot] = h[b - 1]
        return (h + (prev - h) * mu.float()).to(out_dtype)
    for a in addends:  # a row also norms its predecessor, so the stream is complete before the launch
        residual += a
    out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
    native().norm_shift(out, residual, w, float(eps), bool(one_plus), mu, state, seg_cu, seg_ctx, seg_slot,
                        bool(advance), bool(multi))
    return out


def depth_mix(stack: torch.Tensor, n: int, addend: Optional[torch.Tensor], coef: torch.Tensor) -> torch.Tensor:
    """Depth-weighted average.  ``stack`` [L, T, d] fp32 holds the embedding output and the layer
    results so far in entries 0 .. n (entry n is the newest, still missing ``addend``):
    ``stack[n] += addend``, then ``stack[n + 1] = sum_j coef[j] * stack[j]`` over j = 0 .. n
    (``coef`` [n + 1] fp32).  Returns ``stack[n + 1]``, the next layer's input."""
    if not stack.is_cuda:
        if addend is not None:
            stack[n] += addend.float()
        stack[n + 1] = torch.einsum("j,jtd->td", coef.float(), stack[: n + 1])
        return stack[n + 1]
    native().depth_mix(stack, int(n), addend, coef)
    return stack[n + 1]


ACTS = {"gelu": 0, "gelu_tanh": 1, "xielu": 2, "silu": 3, "relu": 4, "clamped_swish": 5, "relu_sq": 6, "tanh": 7}


def _act_torch(z: torch.Tensor, kind: str) -> torch.Tensor:
    if kind == "gelu":
        return F.gelu(z)
    if kind == "gelu_tanh":
        return F.gelu(z, approximate="tanh")
    if kind == "silu":
        return _silu(z)
    if kind == "relu":
        return torch.relu(z)
    if kind == "relu_sq":
        return torch.relu(z) ** 2
    if kind == "tanh":
        return torch.tanh(z)
    raise ValueError(kind)


def _clamped_unit(g: torch.Tensor, u: torch.Tensor, limit: float) -> torch.Tensor:
    """Experts with clamped pre-activations: g <- min(g, limit), u <- clamp(u, -limit, limit);
    g * sigmoid(1.702 g) * (u + 1)."""
    g = g.clamp(max=limit)
    u = u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def activation(x: torch.Tensor, kind: str, a: float = 0.0, b: float = 0.0) -> torch.Tensor:
    """Elementwise on [T, f] rows, evaluated in fp32: ``gelu`` (erf form), ``gelu_tanh``, ``silu``, ``relu_sq``, ``tanh``, or
    ``xielu`` with the two positive constants ``a``, ``b``:  z > 0: a z^2 + z / 2;  z <= 0:
    b (exp(z) - 1 - z) + z / 2."""
    if not x.is_cuda:
        z = x.float()
        if kind == "xielu":
            y = torch.where(z > 0, a * z * z + 0.5 * z, b * (torch.expm1(z.clamp(max=0.0)) - z) + 0.5 * z)
        else:
            y = _act_torch(z, kind)
        return y.to(x.dtype)
    out = torch.empty_like(x)
    native().activation(out, x, ACTS[kind], float(a), float(b))
    return out


def activation_cols(proj: torch.Tensor, col: int, n: int, kind: str) -> torch.Tensor:
    """``act(proj[:, col : col + n])`` as a contiguous [T, n] tensor (``gelu``, ``gelu_tanh`` or
    ``silu``, evaluated in fp32): the activation of a column range of a wider projection."""
    if not proj.is_cuda:
        return _act_torch(proj[:, col:col + n].float(), kind).to(proj.dtype)
    out = torch.empty(proj.shape[0], n, dtype=proj.dtype, device=proj.device)
    native().activation_cols(out, proj, int(col), ACTS[kind])
    return out


def glu(proj: torch.Tensor, col: int, f: int, kind: str, limit: float = 0.0) -> torch.Tensor:
    """Gated linear unit ``act(proj[:, col : col + f]) * proj[:, col + f : col + 2 f]`` ([gate | up]
    columns of a possibly wider projection) with ``kind`` ``gelu_tanh``, ``silu`` or ``relu``, or
    ``clamped_swish``: with g = min(gate, limit) and u = clamp(up, -limit, limit),
    ``g * sigmoid(1.702 g) * (u + 1)``.  fp32 arithmetic, [T, f] in the activation dtype."""
    if not proj.is_cuda:
        g, u = proj[:, col:col + f].float(), proj[:, col + f:col + 2 * f].float()
        if kind == "clamped_swish":
            return _clamped_unit(g, u, limit).to(proj.dtype)
        return (_act_torch(g, kind) * u).to(proj.dtype)
    out = torch.empty(proj.shape[0], f, dtype=proj.dtype, device=proj.device)
    native().glu(out, proj, int(col), ACTS[kind], float(limit))
    return out


def sigmoid_gate(x: torch.Tensor, proj: torch.Tensor, col: int) -> torch.Tensor:
    """In place: ``x`` [T, n] *= sigmoid(proj[:, col : col + n]) (fp32 arithmetic)."""
    n = x.shape[1]
    if not x.is_cuda:
        x.copy_((x.float() * torch.sigmoid(proj[:, col:col + n].float())).to(x.dtype))
        return x
    native().sigmoid_gate(x, proj, int(col))
    return x


def _gate_values(x: torch.Tensor, gate: torch.Tensor, col: int) -> torch.Tensor:
    return sigmoid_gate(x, gate if gate.shape[0] == x.shape[0] else gate[:x.shape[0]], col)


def softcap(logits: torch.Tensor, cap: float) -> torch.Tensor:
    """In place on fp32 logits: ``cap * tanh(logits / cap)``."""
    if not logits.is_cuda:
        return logits.copy_(cap * torch.tanh(logits / cap))
    native().softcap(logits, float(cap))
    return logits


# ---------------------------------------------------------------- windowed attention with a sink

def qk_norm_cache(qkv: torch.Tensor, qw: torch.Tensor, kw: torch.Tensor, eps: float, Hq: int, Hkv: int, dk: int,
                  dv: int, k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor],
                  slot_mapping: Optional[torch.Tensor], singles: bool = False) -> None:
    """In place on the fused rows [T, Hq*dk | Hkv*dk | Hkv*dv]: q and k are each divided by the
    root mean square of their WHOLE projection (all heads together, fp32) and multiplied by
    ``qw`` / ``kw``; the normed k and v go to the paged cache at ``slot_mapping`` (< 0: not
    written).  ``singles``: as in rotary_cache."""
    nq, nk = Hq * dk, Hkv * dk
    if not qkv.is_cuda:
        q, k = qkv[:, :nq].float(), qkv[:, nq:nq + nk].float()
        q = q * torch.rsqrt(q.pow(2).mean(-1, keepdim=True) + eps) * qw.float()
        k = k * torch.rsqrt(k.pow(2).mean(-1, keepdim=True) + eps) * kw.float()
        qkv[:, :nq] = q.to(qkv.dtype)
        qkv[:, nq:nq + nk] = k.to(qkv.dtype)
        if k_cache is not None:
            ok = slot_mapping >= 0
            s = slot_mapping[ok].long()
            k_cache.view(-1, nk)[s] = qkv[ok, nq:nq + nk]
            bs = k_cache.shape[1]
            v_cache.view(-1, Hkv * dv, bs)[s // bs, :, s % bs] = qkv[ok, nq + nk:]
        return
    native().qk_norm_cache(qkv, qw, kw, float(eps), Hq, Hkv, dk, dv, k_cache, v_cache, slot_mapping, bool(singles))


def rotary_cache(qkv: torch.Tensor, Hq: int, Hkv: int, dk: int, dv: int, positions: torch.Tensor, freq: torch.Tensor,
                 pairs: bool, q_scale: Optional[torch.Tensor], k_cache: Optional[torch.Tensor],
                 v_cache: Optional[torch.Tensor], slot_mapping: Optional[torch.Tensor], norm: int = 0,
                 qw: Optional[torch.Tensor] = None, kw: Optional[torch.Tensor] = None,
                 eps: float = 0.0, v_from_k: bool = False, singles: bool = False) -> None:
    """In place on the fused rows [T, Hq*dk | Hkv*dk | Hkv*dv | ...]: the first ``2 len(freq)`` entries
    of every query and key head turn by the angle ``position * freq[i]`` (fp32; ``pairs``: entry 2i
    with 2i + 1, else entry i with i + len(freq); rotary_freq); the rest of a head passes.  ``q_scale``
    [Hq] fp32 (optional): every query head is multiplied by its number in the same pass (a per-head
    temperature folded into the query).  Keys (turned) and values go to the paged cache at
    ``slot_mapping`` (< 0: not written).

    ``norm``: every query and key head is also RMS-normed over its ``dk`` entries (fp32, ``eps`` inside
    the root) - 1: BEFORE the turn, times ``qw`` / ``kw`` ([dk] fp32, shared by the heads); 2: AFTER the
    turn, no weight.  ``v_from_k``: there are no value columns; the values are the keys as projected
    (before norm and turn), ``dv == dk``.  ``singles``: every row is another sequence's (GPU: values are then not written by
    runs of slots)."""
    nq, nk, nv = Hq * dk, Hkv * dk, Hkv * dv
    if not qkv.is_cuda:
        T = qkv.shape[0]

        def rms(x):
            return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)

        def turn(x, w):
            x = x.clone()
            if norm == 1:
                x = rms(x) * w.float()
            x = _rotate(x, positions, freq, pairs)
            return rms(x) if norm == 2 else x

        q = turn(qkv[:, :nq].float().view(T, Hq, dk), qw)
        if q_scale is not None:
            q = q * q_scale.float().view(1, Hq, 1)
        k_raw = qkv[:, nq:nq + nk].clone()
        k = qkv[:, nq:nq + nk].float().view(T, Hkv, dk)
        k = turn(k, kw)
        qkv[:, :nq] = q.reshape(T, nq).to(qkv.dtype)
        qkv[:, nq:nq + nk] = k.reshape(T, nk).to(qkv.dtype)
        if k_cache is not None:
            ok = slot_mapping[:T] >= 0
            s = slot_mapping[:T][ok].long()
            k_cache.view(-1, nk)[s] = qkv[ok, nq:nq + nk]
            bs = k_cache.shape[1]
            v_cache.view(-1, nv, bs)[s // bs, :, s % bs] = k_raw[ok] if v_from_k else qkv[ok, nq + nk:nq + nk + nv]
        return
    if norm or v_from_k:
        native().rotary_norm_cache(qkv, Hq, Hkv, dk, dv, positions, freq, bool(pairs), int(norm), qw, kw, float(eps), q_scale,
                                   k_cache, v_cache, slot_mapping, bool(v_from_k))
        return
    native().rotary_cache(qkv, Hq, Hkv, dk, dv, positions, freq, bool(pairs), q_scale, k_cache, v_cache, slot_mapping, bool(singles))


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float, sink: bool,
            sinks: Optional[torch.Tensor] = None, cap: float = 0.0) -> torch.Tensor:
    """q [H, dk], k [n, G, dk], v [n, G, dv] (fp32) -> [H, dv].  ``sinks`` [H]: the sink's logit per
    head (absent: 0)."""
    H, G = q.shape[0], k.shape[1]
    kk = k.repeat_interleave(H // G, dim=1)
    vv = v.repeat_interleave(H // G, dim=1)
    s = torch.einsum("hd,nhd->hn", q, kk) * scale
    if cap > 0:
        s = cap * torch.tanh(s / cap)
    m = s.max(-1, keepdim=True).values
    z = sinks.float().view(H, 1) if sinks is not None else torch.zeros(H, 1)
    if sink:
        m = torch.maximum(m, z)
    e = torch.exp(s - m)
    den = e.sum(-1, keepdim=True) + (torch.exp(z - m) if sink else 0.0)
    return torch.einsum("hn,nhd->hd", e / den, vv)


def _first_key(p: int, window: int, chunked: bool) -> int:
    """The first position that a row at position ``p`` sees."""
    if window <= 0:
        return 0
    return p - p % window if chunked else max(0, p - window + 1)


def _visible(p: int, window: int, chunked: bool, keep: int) -> list:
    """The positions that a row at position ``p`` sees."""
    lo = _first_key(p, window, chunked)
    return list(range(min(keep, lo))) + list(range(lo, p + 1))


def _head_gate(o: torch.Tensor, gate: Optional[torch.Tensor], g_col: int) -> torch.Tensor:
    """o [H, dv] (one row's heads) times sigmoid of that row's gate logits."""
    return o if gate is None else o * torch.sigmoid(gate[g_col:g_col + o.shape[0]].float()).unsqueeze(-1)


def window_attention_prefill(qkv: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cu: torch.Tensor,
                             ctx: torch.Tensor, block_tables: torch.Tensor, Hq: int, Hkv: int, dk: int, dv: int,
                             scale: float, window: int, sink: bool, mfma: int = 1,
                             sinks: Optional[torch.Tensor] = None, chunked: bool = False, cap: float = 0.0, keep: int = 0,
                             gate: Optional[torch.Tensor] = None, g_col: int = 0, by_value: bool = False,
                             out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Attention of the step's prompt chunks over the paged cache (which already holds their own
    keys): row r of segment s at position p = ctx[s] + r sees positions max(0, p - window + 1) .. p
    (``window`` 0: all of 0 .. p), or with ``chunked`` those of its own chunk of ``window`` positions,
    p - p % window .. p (chunks count from position 0).  ``keep``: with a sliding window, the first ``keep``
    positions of the sequence stay visible too.  ``gate``: rows of a projection [T, *]; head h of a row is
    multiplied by sigmoid(gate[row, g_col + h]) before it is rounded; ``by_value``: value d of head h of the rounded row by
    sigmoid(gate[row, g_col + h * dv + d]), as sigmoid_gate does.  ``out``: the rows to write [T, Hq*dv].  ``cap`` > 0: a score s (after ``scale``) becomes
    ``cap * tanh(s / cap)``.  ``sink``: the softmax denominator has one more term that carries
    no value - exp(0), or exp(sinks[h]) for head h where ``sinks`` [Hq] fp32 is given (a learned,
    unscaled logit).  Scores and weights are fp32.  Returns [T, Hq*dv].  GPU, bf16, head sizes
    64 / 128: the matrix-core kernels - tiles staged in LDS for large steps and long contexts, else 16
    query rows per wave (``mfma`` 0: the any-size wave-per-row kernel; 2: the register kernel; 16 / 32 / 64: with
    that many rows per wave; 256: the staged kernel); fp32, the same sizes: 16 rows per wave on the fp32
    matrix instruction."""
    T = qkv.shape[0]
    if out is None:
        out = torch.empty(T, Hq * dv, dtype=qkv.dtype, device=qkv.device)
    hg = None if by_value else gate
    if not qkv.is_cuda:
        bs = k_cache.shape[1]
        cul, ctxl = cu.tolist(), ctx.tolist()
        for s in range(len(ctxl)):
            n_all = ctxl[s] + cul[s + 1] - cul[s]
            bt = block_tables[s, : (n_all + bs - 1) // bs].long()
            ks = k_cache[bt].reshape(-1, Hkv, dk)[:n_all].float()
            vs = v_cache[bt].permute(0, 3, 1, 2).reshape(-1, Hkv, dv)[:n_all].float()
            for r in range(cul[s], cul[s + 1]):
                p = ctxl[s] + r - cul[s]
                js = _visible(p, window, chunked, keep)
                o = _attend(qkv[r, : Hq * dk].float().view(Hq, dk), ks[js], vs[js], scale, sink, sinks, cap)
                out[r] = _head_gate(o, hg[r] if hg is not None else None, g_col).reshape(-1).to(qkv.dtype)
        return _gate_values(out, gate, g_col) if by_value and gate is not None else out
    gated = native().window_attention_prefill(out, qkv, k_cache, v_cache, cu, ctx, block_tables, Hq, Hkv, dk, dv, float(scale),
                                              int(window), bool(sink), sinks, int(mfma), bool(chunked), float(cap), int(keep), gate,
                                              int(g_col), bool(by_value))
    return _gate_values(out, gate, g_col) if by_value and gate is not None and not gated else out


def window_attention_decode(qkv: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                            block_tables: torch.Tensor, seq_lens: torch.Tensor, Hq: int, Hkv: int, dk: int, dv: int,
                            scale: float, window: int, sink: bool, vec: bool = True,
                            sinks: Optional[torch.Tensor] = None, chunked: bool = False, cap: float = 0.0, keep: int = 0,
                            gate: Optional[torch.Tensor] = None, g_col: int = 0, heads: int = 0, by_value: bool = False,
                            out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One query per sequence (its newest token, already in the cache) over the last ``window``
    cached positions (``chunked``: those of its own chunk; ``cap``, ``keep``, ``gate``, ``by_value``, ``out``: as in
    window_attention_prefill);
    ``seq_lens`` count that token (0: a padding row, output zero).  ``heads``: query heads of a kv
    head that a workgroup takes (GPU, ``vec``, bf16, head sizes of 64 and 128; 0: its choice, others are refused elsewhere)."""
    B = qkv.shape[0]
    if out is None:
        out = torch.empty(B, Hq * dv, dtype=qkv.dtype, device=qkv.device)
    hg = None if by_value else gate
    if not qkv.is_cuda:
        out.zero_()
        bs = k_cache.shape[1]
        for b, n in enumerate(seq_lens.tolist()):
            if n <= 0:
                continue
            js = _visible(n - 1, window, chunked, keep)
            bt = block_tables[b, : (n + bs - 1) // bs].long()
            ks = k_cache[bt].reshape(-1, Hkv, dk)[js].float()
            vs = v_cache[bt].permute(0, 3, 1, 2).reshape(-1, Hkv, dv)[js].float()
            o = _attend(qkv[b, : Hq * dk].float().view(Hq, dk), ks, vs, scale, sink, sinks, cap)
            out[b] = _head_gate(o, hg[b] if hg is not None else None, g_col).reshape(-1).to(qkv.dtype)
        return _gate_values(out, gate, g_col) if by_value and gate is not None else out
    gated = native().window_attention_decode(out, qkv, k_cache, v_cache, block_tables, seq_lens, Hq, Hkv, dk, dv, float(scale),
                                             int(window), bool(sink), sinks, bool(vec), bool(chunked), float(cap), int(keep), gate,
                                             int(g_col), int(heads), bool(by_value))
    return _gate_values(out, gate, g_col) if by_value and gate is not None and not gated else out


# ---------------------------------------------------------------- latent attention

def rotary_freq(base: float, dims: int, device=None, scaling: Optional[dict] = None) -> torch.Tensor:
    """The ``dims / 2`` rotation frequencies base^(-2i/dims) as fp32 (evaluated in float64).
    ``scaling`` {factor, low, high, original}: the long-context rescaling of Llama 3.1 - with the
    wavelength ``l = 2 pi / f``, a frequency stays where ``l < original / high``, becomes ``f / factor``
    where ``l > original / low``, and in between is ``(1 - s) f / factor + s f`` with
    ``s = (original / l - low) / (high - low)``."""
    f = torch.pow(torch.tensor(float(base), dtype=torch.float64), -2.0 * torch.arange(dims // 2, dtype=torch.float64) / dims)
    if scaling:
        fac, lo, hi, orig = (float(scaling[k]) for k in ("factor", "low", "high", "original"))
        lam = 2.0 * math.pi / f
        s = (orig / lam - lo) / (hi - lo) if hi != lo else torch.ones_like(f)
        mid = (1.0 - s) * f / fac + s * f
        f = torch.where(lam < orig / hi, f, torch.where(lam > orig / lo, f / fac, mid))
    return f.float().to(device) if device is not None else f.float()


def _rotate_half(v: torch.Tensor, pos: torch.Tensor, freq: torch.Tensor) -> torch.Tensor:
    """v [T, ..., n] fp32: with nf = len(freq), entries i and i + nf of the last axis (i < nf) turn by
    the angle pos * freq[i] (angles in fp32); entries from 2 nf on pass."""
    half = freq.numel()
    a = pos.float().view(-1, *([1] * (v.dim() - 1))) * freq.float()
    c, s = torch.cos(a), torch.sin(a)
    u, x = v[..., :half], v[..., half:2 * half]
    return torch.cat([u * c - x * s, x * c + u * s, v[..., 2 * half:]], -1)


def _rotate_pairs(v: torch.Tensor, pos: torch.Tensor, freq: torch.Tensor) -> torch.Tensor:
    """The same turn with entries 2i and 2i + 1 paired (i < len(freq))."""
    nf = freq.numel()
    a = pos[:v.shape[0]].float().view(-1, *([1] * (v.dim() - 1))) * freq.float()
    c, s = torch.cos(a), torch.sin(a)
    u, x = v[..., 0:2 * nf:2], v[..., 1:2 * nf:2]
    out = v.clone()
    out[..., 0:2 * nf:2] = u * c - x * s
    out[..., 1:2 * nf:2] = x * c + u * s
    return out


def _rotate(v: torch.Tensor, pos: torch.Tensor, freq: torch.Tensor, pairs: bool) -> torch.Tensor:
    return _rotate_pairs(v, pos, freq) if pairs else _rotate_half(v, pos[:v.shape[0]], freq)


def latent_prep(proj: torch.Tensor, q_rank: int, kv_rank: int, rot_dim: int, qw: torch.Tensor,
                kw: Optional[torch.Tensor], eps: float, positions: torch.Tensor, freq: torch.Tensor,
                k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor],
                slot_mapping: Optional[torch.Tensor], pairs: bool = False) -> None:
    """In place on the fused down-projections [T, q_rank | kv_rank | rot_dim] (or [T, q_rank] for a
    layer that reads another layer's cache): the query latent is RMS-normed (weight ``qw``); the
    key/value latent is RMS-normed (weight ``kw``) and the shared key part behind it is rotated by
    its position (``freq``: rotary_freq; ``pairs``: entries 2i and 2i + 1 turn together instead of i
    and i + len(freq)); both go to the pages at ``slot_mapping`` - the key page
    row is [latent | rotated part] (the page's rows may be wider: what lies behind is left as it is,
    zero), the value page holds the latent once more, dim-major."""
    T = proj.shape[0]
    if not proj.is_cuda:
        q = proj[:, :q_rank].float()
        proj[:, :q_rank] = (q * torch.rsqrt(q.pow(2).mean(-1, keepdim=True) + eps) * qw.float()).to(proj.dtype)
        if k_cache is None:
            return
        c = proj[:, q_rank:q_rank + kv_rank].float()
        c = (c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * kw.float()).to(proj.dtype)
        kr = _rotate(proj[:, q_rank + kv_rank:q_rank + kv_rank + rot_dim].float(), positions, freq, pairs).to(proj.dtype)
        proj[:, q_rank:q_rank + kv_rank] = c
        proj[:, q_rank + kv_rank:q_rank + kv_rank + rot_dim] = kr
        ok = slot_mapping[:T] >= 0
        s = slot_mapping[:T][ok].long()
        bs = k_cache.shape[1]
        k_cache.view(-1, k_cache.shape[2])[s, :kv_rank + rot_dim] = proj[ok, q_rank:q_rank + kv_rank + rot_dim]
        v_cache.view(-1, kv_rank, bs)[s // bs, :, s % bs] = c[ok]
        return
    native().latent_prep(proj, int(q_rank), int(kv_rank), int(rot_dim), qw, kw, float(eps), positions, freq,
                         k_cache, v_cache, slot_mapping, bool(pairs))


def latent_queries(q: torch.Tensor, q_lat: torch.Tensor, H: int, dim: int, rot_dim: int, positions: torch.Tensor,
                   freq: torch.Tensor, pitch: int = 0, pairs: bool = False) -> torch.Tensor:
    """The queries against the latent cache: per head [q_lat | rotated part | zeros], [T, H * pitch]
    (``pitch`` 0: R + rot_dim, no padding; else the key pages' row width).
    ``q`` [T, H * (dim + rot_dim)] are the up-projected queries (their last ``rot_dim`` entries per
    head are rotated by the position) and ``q_lat`` [H, T, R] the unrotated parts already
    multiplied into the latent space."""
    T, R = q.shape[0], q_lat.shape[2]
    pitch = pitch or R + rot_dim
    if not q.is_cuda:
        qr = _rotate(q.view(T, H, dim + rot_dim)[..., dim:].float(), positions, freq, pairs).to(q.dtype)
        pad = torch.zeros(T, H, pitch - R - rot_dim, dtype=q.dtype)
        return torch.cat([q_lat.transpose(0, 1), qr, pad], -1).reshape(T, H * pitch)
    out = torch.empty(T, H * pitch, dtype=q.dtype, device=q.device)
    native().latent_queries(out, q, q_lat, int(H), int(dim), int(rot_dim), positions, freq, bool(pairs))
    return out


# Up to these rows the per-head products of latent attention are latent_heads.hip's.  Us, library (with the rows put together) / own: queries,
# 8 heads of 96 + 32 over 256, 1 row 11.6 / 4.2, 64 13.5 / 4.7, 2048 23 / 10.7; 32 of 128 + 64 over 512, 64 rows 45 / 7.5, 2048 101 / 94.  Values,
# 8 of 128 over 256, 1 row 7.3 / 4.5, 256 9.7 / 5.9, 512 5.6 / 7.6; 32 of 128 over 512, 64 rows 9.4 / 8.5, 128 10.5 / 11.1, 256 14.3 / 19.4: there by
# their multiplications too.
HEAD_QUERY_ROWS, HEAD_VALUE_ROWS, HEAD_VALUE_WORK = 2048, 256, 1 << 28


def _head_rows(most: int, *ts: torch.Tensor) -> bool:
    return (ts[0].dtype == torch.bfloat16 and ts[0].is_cuda and ts[0].shape[0] <= most
            and all(t.dtype == torch.bfloat16 and t.data_ptr() % 16 == 0 for t in ts)
            and not (torch.is_grad_enabled() and any(t.requires_grad for t in ts)))


def latent_head_queries(q: torch.Tensor, w_uk: torch.Tensor, H: int, dim: int, rot_dim: int, positions: torch.Tensor,
                        freq: torch.Tensor, pitch: int = 0, pairs: bool = False) -> torch.Tensor:
    """latent_queries of the unrotated parts times each head's key expansion ``w_uk`` [H * dim, R]."""
    T, R = q.shape[0], w_uk.shape[1]
    pitch = pitch or R + rot_dim
    if _head_rows(HEAD_QUERY_ROWS, q, w_uk) and not (dim % 8 or rot_dim % 8 or R % 8 or pitch % 8 or q.stride(0) % 8):
        out = torch.empty(T, H * pitch, dtype=q.dtype, device=q.device)
        native().latent_head_queries(out, q, w_uk, int(H), int(dim), int(rot_dim), positions, freq, bool(pairs))
        return out
    q_lat = torch.bmm(q.view(T, H, dim + rot_dim)[:, :, :dim].transpose(0, 1), w_uk.view(H, dim, R))
    return latent_queries(q, q_lat, H, dim, rot_dim, positions, freq, pitch, pairs)


def latent_head_values(o: torch.Tensor, w_uv: torch.Tensor, H: int, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Per head ``W_uv[h] o[t][h]``: [T, H * R] and ``w_uv`` [H * vdim, R] -> [T, H * vdim] (``out``: its rows)."""
    T, R = o.shape[0], w_uv.shape[1]
    dv = w_uv.shape[0] // H
    v = (torch.empty(T, H * dv, dtype=o.dtype, device=o.device) if out is None else out).view(T, H, dv)
    if _head_rows(HEAD_VALUE_ROWS, o, w_uv) and R % 8 == 0 and T * H * dv * R < HEAD_VALUE_WORK:
        native().latent_head_values(v, o, w_uv, int(H))
    else:  # written head by head into the rows that the out-projection reads (a right operand that is a transposed view has faulted in bf16)
        torch.bmm(o.view(T, H, R).transpose(0, 1), w_uv.view(H, dv, R).transpose(1, 2).contiguous(), out=v.transpose(0, 1))
    return v.view(T, H * dv)


def rotate_heads(x: torch.Tensor, heads: int, dim: int, positions: torch.Tensor, freq: torch.Tensor, pairs: bool,
                 rot_off: int = 0) -> None:
    """In place on rows [T, heads * dim]: entries ``rot_off .. rot_off + 2 len(freq)`` of every head turn by the
    row's position, as in rotary_cache."""
    if not x.is_cuda:
        T = x.shape[0]
        v = x[:, :heads * dim].float().view(T, heads, dim)
        turned = _rotate(v[..., rot_off:], positions, freq, pairs)
        x[:, :heads * dim] = torch.cat([v[..., :rot_off], turned], -1).reshape(T, heads * dim).to(x.dtype)
        return
    native().rotate_heads(x, int(heads), int(dim), positions, freq, bool(pairs), int(rot_off))


def latent_expand(k_cache: torch.Tensor, page_list: torch.Tensor, w_uk: torch.Tensor, w_uv: torch.Tensor, H: int, kv_rank: int,
                  rot_dim: int) -> tuple:
    """Per-head keys and values of the latent pages ``page_list`` names, as temporary pages of the windowed
    attention kernels in the list's order: ([n, 16, H * (dim + rot_dim)], [n, H, vdim, 16]).  A key is ``[W_uk[h] c |
    shared part]``, a value ``W_uv[h] c``, rounded once.  GPU, bf16, kv_rank 128 / 256, dim and vdim multiples of 32,
    rot_dim of 8: one kernel; else matrix products over the gathered pages."""
    n, R = page_list.numel(), kv_rank
    dn, dv = w_uk.shape[0] // H, w_uv.shape[0] // H
    D = dn + rot_dim
    if k_cache.is_cuda and k_cache.dtype == torch.bfloat16 and R in (128, 256) and dn % 32 == 0 and dv % 32 == 0 and \
            rot_dim % 8 == 0 and k_cache.shape[2] % 8 == 0:
        kt = torch.empty(n, 16, H * D, dtype=k_cache.dtype, device=k_cache.device)
        vt = torch.empty(n, H, dv, 16, dtype=k_cache.dtype, device=k_cache.device)
        native().latent_expand(kt, vt, k_cache, page_list, w_uk, w_uv, int(H), int(rot_dim))
        return kt, vt
    rows = k_cache.index_select(0, page_list.long())
    bs = rows.shape[1]
    c = rows[..., :R].reshape(n * bs, R)
    kt = torch.empty(n, bs, H, D, dtype=k_cache.dtype, device=k_cache.device)
    kt[..., :dn] = F.linear(c, w_uk).view(n, bs, H, dn)
    kt[..., dn:] = rows[..., R:R + rot_dim].unsqueeze(2)
    vt = F.linear(c, w_uv).view(n, bs, H, dv).permute(0, 2, 3, 1).contiguous()
    return kt.view(n, bs, H * D), vt


_NO_SINK: dict = {}


def _no_sink(H: int, device) -> torch.Tensor:
    key = (H, str(device))
    if key not in _NO_SINK:
        _NO_SINK[key] = torch.full((H,), -1.0e30, dtype=torch.float32, device=device)
    return _NO_SINK[key]


def latent_attention(qa: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, block_tables: torch.Tensor,
                     H: int, scale: float, window: int, sinks: Optional[torch.Tensor], cu: Optional[torch.Tensor] = None,
                     ctx: Optional[torch.Tensor] = None, seq_lens: Optional[torch.Tensor] = None, fast: int = 1,
                     split: int = 0, sink: bool = True, gate: Optional[torch.Tensor] = None, g_col: int = 0) -> torch.Tensor:
    """Attention of ``qa`` [T, H * pitch] (latent_queries) over the latent pages: every head reads
    the one key stream ``k_cache`` [blocks, bs, pitch] and the one value stream ``v_cache`` [blocks, 1,
    kv_rank, bs]; sliding window and learned sinks as in window_attention_* (``sink`` False: an
    ordinary softmax, nothing but the keys in the denominator).  ``gate``: a sigmoid gate per row and head, as in
    window_attention_prefill.  ``cu`` / ``ctx``: prompt
    chunks (rows of segment s at positions ctx[s] ..); else ``seq_lens``: one row per sequence, at its
    newest token.  Returns [T, H * kv_rank].  GPU, bf16, pitch a multiple of 32 up to 320 and kv_rank a
    multiple of 16 up to 256 (``fast``): the matrix-core kernel, 16 heads of one token per tile
    (``split`` 1 / 2: one wave per one / two tokens, 4 / 8: that many waves share a token's window,
    32 / 33: pages staged in LDS for eight / four tokens of a chunk at a time; 0: by the step's size -
    large steps' chunks take 33, few rows 8); other sizes and fp32:
    the any-size kernels with one shared key/value head."""
    T, pitch, dv = qa.shape[0], k_cache.shape[2], v_cache.shape[2]
    if not sink:
        sinks = None
    if qa.is_cuda and fast and qa.dtype == torch.bfloat16:
        out = torch.empty(T, H * dv, dtype=qa.dtype, device=qa.device)
        # the matrix-core kernels start every row from a sink term; without one that term gets a logit
        # so low that its weight exp(logit - max) is exactly zero in fp32
        sk = sinks if sink else _no_sink(H, qa.device)
        if native().latent_attention(out, qa, k_cache, v_cache, cu, ctx, seq_lens, block_tables, int(H), float(scale),
                                     int(window), sk, int(split), gate, int(g_col)):
            return out
    args = (H, 1, pitch, dv, scale, window, bool(sink))
    kw = dict(sinks=sinks, gate=gate, g_col=g_col)
    if cu is not None:
        return window_attention_prefill(qa, k_cache, v_cache, cu, ctx, block_tables, *args, mfma=fast, **kw)
    return window_attention_decode(qa, k_cache, v_cache, block_tables, seq_lens, *args, vec=bool(fast), **kw)


def latent_parts(T: int, H: int, R: int, pages: int, window: int) -> tuple:
    """(parts, tiles from which on a row has them) of latent attention's T rows over tables of ``pages`` pages; one part: as a whole.  A workgroup of
    eight waves takes 4 us for each eight tiles (its loads of 16 key rows ask for 16 lines at a time), one a CU, so few rows are cut until half of the chip
    is busy, a tile a wave at least; behind that parts cost more in the merge than they save (1.2 us for each four, and their outputs' way through memory).
    Tables are as wide as the longest sequence may become, so a row of few tiles is one part by itself.  us with the values behind it, whole / so, tables of
    512 pages: 8 heads, 128 + 32 wide, 1 row of 20 keys 7.8 / 7.9, 333 10.6 / 10.2, 1500 21.4 / 12.2, 4800 51 / 14.4; 16 rows of 100 8.8 / 9.0, 700 14.2 / 13.4,
    1500 22.0 / 15.2; 64 of 333 11.3 / 11.4, 1500 26.1 / 19.9, 4800 62 / 36; 16 heads, 256 + 32, 1 of 20 11.9 / 11.5, 1500 36 / 16.0; 32 of 1500 39.9 / 24.0, 64 of
    333 18.5 / 18.7, 1500 40.3 / 32.3.  (With every row of such a table in 3 to 16 parts, 1 row of 20 keys took 10.6, 64 of 333 12.3 and 21.3.)"""
    wgs = T * -(-H // 16)
    if wgs == 0 or wgs > 64:
        return 1, 1
    least = 16 if wgs < 16 or (wgs <= 32 and R > 128) else 40  # 333 keys, 16 heads, 256 + 32: 16 rows 17.7 / 15.9, 64 18.5 / 21.3
    tiles = min(pages, window // 16 + 2) if window > 0 else pages
    return (min(max(128 // wgs, 3), 16, -(-tiles // 8)) if tiles >= least else 1), least


def latent_attention_values(qa: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, block_tables: torch.Tensor, H: int,
                            scale: float, window: int, sinks: Optional[torch.Tensor], w_uv: torch.Tensor, out: torch.Tensor,
                            cu: Optional[torch.Tensor] = None, ctx: Optional[torch.Tensor] = None,
                            seq_lens: Optional[torch.Tensor] = None, fast: int = 1, sink: bool = True,
                            gate: Optional[torch.Tensor] = None, g_col: int = 0, parts: int = 0, least: int = 1) -> bool:
    """``latent_attention`` and ``latent_head_values`` into ``out`` of rows too few to fill the chip, the window of a row of ``least`` tiles or more cut
    into up to ``parts`` (0: as many as pay) whose merge is the value expansion's prologue.  False: nothing was done, these are not such rows."""
    if parts == 0:
        parts, least = latent_parts(qa.shape[0], H, w_uv.shape[1], block_tables.shape[1], window)
        if parts == 1:
            return False
    if not (fast and _head_rows(HEAD_VALUE_ROWS, qa, w_uv) and out.is_contiguous()):
        return False
    return native().latent_attention_values(out, qa, k_cache, v_cache, cu, ctx, seq_lens, block_tables, int(H), float(scale), int(window),
                                            sinks if sink else _no_sink(H, qa.device), gate, int(g_col), w_uv, int(parts), int(least))


# ---------------------------------------------------------------- Mamba-2

def conv_silu(proj: torch.Tensor, col0: int, C: int, conv_w: torch.Tensor, conv_b: Optional[torch.Tensor],
              conv_state: torch.Tensor, seg_cu: torch.Tensor, seg_ctx: torch.Tensor,
              seg_slot: torch.Tensor) -> torch.Tensor:
    """Causal per-channel convolution + SiLU over columns [col0, col0 + C) of ``proj`` [T, *];
    ``conv_w`` [C, taps] (the last tap multiplies the current token), ``conv_b`` [C] (None: no bias).  The taps - 1
    inputs before a segment come from ``conv_state`` [slots, taps - 1, C] (zeros where seg_ctx is
    0), which is then advanced to the segment's end."""
    T = proj.shape[0]
    taps = conv_w.shape[1]
    if not proj.is_cuda:
        out = torch.empty(T, C, dtype=proj.dtype)
        wt = conv_w.float().t()  # [taps, C]
        bf = conv_b.float() if conv_b is not None else torch.zeros(C)
        cul = seg_cu.tolist()
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if slot < 0 or b <= a:
                continue
            x = proj[a:b, col0:col0 + C]
            hist = conv_state[slot, : taps - 1]
            if c0 <= 0:
                hist = torch.zeros_like(hist)
            full = torch.cat([hist.to(proj.dtype), x]).float()  # [taps - 1 + n, C]
            acc = bf.expand(b - a, C).clone()
            for j in range(taps):
                acc += full[j:j + b - a] * wt[j]
            out[a:b] = _silu(acc).to(proj.dtype)
            if taps > 1:
                conv_state[slot] = full[full.shape[0] - (taps - 1):].to(conv_state.dtype)
        return out
    out = torch.empty(T, C, dtype=proj.dtype, device=proj.device)
    native().conv_silu(out, proj, int(col0), conv_w, conv_b, conv_state, seg_cu, seg_ctx, seg_slot)
    return out


def ssm_scan(xbc: torch.Tensor, proj: Optional[torch.Tensor], dt_col: int, dt_bias: Optional[torch.Tensor],
             a_log: Optional[torch.Tensor], d_skip: Optional[torch.Tensor], state: torch.Tensor, seg_cu: torch.Tensor,
             seg_ctx: torch.Tensor, seg_slot: torch.Tensor, nh: int, P: int, N: int, G: int, mode: int = 0,
             decay: Optional[torch.Tensor] = None, col_tiles: int = 0, longest: int = 0, singles: int = 0) -> torch.Tensor:
    """The selective state-space recurrence, fp32, token by token within each segment:

        dt = softplus(proj[t, dt_col + h] + dt_bias[h]);  S <- exp(-exp(a_log[h]) dt) S + dt B_t x_t^T
        y_t = S^T C_t + d_skip[h] x_t

    ``xbc`` [T, nh*P | G*N | G*N] holds x, B, C (head h reads group h // (nh / G)); ``state``
    [slots, nh, N, P] fp32 is read at the segment's start (zero where seg_ctx is 0) and written
    back at its end.  Returns y [T, nh*P] fp32.

    GPU: two lane mappings of the same arithmetic, chosen by the step's mean segment length (``mode`` 1 / 2 forces the
    decode / the prompt one); steps of one token a segment take a pass over the states, with the decode mapping's bits.

    ``decay`` [nh] fp32 (then ``proj``, ``dt_bias``, ``a_log``, ``d_skip`` are not read): the
    recurrence with a fixed decay per head, step size 1 and no skip term,
    ``S <- decay[h] S + B_t x_t^T;  y_t = S^T C_t`` - linear attention with B, C, x = k, q, v
    (linear_attention below)."""
    T = xbc.shape[0]
    if not xbc.is_cuda:
        y = torch.zeros(T, nh * P, dtype=torch.float32)
        fixed = decay is not None
        A = torch.exp(a_log.float()) if not fixed else None
        Dk = d_skip.float() if not fixed else torch.zeros(nh)
        cul = seg_cu.tolist()
        inner = nh * P
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if slot < 0 or b <= a:
                continue
            S = state[slot].clone() if c0 > 0 else torch.zeros_like(state[slot])
            xs = xbc[a:b, :inner].float().view(-1, nh, P)
            Bs = xbc[a:b, inner:inner + G * N].float().view(-1, G, N).repeat_interleave(nh // G, dim=1)
            Cs = xbc[a:b, inner + G * N:].float().view(-1, G, N).repeat_interleave(nh // G, dim=1)
            if fixed:
                dt = torch.ones(b - a, nh)
                dec = decay.float().expand(b - a, nh)
            else:
                dt = F.softplus(proj[a:b, dt_col:dt_col + nh].float() + dt_bias.float(), threshold=30.0)
                dec = torch.exp(-A * dt)
            for t in range(b - a):
                S = dec[t, :, None, None] * S + dt[t, :, None, None] * Bs[t, :, :, None] * xs[t, :, None, :]
                y[a + t] = (torch.einsum("hnp,hn->hp", S, Cs[t]) + Dk[:, None] * xs[t]).reshape(-1)
            state[slot] = S
        return y
    y = torch.empty(T, nh * P, dtype=torch.float32, device=xbc.device)
    native().ssm_scan(y, xbc, proj, int(dt_col), dt_bias, a_log, d_skip, decay, state, seg_cu, seg_ctx, seg_slot, nh, P,
                      N, G, int(mode), int(col_tiles), int(longest), int(singles))
    return y


def linear_attention(vkq: torch.Tensor, decay: torch.Tensor, state: torch.Tensor, seg_cu: torch.Tensor,
                     seg_ctx: torch.Tensor, seg_slot: torch.Tensor, H: int, dk: int, dv: int, mode: int = 0,
                     col_tiles: int = 0, longest: int = 0, singles: int = 0, silu: bool = False) -> torch.Tensor:
    """Linear attention with a fixed decay per head, as a recurrence over each segment:

        S_t = decay[h] S_(t-1) + k_t v_t^T;   o_t = S_t^T q_t

    ``vkq`` [T, H*dv | H*dk | H*dk] holds v, k, q head by head (contiguous; ``silu``: they are the SiLU of a wider projection's first
    columns, which steps of one token a segment form where they read them); ``state`` [slots, H, dk,
    dv] fp32 is read at a segment's start (zero where seg_ctx is 0) and written back at its end.
    Returns o [T, H*dv] fp32.  State, products and sums are fp32.

    GPU: bf16 prompts (a mean of 32 rows per segment and more, or a ``longest`` segment of 256 if that is given), ``dim`` a
    multiple of 32 up to 128, ``vdim`` of 16 (``mode`` 3 forces it, ``col_tiles`` 1 / 2 / 4 its value columns per workgroup, 16 / 32 / 64; 0: its choice): chunks of 64
    tokens on the matrix cores, only the state crossing chunks - fp32 scores, decays and state enter the products as three
    bf16 parts that add up to them, so only the order of the fp32 sums differs, which follows the chunk grid from the
    segment's first row on.  The first ``singles`` segments, running sequences' next tokens, stay on the scan of a decode step
    beside them.  Else the sequential scan (``ssm_scan`` with the decay
    table; ``mode`` 1 / 2 force its decode / prompt lane mapping)."""
    if silu:
        T = vkq.shape[0]
        if vkq.is_cuda and mode == 0 and T <= seg_ctx.numel():
            y = torch.empty(T, H * dv, dtype=torch.float32, device=vkq.device)
            if native().linear_step(y, vkq, decay, state, seg_cu, seg_ctx, seg_slot, int(H), int(dk), int(dv)):
                return y
        vkq = activation_cols(vkq, 0, H * (2 * dk + dv), "silu")
    return ssm_scan(vkq, None, 0, None, None, None, state, seg_cu, seg_ctx, seg_slot, H, dv, dk, H, mode, decay=decay,
                    col_tiles=col_tiles, longest=longest, singles=singles)


def decay_scan(qkv: torch.Tensor, q_col: int, k_col: int, v_col: int, z: torch.Tensor, z_bias: torch.Tensor,
               state: torch.Tensor, seg_cu: torch.Tensor, seg_ctx: torch.Tensor, seg_slot: torch.Tensor, H: int, Gk: int,
               dk: int, dv: int, q_scale: float, a_log: Optional[torch.Tensor] = None, tau: float = 1.0,
               beta: Optional[torch.Tensor] = None, beta_col: int = 0, unit: bool = False, mode: int = 0, z_col: int = 0,
               decay: Optional[str] = None, bonus: Optional[torch.Tensor] = None, longest: int = 0, singles: int = 0) -> torch.Tensor:
    """Linear attention with a decay per head and key channel (or per head), optionally with the delta rule
    or a bonus for the current token, as an fp32 recurrence over each segment.  Per head h (reading query / key head ``h // (H / Gk)``) and token:

        S <- diag(g_t) S                       g_t [dk]: this token's decays
        delta rule:   u = beta_t (v_t - S^T k_t);   S <- S + k_t u^T
        otherwise:                                  S <- S + k_t v_t^T
        o_t = S^T q_t

    or with ``bonus`` [H, dk] fp32 (the read-out sees the state before this token's decay and write):

        o_t = (S + diag(bonus) k_t v_t^T)^T q_t;   S <- diag(g_t) S + k_t v_t^T

    ``qkv`` [T, *] holds q, k ([Gk*dk] each) and v ([H*dv]) from columns ``q_col``, ``k_col``, ``v_col``
    on; q is multiplied by ``q_scale``.  ``unit``: q and k heads are first made unit vectors,
    ``x / sqrt(sum(x^2) + 1e-6)``.  The decays come from ``z`` [T, H*dk] (a projection, activation dtype)
    (columns from ``z_col`` on) and ``z_bias`` [H*dk] fp32 - or [H]: one decay per head (delta rule) -:
    ``a_log`` [H] given: ``g = exp(-exp(a_log[h]) softplus(z + z_bias))``; ``decay`` "exp_exp":
    ``g = exp(-exp(z + z_bias))``; else ``g = sigmoid(z + z_bias)^(1 / tau)``.  ``beta`` [T, *] (given = the delta rule): column
    ``beta_col + h`` holds head h's logit, ``beta_t = sigmoid(logit)``.  ``state`` [slots, H, dv, dk] fp32
    (a value row's key channels contiguous) is read at a segment's start (zero where seg_ctx is 0) and
    written back at its end.  Returns o [T, H*dv] fp32.  Decays, unit norms, gates, state, products and
    sums are fp32.

    GPU: steps of prompts (a mean segment length of 32 rows or more, or a ``longest`` segment of 256) run as two launches - everything
    that does not depend on the state (decays, unit norms, k . q, beta) for all rows at once into a
    workspace, then the recurrence over it; decode steps run as one launch, of one token a segment as a pass over the states.  bf16 prompts of the delta rule with one decay
    per head, and without the delta rule and unit norms of decays per channel (``dk`` a multiple of 32 up to 128, ``dv`` of
    16), go in chunks of 64 tokens on the matrix cores, fp32 operands as three bf16 parts that add up to them, and the first
    ``singles`` segments, running sequences' next tokens, beside them as in a decode step: their bits do not depend on what else
    is in the step.  Else token by token.  ``mode`` 1 / 2 force the one-launch / two-launch
    scan, 3 the chunks, 4 the chunks in spans where decays are per channel (tests)."""
    T = qkv.shape[0]
    nz = z_bias.numel()
    dkind = 0 if a_log is not None else 2 if decay == "exp_exp" else 1
    if not qkv.is_cuda:
        o = torch.zeros(T, H * dv, dtype=torch.float32)
        rep = H // Gk
        cul = seg_cu.tolist()
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if slot < 0 or b <= a:
                continue
            n = b - a
            q = qkv[a:b, q_col:q_col + Gk * dk].float().view(n, Gk, dk)
            k = qkv[a:b, k_col:k_col + Gk * dk].float().view(n, Gk, dk)
            v = qkv[a:b, v_col:v_col + H * dv].float().view(n, H, dv)
            if unit:
                q = q * torch.rsqrt(q.pow(2).sum(-1, keepdim=True) + 1e-6)
                k = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
            q = (q * q_scale).repeat_interleave(rep, dim=1)
            k = k.repeat_interleave(rep, dim=1)
            zz = (z[a:b, z_col:z_col + nz].float() + z_bias.float()).view(n, H, nz // H)
            if dkind == 2:
                g = torch.exp(-torch.exp(zz))
            elif a_log is not None:
                g = torch.exp(-torch.exp(a_log.float()).view(1, H, 1) * F.softplus(zz, threshold=30.0))
            else:
                g = torch.exp(F.logsigmoid(zz) / tau)
            bt = torch.sigmoid(beta[a:b, beta_col:beta_col + H].float()) if beta is not None else None
            S = state[slot].clone() if c0 > 0 else torch.zeros_like(state[slot])  # [H, dv, dk]
            for t in range(n):
                if bonus is not None:
                    kq = (k[t] * q[t] * bonus.float().view(H, dk)).sum(-1, keepdim=True)
                    o[a + t] = (torch.einsum("hpn,hn->hp", S, q[t]) + v[t] * kq).reshape(-1)
                    S = S * g[t, :, None, :] + v[t][:, :, None] * k[t, :, None, :]
                    continue
                S = S * g[t, :, None, :]
                if bt is not None:
                    u = bt[t, :, None] * (v[t] - torch.einsum("hpn,hn->hp", S, k[t]))
                else:
                    u = v[t]
                S = S + u[:, :, None] * k[t, :, None, :]
                o[a + t] = torch.einsum("hpn,hn->hp", S, q[t]).reshape(-1)
            state[slot] = S
        return o
    o = torch.empty(T, H * dv, dtype=torch.float32, device=qkv.device)
    native().decay_scan(o, qkv, int(q_col), int(k_col), int(v_col), z, z_bias, a_log, float(tau), beta, int(beta_col),
                        state, seg_cu, seg_ctx, seg_slot, int(H), int(Gk), int(dk), int(dv), float(q_scale), bool(unit), int(mode), int(z_col), dkind,
                        bonus, int(longest), int(singles))
    return o


def selective_scan(xc: torch.Tensor, q: torch.Tensor, b_col: int, c_col: int, dt: torch.Tensor, dt_bias: torch.Tensor,
                   a_log: torch.Tensor, d_skip: torch.Tensor, proj: torch.Tensor, z_col: int, state: torch.Tensor,
                   seg_cu: torch.Tensor, seg_ctx: torch.Tensor, seg_slot: torch.Tensor, longest: int = 0, mode: int = 0) -> torch.Tensor:
    """The selective state-space recurrence with a decay per channel and state, fp32, token by token within
    each segment, and its output gate.  Per channel c and state n:

        d = softplus(dt[t, c] + dt_bias[c]);   S[c, n] <- exp(-exp(a_log[c, n]) d) S[c, n] + d x_c B_n
        y_c = sum_n S[c, n] C_n + d_skip[c] x_c;   out = y_c silu(proj[t, z_col + c])

    ``xc`` [T, C] (contiguous), ``dt`` [T, C] (a projection), B and C: columns ``b_col`` / ``c_col`` .. of ``q``
    (N each); ``state`` [slots, C, N] fp32 is read at the segment's start (zero where seg_ctx is 0) and
    written back at its end.  ``longest``: rows of the longest segment (0: not known); ``mode``
    (device only): 0 whole segments (of one token each: a pass over the states) or spans of tokens side by side, by the sizes, 1 whole, 2 spans.  Returns out [T, C] in the activation dtype."""
    T, C = xc.shape
    N = a_log.shape[1]
    if not xc.is_cuda:
        out = torch.zeros(T, C, dtype=xc.dtype)
        A = -torch.exp(a_log.float())
        cul = seg_cu.tolist()
        for s, (c0, slot) in enumerate(zip(seg_ctx.tolist(), seg_slot.tolist())):
            a, b = cul[s], cul[s + 1]
            if slot < 0 or b <= a:
                continue
            S = state[slot].clone() if c0 > 0 else torch.zeros_like(state[slot])
            d = F.softplus(dt[a:b].float() + dt_bias.float(), threshold=30.0)
            x = xc[a:b].float()
            y = d_skip.float() * x
            B, Cc = q[a:b, b_col:b_col + N].float(), q[a:b, c_col:c_col + N].float()
            for t in range(b - a):
                S = torch.exp(d[t, :, None] * A) * S + (d[t] * x[t])[:, None] * B[t]
                y[t] += S @ Cc[t]
            state[slot] = S
            out[a:b] = (y * _silu(proj[a:b, z_col:z_col + C].float())).to(xc.dtype)
        return out
    out = torch.empty(T, C, dtype=xc.dtype, device=xc.device)
    native().selective_scan(out, xc, q, int(b_col), int(c_col), dt, dt_bias, a_log, d_skip, proj, int(z_col), state, seg_cu,
                            seg_ctx, seg_slot, int(longest), int(mode))
    return out


def gated_group_norm(y: torch.Tensor, proj: torch.Tensor, z_col: int, w: torch.Tensor, eps: float, groups: int,
                     out_dtype: torch.dtype, after: bool = False, gate: str = "sigmoid") -> torch.Tensor:
    """``y`` [T, n] fp32 times silu of the gate ``proj[:, z_col : z_col + n]``, then RMS-normed in
    ``groups`` equal parts (each by its own root mean square) times ``w`` [n].  ``after``: the norm
    first (of ``y`` as it is), then times ``w`` and the SIGMOID of the gate (``gate`` "silu": its SiLU)."""
    T, n = y.shape
    if not y.is_cuda:
        if after:
            g = y.view(T, groups, n // groups)
            g = g * torch.rsqrt(g.pow(2).mean(-1, keepdim=True) + eps)
            z = proj[:, z_col:z_col + n].float()
            return (g.reshape(T, n) * w.float() * (torch.sigmoid(z) if gate == "sigmoid" else _silu(z))).to(out_dtype)
        g = y * _silu(proj[:, z_col:z_col + n].float())
        g = g.view(T, groups, n // groups)
        g = g * torch.rsqrt(g.pow(2).mean(-1, keepdim=True) + eps)
        return (g.reshape(T, n) * w.float()).to(out_dtype)
    out = torch.empty(T, n, dtype=out_dtype, device=y.device)
    native().gated_group_norm(out, y, proj, int(z_col), w, float(eps), int(groups), (2 if gate == "silu" else 1) if after else 0)
    return out


# ---------------------------------------------------------------- routed experts

def moe_router(h: torch.Tensor, wr: torch.Tensor, bias: Optional[torch.Tensor], E: int, K: int,
               over_all: bool = False) -> tuple:
    """fp32 router: logits = ``wr[:E] h + bias[:E]`` (``bias`` None: none), the ``K`` largest are
    chosen and weighted by the softmax over the chosen logits only - or, ``over_all``, by their
    probabilities in the softmax over all E logits, as they are.  ``wr`` may hold one more row (E + 1 in all): then
    ``gate = sigmoid(wr[E] h)`` per token is returned too (the shared expert's gate).
    Returns (ids [T, K] int32, weights [T, K] fp32, gate [T] fp32 or None)."""
    T = h.shape[0]
    has_gate = wr.shape[0] == E + 1
    if not h.is_cuda:
        lg = h.float() @ wr.float().t()
        gate = torch.sigmoid(lg[:, E]) if has_gate else None
        z = lg[:, :E] + bias.float()[:E] if bias is not None else lg[:, :E]
        top, idx = torch.topk(z, K, dim=-1)
        if over_all:
            return idx.to(torch.int32), torch.softmax(z, -1).gather(1, idx), gate
        return idx.to(torch.int32), torch.softmax(top, -1), gate
    ids = torch.empty(T, K, dtype=torch.int32, device=h.device)
    wts = torch.empty(T, K, dtype=torch.float32, device=h.device)
    gate = torch.empty(T, dtype=torch.float32, device=h.device) if has_gate else None
    native().moe_router(ids, wts, gate, h, wr, bias, E, K, bool(over_all))
    return ids, wts, gate


def moe_router_grouped(h: torch.Tensor, wr: torch.Tensor, E: int, K: int, groups: int, keep: int, scale: float,
                       soft: bool = False, corr: Optional[torch.Tensor] = None, best2: bool = True,
                       renorm: bool = True) -> tuple:
    """fp32 router whose choice is restricted to groups.  Scores ``s = sigmoid(wr h)``, or with ``soft`` the
    softmax over all E logits; choice scores ``s + corr`` (``corr`` [E] fp32, None: zeros - they may be
    negative).  The E experts form ``groups`` equal groups of neighbours; a group counts as the sum of its two
    largest choice scores (its one where a group is one expert), or without ``best2`` as its largest; only
    experts of the ``keep`` best groups can be chosen.  The ``K`` largest choice scores among those are taken
    (lowest index wins a tie) and weighted ``s / (sum of the chosen s + 1e-20) * scale``, or without
    ``renorm`` ``s * scale``.  Returns (ids [T, K] int32, weights [T, K] fp32)."""
    T = h.shape[0]
    if not h.is_cuda:
        lg = h.float() @ wr.float().t()
        sc = torch.softmax(lg, -1) if soft else torch.sigmoid(lg)
        choice = sc if corr is None else sc + corr.float()
        if groups > 1:
            per = E // groups
            gs = choice.view(T, groups, per).topk(min(2, per) if best2 else 1, dim=-1).values.sum(-1)
            best = gs.topk(keep, dim=-1).indices
            ok = torch.zeros(T, groups, dtype=torch.bool).scatter_(1, best, True)
            choice = torch.where(ok.repeat_interleave(per, dim=1), choice, torch.full_like(sc, -math.inf))
        idx = choice.topk(K, dim=-1).indices
        w = sc.gather(1, idx)
        return idx.to(torch.int32), (w / (w.sum(-1, keepdim=True) + 1e-20) if renorm else w) * scale
    ids = torch.empty(T, K, dtype=torch.int32, device=h.device)
    wts = torch.empty(T, K, dtype=torch.float32, device=h.device)
    native().moe_router_grouped(ids, wts, h, wr, corr, int(E), int(K), int(groups), int(keep), float(scale), bool(soft), bool(best2),
                                bool(renorm))
    return ids, wts


# expert-sorted rows from which the routed GEMMs of an interleaved (``il``) layer go to the
# framework's 256 x 256 prefill tile kernel (ops.moe_grouped_gemm) instead of the 16-row kernel
TILE_MIN_ROWS = 1024


def moe_experts(h: torch.Tensor, ids: torch.Tensor, wts: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor,
                shared: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None, il: bool = False,
                mfma: bool = True, act: str = "swiglu", limit: float = 0.0, tile: bool = False,
                identity: int = 0, join: bool = False):
    """Sum over each token's chosen experts of ``wts * down_e(silu(gate_e h) * up_e h)`` with
    ``w13`` [E, 2*ff, d] (gate rows then up rows; ``il``: interleaved per 128 rows as [64 gate |
    64 up], ops.interleave_gate_up) and ``w2`` [E, d, ff], plus ``gate * shared`` (the shared
    expert's output [T, d] and its per-token gate; ``gate`` None: 1).  ``act`` "gelu": ungated
    experts ``down_e(gelu(up_e h))`` with ``w13`` [E, ff, d]; "relu_sq": the same with the squared ReLU.
    ``identity``: ids E .. E + identity - 1 are experts whose output is h itself.  ``act`` "clamped_swish": gated experts whose
    unit is ``g * sigmoid(1.702 g) * (u + 1)`` with g = min(gate_e h, limit), u = clamp(up_e h, -limit,
    limit).  fp32 [T, d]; ``join``: on the GPU, where add_norm can form the sum, an ExpertSum.

    GPU: the (token, slot) pairs are counting-sorted by expert on the device and both projections
    run as ONE grouped launch each over the sorted rows (SwiGLU in the first epilogue); no host
    synchronisation.  bf16: matrix-core kernels - tiles of 16, 32 or 64 rows by the mean rows of an expert, gathered on load
    (decode, small steps), or from TILE_MIN_ROWS sorted rows of an ``il`` layer the prefill tile
    GEMM of the Mixtral path, which reads the rows in sorted order from where they are (ungated experts whose widths are multiples of 256 take it too, with
    the GELU as a launch between); fp32: three-part operands on the bf16 matrix instruction (experts_f32.hip).  K that is no multiple of 32
    and unaligned fp32 rows: 64 x 64 tiles on the vector unit."""
    T, d = h.shape
    E, K = w13.shape[0], ids.shape[1]
    ff = w2.shape[2]
    if not h.is_cuda:
        out = torch.zeros(T, d, dtype=torch.float32)
        hf = h.float()
        for e in range(E):
            rows, slot = torch.nonzero(ids == e, as_tuple=True)
            if rows.numel():
                we = w13[e].float()
                if il:
                    we = we.view(ff // 64, 2, 64, d).permute(1, 0, 2, 3).reshape(2 * ff, d)
                gu = (hf[rows] @ we.t()).to(h.dtype).float()
                if act in ("gelu", "relu_sq"):
                    a = _act_torch(gu, act).to(h.dtype).float()
                elif act == "clamped_swish":
                    a = _clamped_unit(gu[:, :ff], gu[:, ff:], limit).to(h.dtype).float()
                else:
                    a = (_silu(gu[:, :ff]) * gu[:, ff:]).to(h.dtype).float()
                out.index_add_(0, rows, (a @ w2[e].float().t()).to(h.dtype).float() * wts[rows, slot].unsqueeze(-1))
        if identity:
            out += hf * (wts * (ids >= E)).sum(-1, keepdim=True)
        if shared is not None:
            out += shared.float() * gate.unsqueeze(-1) if gate is not None else shared.float()
        return out
    ext = native()
    n = T * K
    # identity experts sort behind the others: the GEMMs run over the first E experts' rows only
    offsets = torch.empty(E + identity + 1, dtype=torch.int32, device=h.device)
    sorted_idx = torch.empty(n, dtype=torch.int32, device=h.device)
    inv_idx = torch.empty(n, dtype=torch.int32, device=h.device)
    ext.moe_align(ids, E + identity, offsets, sorted_idx, inv_idx)
    offsets = offsets[:E + 1]
    code = {"swiglu": 1, "gelu": 2, "clamped_swish": 3, "relu_sq": 4}[act]
    if act in ("gelu", "relu_sq") and n >= TILE_MIN_ROWS and h.dtype == torch.bfloat16 and ff % 256 == 0 and d % 256 == 0:
        from .. import ops  # large steps of plain experts: the prefill tile GEMM twice, the activation between

        a = activation(ops.moe_grouped_gemm(h, w13, offsets, zero_fill=False, rows=sorted_idx, div=K), act)
        ys = ops.moe_grouped_gemm(a, w2, offsets, zero_fill=False)
    elif act == "clamped_swish" and tile and n >= TILE_MIN_ROWS and h.dtype == torch.bfloat16:
        from .. import ops  # large steps: the prefill tile GEMM twice, the clamped unit as a launch between

        a = glu(ops.moe_grouped_gemm(h, w13, offsets, zero_fill=False, rows=sorted_idx, div=K), 0, ff, "clamped_swish", limit)
        ys = ops.moe_grouped_gemm(a, w2, offsets, zero_fill=False)
    elif il and n >= TILE_MIN_ROWS and h.dtype == torch.bfloat16:
        from .. import ops  # the Mixtral path's kernels (_k8sllm_ops)

        a = ops.moe_grouped_gemm(h, w13, offsets, swiglu=True, zero_fill=False, rows=sorted_idx, div=K)
        ys = ops.moe_grouped_gemm(a, w2, offsets, zero_fill=False)
    else:
        a = torch.empty(n, ff, dtype=h.dtype, device=h.device)
        ext.grouped_gemm(a, h, w13, offsets, sorted_idx, K, code, il, mfma, float(limit))
        ys = torch.empty(n, d, dtype=h.dtype, device=h.device)
        ext.grouped_gemm(ys, a, w2, offsets, None, 1, 0, False, mfma, 0.0)
    if join and not identity and d % 8 == 0:
        return ExpertSum(ys, inv_idx, wts, shared, gate)
    out = torch.empty(T, d, dtype=torch.float32, device=h.device)
    ext.moe_combine(out, ys, inv_idx, wts, shared, gate, ids if identity else None, h if identity else None, E)
    return out


def _rows_form(M: int, N: int, K: int, end: str = "") -> Optional[str]:
    """Which kernel of few_rows.hip takes a bf16 product of M rows with weights [N, K]; ``end``: what stands behind it and would be a launch
    of its own, a gated unit of its first rows ("glu") or something elementwise ("act").  None: the BLAS library.  us, library (and launch)
    / own / shared, in a graph over weights from memory:
    plain     up to 16 rows: 2048 x 2048, 1 row 8.5 / 4.0 / 7.4; 4096 x 4096, 16 rows 16.4 / 8.3 / 14.6; 7168 x 4096, 16 rows 16.3 / 13.7 / 16.5;
              16384 x 1024, 4 rows 10.3 / 9.9 / 8.4; 16384 x 4096, 8 rows 34.7 / 24.8 / 29.2; 128256 x 4096, 4 rows 193 / 164 / 180; 4096 x
              11008, 4 rows 39 / 18.7 / 35; 8192 x 16384, 16 rows 62 / 56 / 63
              up to 32: 4096 x 4096 14.0 / 9.2 / 15.9; 8192 x 2048 14.4 / 10.4 / 11.1; 11312 x 4096 23.2 / 26.1 / 21.0; 32768 x 4096 69.7 / 68 /
              52.4; 4096 x 11008 32 / 25.6 / 41; 6144 x 5632 20.4 / 23.5 / 23.7
              up to 64: 4096 x 2048 12.3 / 8.2 / 12; 10240 x 4096 29.4 / 31 / 24.7; 16384 x 2048 19.7 / 26 / 19.3; 24576 x 2048 28 / 37 / 31; 32768
              x 4096 66 / 90 / 58; 6144 x 4096 18.7 / 23 / 21.8; of few k and many columns 28672 x 256, 48 rows 10.8 / 13.1 / 9.1; 37632 x 256 11.8 /
              17.1 / 13.8; 54944 x 2496, 56 rows 52 / 91 / 69
    act       8192 x 4096, 64 rows 26.1 / 24.8 / 25.3; 32768 x 2048, 64 rows 50 / 51 / 39; 24576 x 5632, 64 rows 74 / 110 / 70
    glu       (a workgroup of either takes half as many columns) 8192 x 2048, 64 rows 17 / 13 / 19; 16384 x 4096, 16 rows 37 / 27 / 36, 32 rows
              37 / 30 / 35; 24576 x 4096, 24 rows 52 / 41 / 43, 64 rows 53 / 58 / 46; 32768 x 4096, 8 rows 66 / 47 / 60, 16384 x 2048, 24 rows
              20 / 17 / 20; 32768 x 1024, 4 rows 20 / 18 / 14; of few k 29952 x 64, 16 rows 8.7 / 9.2 / 4.8; 13248 x 256, 48 rows 11.1 / 8.5 / 7.8;
              23824 x 160, 48 rows 16 / 10.4 / 8.0
    Over 7000 products of 1 to 64 rows, 256 to 60000 columns and 64 to 16384 k from memory a call takes 1.07 times the least of the three in the
    mean, a unit 1.08."""
    if M > 64 or K > 16384 or (N * K > 1 << 28 and (M > 4 or end == "glu")):
        return None
    if end == "glu":
        if K > 4096:
            return None
        if N >= 24576 and (K <= 1024 or M > 8):
            return "shared"
        if M > 16 and N > 8192 and K <= 1024:
            return "shared" if N > 16384 or (M <= 32 and K <= 512) else "own"
        return "own" if M <= 16 or (M <= 32 and K > 2048) or N <= 8192 and (M <= 32 or K <= 2048) or (M <= 24 and N <= 16384) else None
    if K > 6144:  # whole lines for each of a workgroup's waves
        return "own" if K % 256 == 0 and (M <= 8 or (M <= 16 and N <= 4096) or (M <= 32 and 2048 < N <= 4096)) else None
    if K > 4096:
        if M <= 2 or (M <= 4 and (end or N <= 4096 or 8192 <= N <= 32768)) or (M <= 32 and 2048 <= N <= 4096):
            return "own"
        return "shared" if N >= 10240 and (M <= 16 or (end and (M <= 32 or N <= 45056))) else None
    if M <= 8:
        return "shared" if N >= 131072 or (N >= 10240 and K <= 1024) else "own"
    if M <= 16:
        return "own" if N * K < 1 << 25 and (N < 10240 or K > 1024) else "shared" if N >= 10240 else None
    if M <= 32:
        if N * K <= 1 << 24 and N <= 8192:
            return "own"
        return "shared" if N >= 10240 or (N >= 8192 and K <= 3072) else None
    if N > 16384 and K <= 512:
        return "shared" if end or N <= (45056 if K > 256 else 32768) else None
    if N * K <= 1 << 23 or (N * K < 1 << 24 and K <= 2048):
        return "own"
    if N > 32768 and not (end and (N <= 45056 or K <= 2048)):
        return None
    return "shared" if 10240 <= N <= 16384 or (N >= 28672 and (end or K >= 2048)) or (end and 8192 <= N < 10240 and K <= 3072) else None


def _few_rows(x: torch.Tensor, w: torch.Tensor, end: str = "") -> Optional[str]:
    if x.shape[0] > 64:  # (_rows_form has none; before the other checks, 1.5 us a product of a prompt step)
        return None
    if torch.is_grad_enabled() and (x.requires_grad or w.requires_grad):  # the library's product has a backward
        return None
    if not (x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2
            and w.shape[1] % 32 == 0 and w.shape[1] >= 32 and x.shape[0] > 0
            and w.is_contiguous() and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0):
        return None
    return _rows_form(x.shape[0], w.shape[0], w.shape[1], end)


def _tile_plain(M: int, N: int, K: int) -> bool:
    """Whether the tile GEMM takes a large product with nothing behind it: where N is no multiple of its 256 columns and K small, the BLAS
    library's kernels fall to 350 (K up to 512), 600 (1024) and 800 TFLOP/s (2048, N below 4096), and the tile GEMM's rounds of 256 tiles, estimated
    here, take less than that.  us, library / tile GEMM: 6403 x 5648 x 1024 127 / 82, 4800 rows 100 / 55; 7830 x 3104 x 2048 131 / 86; 8000 x 1568 x 1024 41 /
    29.  Over 404 products of 1024 to 9000 rows, 1024 to 12000 columns and 256 to 2048 k (N no multiple of 256) the 107 that it takes are 1.36 times faster in the
    mean, the worst 1.10.  The estimate is of 256-row tiles and slower strips than the kernel has: of the 297 that it leaves 174 would be faster too,
    100 slower.  (Multiples of 256 were measured with that kernel: as many would lose as win.)"""
    if M < 1024 or not 1024 <= N < 1 << 19 or N % 256 == 0 or N % 16 or K % 64 or not 192 <= K <= 2048 or (K > 1024 and N >= 4096):
        return False  # (the tile GEMM's offsets into the weights are 31 bits)
    rounds, over = divmod(-(-M // 256) * -(-N // 256), 256)
    last = 0.0 if over == 0 else (0.62 if rounds else 0.85) if over <= 64 else 0.82 + 0.18 * over / 256  # strips, or a round that is not full
    us = (rounds + last) * (9 + 1.45 * K / 64)
    return us * (350 if K <= 512 else 600 if K <= 1024 else 800) < 2e-6 * M * N * K


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x`` [T, K] times ``w`` [N, K] transposed.  The BLAS library's product, but for bf16 on the device with rows 16-byte aligned: the
    few rows of a decode step, K a multiple of 32, where a call takes what it takes to get enough loads in flight
    (few_rows.hip, by the rule of ``_rows_form``), and large products by the rule of ``_tile_plain``."""
    if isinstance(x, GatedRows):
        made = x.product(w)
        if made is not None:
            return made[1]
        x = x.tensor()
    M = x.shape[0]
    if M <= 64:  # (rows between the two rules are a prompt's whose step the host's time bounds: they meet no other check)
        form = _few_rows(x, w)
        if form is not None:
            y = torch.empty(M, w.shape[0], dtype=x.dtype, device=x.device)
            native().few_rows(y, None, x, w, -1, 0.0, form == "shared")
            return y
    elif M >= 1024 and w.dim() == 2 and _tile_plain(M, w.shape[0], w.shape[1]) and _tile_operands(x, w) and not (
            torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)):
        from .. import ops

        y = torch.empty(M, w.shape[0], dtype=x.dtype, device=x.device)
        ops.native().gemm_tile(y, x, w, None, 0, 1)
        return y
    return F.linear(x, w)


TILE_UNITS = {"gelu_tanh": 5, "silu": 6, "relu": 7, "relu_sq": 8}  # epilogues of ops.gemm_tile_unit
GLU_ENDS = ("gelu_tanh", "silu", "relu")  # gated units that the projections' kernels have at their end; ``glu`` has others


def _tile_form(M: int, N: int, K: int, f: int) -> bool:
    """Whether the tile GEMM takes a large product with a unit at its end (a gated one of f features, or f 0), which the BLAS library leaves a
    launch of its own that reads and writes the products once more.  us, library and launch / tile GEMM: 7830 rows, 2 x 5632 + 2048 columns, K
    2048 377 + 54 / 339; 3749 rows 225 + 23 / 168; 6403 x 4096 x 1024 (1.6 rounds of tiles) 49 + 17 / 53.  At least four fifths of the tiles' area
    must be products: 53248 columns, K 2048 1 row 52 / 57, 128 rows 61 / 59, 300 rows (two row tiles) 89 / 91, 256 rows 70 / 62, 1300 rows
    (six) 308 / 235.  Rounds are counted in tiles of 256 rows without strips, as the kernel was when the rule was made; it leaves the library some
    products that would be faster now: 4300 x 4096 x 1024 55 / 46, 2500 x 8192 x 1024 63 / 50, 2700 x 4096 x 1024 34 / 28."""
    tiles = -(-M // 256) * (-(-f // 128) + -(-(N - 2 * f) // 256))
    return (tiles >= 200 and tiles >= 0.7 * 256 * -(-tiles // 256) and M * N >= 0.8 * 256 * 256 * tiles
            and K % 64 == 0 and K >= 192 and N % 16 == 0 and f % 16 == 0 and 2 * f <= N and max(N, 256) * max(K, 256) * 2 < 1 << 31
            and 256 * N * 2 < 1 << 31)


def _transformed(*ts: torch.Tensor) -> bool:
    """Whether something beside the values hangs on a product that only torch's own carries on: a tangent, a function transform (vmap, jvp), a trace."""
    return (torch._C._are_functorch_transforms_active() or torch.jit.is_tracing()
            or any(torch.autograd.forward_ad.unpack_dual(t).tangent is not None for t in ts))


def _tile_operands(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2 and w.dim() == 2 and x.is_contiguous()
            and w.is_contiguous() and not _transformed(x, w) and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def _tile_unit(x: torch.Tensor, w: torch.Tensor, f: int) -> bool:
    """Whether ``gemm_tile_unit`` takes these operands, by the rule of ``_tile_form`` (which takes no fewer rows than 0.8 of a tile's)."""
    M = x.shape[0]
    return M > 204 and w.dim() == 2 and _tile_form(M, w.shape[0], w.shape[1], f) and _tile_operands(x, w)


def linear_act(x: torch.Tensor, w: torch.Tensor, kind: str) -> torch.Tensor:
    """``activation(linear(x, w), kind)``, in one launch for the rows that few_rows.hip takes (``relu_sq`` and ``tanh``) and for large
    steps (``relu_sq``, by the rule of ``_tile_form``)."""
    if kind == "relu_sq" and _tile_unit(x, w, 0):
        from .. import ops

        y = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
        ops.native().gemm_tile_unit(y, None, x, w, TILE_UNITS[kind])
        return y
    form = _few_rows(x, w, "act") if kind in ("relu_sq", "tanh") else None
    if form is not None:
        y = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
        native().few_rows(y, None, x, w, 16 + ACTS[kind], 0.0, form == "shared")
        return y
    return activation(linear(x, w), kind)


def linear_glu(x: torch.Tensor, w: torch.Tensor, f: int, kind: str) -> tuple:
    """The gated unit ``act(gate x) * (up x)`` [T, f] of ``w``'s rows [f gate | f up | the rest], and a projection with the column
    at which the rest's outputs begin in it.  ``linear`` and ``glu``, in one launch for the rows that few_rows.hip takes and for large
    steps (by the rule of ``_tile_form``)."""
    if isinstance(x, GatedRows):
        made = x.product(w, f, kind) if f > 0 and f % 16 == 0 and kind in GLU_ENDS else None
        if made is not None:
            return (*made, 0)
        x = x.tensor()
    if f > 0 and kind in GLU_ENDS and _tile_unit(x, w, f):
        from .. import ops

        a = torch.empty(x.shape[0], f, dtype=x.dtype, device=x.device)
        y = torch.empty(x.shape[0], w.shape[0] - 2 * f, dtype=x.dtype, device=x.device)
        ops.native().gemm_tile_unit(a, y, x, w, TILE_UNITS[kind])
        return a, y, 0
    form = _few_rows(x, w, "glu") if f > 0 and f % 16 == 0 and kind in GLU_ENDS else None
    if form is not None:
        a = torch.empty(x.shape[0], f, dtype=x.dtype, device=x.device)
        y = torch.empty(x.shape[0], w.shape[0] - 2 * f, dtype=x.dtype, device=x.device)
        native().few_rows(y, a, x, w, ACTS[kind], 0.0, form == "shared")
        return a, y, 0
    proj = linear(x, w)
    return glu(proj, 0, f, kind), proj, 2 * f


def logits(x: torch.Tensor, w: torch.Tensor, scale: float = 1.0, cap: float = 0.0) -> torch.Tensor:
    """fp32 ``scale * (x w^T)`` of the product rounded to x's dtype, through ``cap * tanh(. / cap)`` if cap > 0.  In one launch for the
    few rows of a decode step (no scale)."""
    form = _few_rows(x, w, "act") if scale == 1.0 else None
    if form is not None:
        z = torch.empty(x.shape[0], w.shape[0], dtype=torch.float32, device=x.device)
        native().few_rows(z, None, x, w, -1, float(cap), form == "shared")
        return z
    z = F.linear(x, w).float()
    if scale != 1.0:
        z = z * scale
    return softcap(z.contiguous(), cap) if cap > 0 else z


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(gu[:, :f]) * gu[:, f:] for [T, 2f] rows ([gate | up])."""
    f = gu.shape[1] // 2
    if not gu.is_cuda:
        return (_silu(gu[:, :f].float()) * gu[:, f:].float()).to(gu.dtype)
    out = torch.empty(gu.shape[0], f, dtype=gu.dtype, device=gu.device)
    native().swiglu(out, gu)
    return out
