"""What a user of this framework has it do on the GPU, as cases that can be timed and compared.

A case is ONE step of a served model through ``ModelRunner``, as the engine drives it: a prefill step over
whole prompts, a step that goes on with prompts whose first part is cached, a mixed step (running sequences'
next tokens beside prompt portions) or a decode step replayed from its hipGraph.  The models are Llama-3-8B (the
headline of bench.py) and three of the layer-list designs at the sizes of ``bench.py --mode arch``, which between
them run every family of mixers: Dunesun (windowed attention with a sink, Mamba-2, routed experts), Bitonex
(rotary attention over the whole prefix, linear attention, latent attention, gated dense layers) and Dopivik
(selective scan, wkv time mixing, chunked capped attention beside the delta rule).

The keys of a case: ``model``; ``width`` (layer-list designs: 1024, 2048 or 4096); ``dtype``; ``decode`` running
sequences with about ``decode_context`` tokens each, of which this step takes one more; ``prompts`` prompts of
which this step takes about ``tokens`` tokens each behind ``context`` cached ones; ``ragged``: by what part of
its length the shortest sequence is shorter than the longest.  Weights, token ids and everything that is in
the caches come from the seed.

``run`` returns the step's logits and the caches and states that it wrote.  The sampled tokens are left out: with
random weights two of 128256 logits are often closer than bf16 results of two correct programs.
"""
from __future__ import annotations

import hashlib
import math

import torch
import torch.nn.functional as F

from k8s_llm_monitor_amd.engine.block_manager import BlockManager
from k8s_llm_monitor_amd.engine.runner import ModelRunner, RunnerConfig
from k8s_llm_monitor_amd.engine.sequence import SamplingParams, Sequence
from k8s_llm_monitor_amd.models import HybridLM, build_model, get_config
from k8s_llm_monitor_amd.models.config import DenseSpec, HybridConfig, LayerSpec, MoESpec

LLAMA = "llama-3-8b"
DESIGNS = ("dunesun", "bitonex", "dopivik")
MAX_POSITION = 8192  # of Llama-3-8B and of the bench's layer-list models
VOCAB = 32000  # of the layer-list models
WINDOW = 1024  # Dunesun's sliding window, Dopivik's chunk
CAP = 50.0  # Dopivik's cap on attention scores


def _case(name, model, width=0, dtype="bfloat16", decode=0, decode_context=0, prompts=0, tokens=0, context=0, ragged=0.0):
    c = dict(model=model, width=width, dtype=dtype, decode=decode, decode_context=decode_context, prompts=prompts,
             tokens=tokens, context=context, ragged=ragged)
    return dict(c, name=name) if name else c


def listed() -> list:
    return [
        # one operator asking: the next token of one answer, 1.7 k tokens into it
        _case("llama-decode-1", LLAMA, decode=1, decode_context=1700),
        # the headline wave's decode step: 64 diagnostic queries at once
        _case("llama-decode-64", LLAMA, decode=64, decode_context=1900, ragged=0.2),
        # the headline wave's prefill step: as many ~1.6 k token prompts as the 16 k token budget takes
        _case("llama-prefill", LLAMA, prompts=10, tokens=1636, ragged=0.05),
        # the arch bench's prefill step: 4 prompts of 2048 tokens
        _case("dunesun-prefill", "dunesun", 2048, prompts=4, tokens=2048),
        # the arch bench's decode step
        _case("dunesun-decode-64", "dunesun", 2048, decode=64, decode_context=2048),
        # a step of a replayed trace in true fp32: a few prompts beside running sequences
        _case("dunesun-mixed-fp32", "dunesun", 1024, "float32", decode=5, decode_context=211, prompts=3, tokens=331, ragged=0.4),
        # prompts of a wave, all in one step, none of a round length
        _case("bitonex-prefill", "bitonex", 2048, prompts=5, tokens=1637, ragged=0.1),
        # chunked prefill under load: two long prompts go on beside the running answers
        _case("bitonex-mixed", "bitonex", 2048, decode=32, decode_context=1500, prompts=2, tokens=2048, context=2816, ragged=0.3),
        # the smallest step: one short conversation
        _case("bitonex-decode-1", "bitonex", 1024, decode=1, decode_context=333),
        # one long document
        _case("dopivik-prefill-long", "dopivik", 2048, prompts=1, tokens=8000),
        # many short prompts of very different lengths
        _case("dopivik-prefill-ragged", "dopivik", 1024, prompts=13, tokens=901, ragged=0.95),
        # a half-full decode batch of the widest size
        _case("dopivik-decode-24", "dopivik", 4096, decode=24, decode_context=1777, ragged=0.5),
    ]


def draw(rng) -> dict:
    """A step of the same models and ranges: 1 to 64 running sequences, 1 to 16 prompts, up to 16 k new tokens a step
    (Llama) or 8 k (layer-list designs), up to 4 k tokens in the caches of a sequence."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice((LLAMA,) + DESIGNS)
    llama = model == LLAMA
    width = 0 if llama else rng.choice((1024, 2048, 4096))
    kind = rng.choice(("prefill", "prefill", "portion", "mixed", "decode", "decode"))
    ragged = round(rng.choice((0.0, rng.uniform(0.0, 0.9))), 3)
    dtype = "bfloat16"
    if not llama and rng.random() < 0.15:  # fp32 is for replays: smaller steps
        dtype, width = "float32", 1024
    small = dtype == "float32"
    c = dict(decode=0, decode_context=0, prompts=0, tokens=0, context=0)
    if kind in ("decode", "mixed"):
        c["decode"] = spread(1, 64 if kind == "decode" else 32)
        c["decode_context"] = spread(16, 500 if small else 2000)
    if kind != "decode":
        c["prompts"] = spread(1, 16)
        rows = spread(64, 1500 if small else 16000 if llama and kind == "prefill" else 8000)
        c["context"] = 0 if kind == "prefill" else spread(16, 500 if small else 4000)
        c["tokens"] = max(1, min(MAX_POSITION - c["context"] - 32, rows // c["prompts"]))
    return _case(None, model, width, dtype, ragged=ragged, **c)


# ---------------------------------------------------------------------------------------------------- models
def _lengths(longest: int, ragged: float, n: int) -> list:
    """``n`` lengths spread over [longest * (1 - ragged), longest], the same for every seed."""
    return [max(1, longest - int(longest * ragged * ((i * 0.6180339887498949) % 1.0))) for i in range(n)]


def _rows(case: dict) -> tuple:
    """(cached tokens, new tokens) of every sequence of the step: running sequences first."""
    dec = [(n, 1) for n in _lengths(case["decode_context"], case["ragged"], case["decode"])]
    return dec + [(case["context"], n) for n in _lengths(case["tokens"], case["ragged"], case["prompts"])]


def _flat(m: dict) -> tuple:
    return tuple(sorted(m.items()))


def _experts(width: int) -> tuple:
    return 8, 2, {1024: 1024, 2048: 2048, 4096: 3584}[width]


def _config(model: str, width: int) -> HybridConfig:
    d, H, G, D = width, width // 128, width // 512, 128
    wide = width == 4096
    scale = D ** -0.5
    rest = {}
    if model == "dunesun":
        moe = MoESpec(*_experts(width), 0)
        att = LayerSpec("attention", _flat({"heads": H, "kv_heads": G, "dim": D, "vdim": D, "mask.size": WINDOW, "scale": scale}), moe)
        ssm = LayerSpec("mamba2", _flat({"heads": 2 * d // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}),
                        moe)
        layers = [att if i % 2 == 0 else ssm for i in range(2 if wide else 4)]
    elif model == "bitonex":
        ff = DenseSpec({1024: 2816, 2048: 5632, 4096: 11008}[width])
        layers = []
        for i in range(3 if wide else 6):
            if i % 3 == 0:
                layers.append(LayerSpec("attention", _flat({"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": scale,
                                                            "rot.dims": 64, "rot.base": 1e6}), ff))
            elif i % 3 == 1:
                decay = tuple(1.0 - 2.0 ** (-3 - 5 * h / max(1, H - 1)) for h in range(H))
                layers.append(LayerSpec("lightning", _flat({"heads": H, "dim": D, "vdim": D, "decay": decay}), ff))
            else:
                m = {"heads": H, "dim": 96, "rot_dim": 32, "vdim": D, "q_rank": 3 * d // 8, "kv_rank": 128 if d == 1024 else 256,
                     "scale": scale, "rot.base": 1e4, "rot.dims": 32}
                layers.append(LayerSpec("latent_attention", _flat(m if i == 2 else dict(m, kv_from=2)), ff))
        rest = dict(norm_eps=1e-6, residual_mult=0.5, logit_softcap=30.0)
    else:
        ff = DenseSpec(4 * d)
        layers = []
        for i in range(3 if wide else 6):
            if i % 3 == 0:
                layers.append(LayerSpec("mamba1", _flat({"inner": 2 * d, "state": 16, "conv": 4, "dt_rank": d // 16}), ff))
            elif i % 3 == 1:
                layers.append(LayerSpec("wkv", _flat({"heads": d // 64, "dim": 64, "w_rank": d // 32}), ff))
            else:
                left = {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": scale, "softcap": CAP, "mask.size": WINDOW,
                        "rot.dims": 64, "rot.base": 5e5}
                right = {"heads": H, "kv_heads": H // 2, "dim": D, "vdim": D, "conv": 4}
                layers.append(LayerSpec("parallel", _flat({**{"left." + k: v for k, v in left.items()},
                                                           **{"right." + k: v for k, v in right.items()}}), ff))
        rest = dict(norm_eps=1e-5, embed_scale=float(d) ** 0.5)
    return HybridConfig(name=f"{model}-d{d}", arch=model, vocab_size=VOCAB, d_model=d, layers=tuple(layers),
                        max_position=MAX_POSITION, **rest)


def _spec(cfg: HybridConfig) -> dict:
    """Checkpoint name -> (shape, standard deviation, mean) of every tensor.  Matrices keep a unit-variance input's
    variance, what leads back to the residual stream a quarter of it, as in trained models the stream is
    larger than what one sublayer adds."""
    d = cfg.d_model
    out = {"embed": ((VOCAB, d), 1.0 / cfg.embed_scale, 0.0), "head": ((VOCAB, d), d ** -0.5, 0.0)}

    def mat(name, n, k, gain=1.0):
        out[name] = ((n, k), gain * k ** -0.5, 0.0)

    def vec(name, shape, std=0.1, mean=1.0):
        out[name] = (shape if isinstance(shape, tuple) else (shape,), std, mean)

    def norm(name):
        if cfg.arch == "bitonex":
            vec(name, ())
        elif cfg.arch == "dunesun":
            vec(name, d, 0.1, 0.0)
        else:
            vec(name, d)
            vec(name + ".b", d, 0.1, 0.0)

    norm("final.norm")
    if cfg.arch == "dunesun":
        out["pos"] = ((cfg.max_position, d), 0.1, 0.0)
    for i, s in enumerate(cfg.layers):
        L, p, m = f"l{i}.", f"l{i}.mix.", s.m
        norm(L + "norm1")
        if cfg.arch == "dunesun" and s.kind == "attention":
            for k, n in (("q", m["heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"])):
                mat(p + k, n, d)
                vec(p + k + ".norm", n, 0.2, 1.0)
            mat(p + "v", m["kv_heads"] * m["vdim"], d)
            mat(p + "o", d, m["heads"] * m["vdim"], 0.5)
        elif s.kind == "mamba2":
            inner = m["heads"] * m["vdim"]
            C = inner + 2 * m["groups"] * m["state"]
            mat(p + "in", inner + C + m["heads"], d)
            vec(p + "conv", (C, m["conv"]), 0.5, 0.0)
            vec(p + "conv.b", C, 0.1, 0.0)
            vec(p + "dt_bias", m["heads"], 1.0, -3.5)  # steps of 0.005 to 0.1 ...
            vec(p + "A_log", m["heads"], 0.7, 1.0)  # ... and decays of a few tokens to a few hundred
            vec(p + "D", m["heads"], 0.3, 1.0)
            vec(p + "norm", inner)
            mat(p + "o", d, inner, 0.5)
        elif cfg.arch == "bitonex":
            if s.kind == "attention":
                nq, nk = m["heads"] * m["dim"], m["kv_heads"] * m["dim"]
                for k, n in (("q", nq), ("k", nk), ("v", nk), ("g", nq)):
                    mat(p + k, n, d)
                vec(p + "temp", m["heads"], 0.2, 1.0)
                mat(p + "o", d, nq, 0.5)
            elif s.kind == "lightning":
                n = m["heads"] * m["dim"]
                for k in "vkqg":
                    mat(p + k, n, d)
                vec(p + "norm", n)
                mat(p + "o", d, n, 0.5)
            else:
                H, dn, dr, dv, Q, R = (m[k] for k in ("heads", "dim", "rot_dim", "vdim", "q_rank", "kv_rank"))
                mat(p + "dq", Q, d)
                vec(p + "dq.norm", Q)
                if "kv_from" not in m:
                    mat(p + "dkv", R + dr, d)
                    vec(p + "dkv.norm", R)
                mat(p + "uq", H * (dn + dr), Q)
                mat(p + "uk", H * dn, R)
                mat(p + "uv", H * dv, R)
                mat(p + "o", d, H * dv, 0.5)
            mat(L + "rg1", d, d)
            vec(L + "rg1.b", d, 0.5, 0.0)
        elif s.kind == "mamba1":
            C, N, r = m["inner"], m["state"], m["dt_rank"]
            mat(p + "in", 2 * C, d)
            vec(p + "conv", (C, m["conv"]), 0.5, 0.0)
            vec(p + "conv.b", C, 0.1, 0.0)
            mat(p + "x", r + 2 * N, C)
            mat(p + "dt", C, r)
            vec(p + "dt.b", C, 1.0, -3.5)
            vec(p + "A_log", (C, N), 0.7, 1.0)
            vec(p + "D", C, 0.3, 1.0)
            mat(p + "o", d, C)
        elif s.kind == "wkv":
            H, n, r = m["heads"], m["heads"] * m["dim"], m["w_rank"]
            for k in "rkvgw":
                vec(p + "mu." + k, d, 0.25, 0.5)
            for k in "rkvg":
                mat(p + k, n, d)
            mat(p + "w1", r, d)
            mat(p + "w2", n, r)
            vec(p + "w0", n, 1.0, -3.0)
            vec(p + "u", (H, m["dim"]), 0.5, 0.3)
            vec(p + "norm", n)
            mat(p + "o", d, n)
        else:
            a, b = s.sub("left", "").m, s.sub("right", "").m
            nq, nk = a["heads"] * a["dim"], a["kv_heads"] * a["dim"]
            for k, n in (("q", nq), ("k", nk), ("v", nk), ("g", nq)):
                mat(p + "left." + k, n, d)
            mat(p + "left.o", d, nq)
            H, dv, n = b["heads"], b["vdim"], b["kv_heads"] * b["dim"]
            for k, c in (("q", n), ("k", n), ("v", H * dv)):
                mat(p + "right." + k, c, d)
                vec(p + "right." + k + ".conv", (c, b["conv"]), 0.5, 0.0)
            mat(p + "right.b", H, d)
            mat(p + "right.a", H, d)
            mat(p + "right.g", H * dv, d)
            vec(p + "right.A_log", H, 0.7, 0.0)
            vec(p + "right.dt_bias", H, 1.0, -3.5)
            vec(p + "right.norm", dv)
            mat(p + "right.o", d, H * dv)
            vec(p + "left.out", d, 0.2, 1.0)
            vec(p + "right.out", d, 0.2, 1.0)
        norm1b = cfg.arch == "dopivik"
        p = L + "mlp."
        if norm1b:
            norm(L + "norm1b")
        if cfg.arch != "dunesun":
            norm(L + "norm2")
        if isinstance(s.mlp, MoESpec):
            for e in range(s.mlp.experts):
                mat(f"{p}e{e}.gate", s.mlp.ff, d)
                mat(f"{p}e{e}.up", s.mlp.ff, d)
                mat(f"{p}e{e}.down", d, s.mlp.ff, 0.5)
            mat(p + "router", s.mlp.experts, d, 2.0)
            vec(p + "router.b", s.mlp.experts, 0.2, 0.0)
        elif cfg.arch == "bitonex":
            mat(p + "gate", s.mlp.ff, d)
            mat(p + "up", s.mlp.ff, d)
            mat(p + "down", d, s.mlp.ff, 0.5)
            mat(L + "rg2", d, d)
            vec(L + "rg2.b", d, 0.5, 0.0)
        else:
            norm(L + "norm2b")
            mat(p + "up", s.mlp.ff, d)
            mat(p + "down", d, s.mlp.ff)
    return out


class _Weights(dict):
    """Random tensors by checkpoint name, with values that a bf16 checkpoint could hold."""

    def __init__(self, cfg: HybridConfig, seed: int, device):
        g = torch.Generator(device=device).manual_seed(seed)
        super().__init__({k: (torch.randn(shape, generator=g, device=device) * std + mean).to(torch.bfloat16)
                          for k, (shape, std, mean) in _spec(cfg).items()})


def _tokens(case: dict, seed: int) -> list:
    """The token ids of every sequence of the step, cached and new ones."""
    g = torch.Generator().manual_seed(seed + 1)
    V = get_config(LLAMA).vocab_size - 256 if case["model"] == LLAMA else VOCAB  # Llama's last ids are special tokens
    return [torch.randint(3, V, (c + n,), generator=g).tolist() for c, n in _rows(case)]


def prepare(case: dict, seed: int, device: str = "cuda:0") -> dict:
    dtype = getattr(torch, case["dtype"])
    if case["model"] == LLAMA:
        model = build_model(get_config(LLAMA), device=device, dtype=dtype, seed=seed)
    else:
        cfg = _config(case["model"], case["width"])
        model = HybridLM(cfg, device=device, dtype=dtype, weights=_Weights(cfg, seed, device))
    rows, ids = _rows(case), _tokens(case, seed)
    blocks = sum((c + n) // 16 + 2 for c, n in rows) + 8
    runner = ModelRunner(model, RunnerConfig(max_num_seqs=len(rows), max_model_len=max(c + n for c, n in rows) + 16,
                                             num_blocks=blocks, seed=seed, keep_logits=True, use_graphs=device != "cpu"))
    manager = BlockManager(blocks, watermark=0.0, prefix_caching=False, state_slots=runner.num_state_slots)
    greedy = SamplingParams(temperature=0.0, ignore_eos=True)
    seqs = []
    for i, ((c, n), t) in enumerate(zip(rows, ids)):
        running = i < case["decode"]
        q = Sequence(prompt_ids=t[:c] if running else t, params=greedy)
        q.output_ids = t[c:] if running else []
        if not manager.allocate(q):
            raise RuntimeError("the step does not fit its pages")
        seqs.append(q)
    batch, held = [], 0
    with torch.no_grad():
        for q, (c, n) in zip(seqs, rows):  # what the step finds in the caches
            if not c:
                continue
            q.num_computed, q.chunk = 0, c
            batch.append(q)
            held += c
            if held >= 8192:
                runner.prefill(batch)
                batch, held = [], 0
        if batch:
            runner.prefill(batch)
        for q, (c, n) in zip(seqs, rows):
            q.num_computed, q.chunk, q.prefilled = c, n, len(q.output_ids) > 0
        if not case["prompts"] and device != "cpu":
            runner.capture_graphs([runner.bucket_for(case["decode"])])
    return {"runner": runner, "decode": seqs[:case["decode"]], "prompts": seqs[case["decode"]:], "flight": None}


def run(state: dict):
    runner, dec, pro = state["runner"], state["decode"], state["prompts"]
    with torch.no_grad():
        step = runner.prefill_launch(pro, dec) if pro else runner.decode_launch(dec)
    if state["flight"] is not None:  # as the engine does: a step's tokens are read while the next one runs
        runner.decode_collect(state["flight"])
    state["flight"] = step
    kv = runner.kv if runner.hybrid else {"k": runner.k_cache, "v": runner.v_cache}
    return {"logits": runner.last_logits[:len(dec) + len(pro)], "kv": kv}


# ---------------------------------------------------------------------------------------------------- work
def work(case: dict) -> dict:
    rows = _rows(case)
    T, R = sum(n for _, n in rows), len(rows)
    es = 4 if case["dtype"] == "float32" else 2

    def pairs(window=0, chunk=False):
        """(query, key) pairs of a causal attention over all sequences, and the cached keys it reads."""
        total = read = 0
        for c, n in rows:
            if not window:
                total += n * c + n * (n + 1) // 2
                read += c
            elif chunk:
                total += sum((p % window) + 1 for p in range(c, c + n))
                read += c % window
            else:
                total += sum(min(p + 1, window) for p in range(c, c + n))
                read += min(c, window - 1)
        return total, read

    if case["model"] == LLAMA:
        c = get_config(LLAMA)
        per = c.d_model * (c.q_dim + 2 * c.kv_dim) + c.q_dim * c.d_model + 3 * c.d_model * c.ffn_dim
        n, old = pairs()
        flops = 2.0 * T * c.n_layers * per + 2.0 * R * c.d_model * c.vocab_size + 4.0 * n * c.n_heads * c.head_dim * c.n_layers
        size = es * (c.n_layers * (per + (old + T) * 2 * c.kv_dim) + c.d_model * c.vocab_size + T * c.d_model) + 4 * R * c.vocab_size
        return {"bytes": float(size), "flops": flops}
    cfg = _config(case["model"], case["width"])
    d = cfg.d_model
    flops, size = 2.0 * R * d * VOCAB, float(es * (d * VOCAB + T * d) + 4 * R * VOCAB)
    spec = _spec(cfg)
    for i, s in enumerate(cfg.layers):
        m = s.m
        for name, (shape, _, _) in spec.items():
            if not name.startswith(f"l{i}.") or len(shape) != 2 or "conv" in name or "A_log" in name or name.endswith(".u"):
                continue
            n = shape[0] * shape[1]
            part = 1.0
            if ".e" in name:  # an expert sees top / experts of the tokens and is read if one chose it
                part = s.mlp.top / s.mlp.experts
                size += es * n * (1.0 - (1.0 - part) ** T)
            else:
                size += es * n
            flops += 2.0 * T * n * part
        if s.kind == "mamba2":
            st, ops = m["heads"] * m["vdim"] * m["state"], 5
        elif s.kind == "lightning":
            st, ops = m["heads"] * m["dim"] * m["vdim"], 5
        elif s.kind == "mamba1":
            st, ops = m["inner"] * m["state"], 7
        elif s.kind == "wkv":
            st, ops = m["heads"] * m["dim"] ** 2, 5
        elif s.kind == "parallel":
            st, ops = m["right.heads"] * m["right.dim"] * m["right.vdim"], 7
        else:
            st, ops = 0, 0
        flops += float(T) * st * ops
        size += 4.0 * st * (R + sum(1 for c, _ in rows if c))  # every state written, those of started sequences read
        if s.kind in ("attention", "parallel"):
            a = s.sub("left", "").m if s.kind == "parallel" else m
            n, old = pairs(a.get("mask.size", 0), s.kind == "parallel")
            flops += 4.0 * n * a["heads"] * a["dim"]
            size += float(es) * (old + T) * 2 * a["kv_heads"] * a["dim"]
        elif s.kind == "latent_attention":
            n, old = pairs()
            flops += 2.0 * n * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            size += float(es) * (old + (T if "kv_from" not in m else 0)) * (m["kv_rank"] + m["rot_dim"])
    return {"bytes": size, "flops": flops}


def tolerance(case: dict) -> dict:
    if case["dtype"] == "float32":
        return {"rel": 1e-4, "max": 2e-2}
    return {"rel": 0.03, "max": 0.9}


# ---------------------------------------------------------------------------------------------------- in 64 bits
F64 = torch.float64


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, dims: int, base: float, interleaved: bool):
    """Rotary positions on the first ``dims`` entries of x [tokens, heads, size]; token i is position i."""
    f = torch.tensor(base, dtype=F64, device=x.device) ** (-torch.arange(0, dims, 2, dtype=F64, device=x.device) / dims)
    a = (torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None] * f)[:, None, :]
    y = x.clone()
    u, w = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, dims // 2), slice(dims // 2, dims))
    y[..., u] = x[..., u] * a.cos() - x[..., w] * a.sin()
    y[..., w] = x[..., w] * a.cos() + x[..., u] * a.sin()
    return y


def _attend(q, k, v, scale, window=0, chunk=0, sink=False, cap=0.0):
    """q [n, H, dk], k [n, G, dk], v [n, G, dv] of one sequence -> [n, H * dv]; ``scale`` a number or one per head."""
    n, H = q.shape[:2]
    per = H // k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=F64, device=q.device)
    j = torch.arange(n, device=q.device)
    for h in range(H):
        sc = scale if isinstance(scale, float) else scale[h]
        for a in range(0, n, 2048):
            b = min(n, a + 2048)
            lo = max(0, a - window + 1) if window else (a // chunk) * chunk if chunk else 0
            i = j[a:b, None]
            s = (q[a:b, h] @ k[lo:b, h // per].T) * sc
            if cap:
                s = cap * torch.tanh(s / cap)
            seen = j[None, lo:b] <= i
            if window:
                seen &= i - j[None, lo:b] < window
            if chunk:
                seen &= j[None, lo:b] // chunk == i // chunk
            s = s.masked_fill(~seen, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink:
                top = top.clamp(min=0.0)
            e = torch.exp(s - top)
            out[a:b, h] = (e @ v[lo:b, h // per]) / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))
    return out.reshape(n, -1)


def _each(lens, fn, *xs):
    """fn over the sequences of [B, T, ...] batches, without their padding; the result padded again."""
    out = None
    for b, n in enumerate(lens):
        y = fn(*(x[b, :n] for x in xs))
        if out is None:
            out = torch.zeros(len(lens), xs[0].shape[1], *y.shape[1:], dtype=F64, device=y.device)
        out[b, :n] = y
    return out


def _conv(x, w, b=None):
    """Causal convolution per channel over [B, T, C], then SiLU."""
    taps = w.shape[1]
    y = sum(F.pad(x, (0, 0, taps - 1 - j, 0))[:, :x.shape[1]] * w[:, j] for j in range(taps))
    return F.silu(y + b if b is not None else y)


def _scan(lens, S, step):
    """The states after every sequence's last token, and step's results [B, T, ...]: step(t, S) updates S in place."""
    last = torch.empty_like(S)
    ys = []
    for t in range(max(lens)):
        ys.append(step(t, S))
        for b, n in enumerate(lens):
            if n == t + 1:
                last[b] = S[b]
    return last, torch.stack(ys, 1)


def _mixer(cfg, s, h, w, lens, kept, i):
    """(result [B, T, d], states laid out as the runner keeps them) of one layer's mixer."""
    B, T, d = h.shape
    m, eps, dev = s.m, cfg.norm_eps, h.device

    def heads(x, n):
        return x.view(B, T, n, -1)

    if cfg.arch == "dunesun" and s.kind == "attention":
        H, G = m["heads"], m["kv_heads"]
        q, k = (heads(_rms(h @ w(x).T, eps) * w(x + ".norm"), n) for x, n in (("q", H), ("k", G)))
        o = _each(lens, lambda *x: _attend(*x, m["scale"], window=m["mask.size"], sink=True), q, k, heads(h @ w("v").T, G))
        return o @ w("o").T, {}
    if s.kind == "mamba2":
        nh, P, N = m["heads"], m["vdim"], m["state"]
        inner = nh * P
        p = h @ w("in").T
        x, Bm, C = _conv(p[..., inner:2 * inner + 2 * N], w("conv"), w("conv.b")).split([inner, N, N], -1)
        x = heads(x, nh)
        dt = F.softplus(p[..., 2 * inner + 2 * N:] + w("dt_bias"))
        a, dx = torch.exp(-torch.exp(w("A_log")) * dt), dt[..., None] * x

        def step(t, S):
            S.mul_(a[:, t, :, None, None]).addcmul_(Bm[:, t, None, :, None], dx[:, t, :, None, :])
            return (S * C[:, t, None, :, None]).sum(2)

        S, y = _scan(lens, torch.zeros(B, nh, N, P, dtype=F64, device=dev), step)
        y = (y + w("D")[:, None] * x).reshape(B, T, inner) * F.silu(p[..., :inner])
        return (_rms(y, eps) * w("norm")) @ w("o").T, {"ssm": S}
    if s.kind == "attention":
        H, G = m["heads"], m["kv_heads"]

        def att(q, k, v):
            q, k = (_turn(x, m["rot.dims"], m["rot.base"], False) for x in (q, k))
            return _attend(q, k, v, m["scale"] * w("temp"))

        o = _each(lens, att, heads(h @ w("q").T, H), heads(h @ w("k").T, G), heads(h @ w("v").T, G))
        return (o * torch.sigmoid(h @ w("g").T)) @ w("o").T, {}
    if s.kind == "lightning":
        H = m["heads"]
        q, k, v = (heads(F.silu(h @ w(x).T), H) for x in "qkv")
        lam = torch.tensor(m["decay"], dtype=torch.float32, device=dev).double()[:, None, None]

        def step(t, S):
            S.mul_(lam).addcmul_(k[:, t, :, :, None], v[:, t, :, None, :])
            return (S * q[:, t, :, :, None]).sum(2)

        S, y = _scan(lens, torch.zeros(B, H, m["dim"], m["vdim"], dtype=F64, device=dev), step)
        y = _rms(y.reshape(B, T, -1), eps) * w("norm") * torch.sigmoid(h @ w("g").T)
        return y @ w("o").T, {"state": S}
    if s.kind == "latent_attention":
        H, dn, R = m["heads"], m["dim"], m["kv_rank"]
        if "kv_from" not in m:
            p = h @ w("dkv").T
            kept[i] = (_rms(p[..., :R], eps) * w("dkv.norm"), p[..., R:])
        c, kr = kept[m.get("kv_from", i)]
        q = heads((_rms(h @ w("dq").T, eps) * w("dq.norm")) @ w("uq").T, H)

        def att(q, c, kr):
            n = q.shape[0]
            qr = _turn(q[..., dn:], m["rot.dims"], m["rot.base"], True)
            kr = _turn(kr[:, None], m["rot.dims"], m["rot.base"], True).expand(n, H, -1)
            return _attend(torch.cat([q[..., :dn], qr], -1), torch.cat([(c @ w("uk").T).view(n, H, dn), kr], -1),
                           (c @ w("uv").T).view(n, H, -1), m["scale"])

        return _each(lens, att, q, c, kr) @ w("o").T, {}
    if s.kind == "mamba1":
        C, N, r = m["inner"], m["state"], m["dt_rank"]
        p = h @ w("in").T
        x = _conv(p[..., :C], w("conv"), w("conv.b"))
        q = x @ w("x").T
        dt = F.softplus(q[..., :r] @ w("dt").T + w("dt.b"))
        A, Bm, Cm = -torch.exp(w("A_log")), q[..., r:r + N], q[..., r + N:]

        def step(t, S):
            S.mul_(torch.exp(dt[:, t, :, None] * A)).addcmul_((dt[:, t] * x[:, t])[..., None], Bm[:, t, None, :])
            return (S * Cm[:, t, None, :]).sum(-1)

        S, y = _scan(lens, torch.zeros(B, C, N, dtype=F64, device=dev), step)
        return ((y + w("D") * x) * F.silu(p[..., C:])) @ w("o").T, {"state": S}
    if s.kind == "wkv":
        H = m["heads"]
        prev = F.pad(h, (0, 0, 1, 0))[:, :T]
        mix = {x: h + (prev - h) * w("mu." + x) for x in "rkvgw"}
        r, k, v = (heads(mix[x] @ w(x).T, H) for x in "rkv")
        dec = heads(torch.exp(-torch.exp(torch.tanh(mix["w"] @ w("w1").T) @ w("w2").T + w("w0"))), H)
        bonus = (r * w("u") * k).sum(-1, keepdim=True) * v

        def step(t, S):  # [value, key], as the runner keeps it
            o = (S * r[:, t, :, None, :]).sum(-1)
            S.mul_(dec[:, t, :, None, :]).addcmul_(v[:, t, :, :, None], k[:, t, :, None, :])
            return o

        S, y = _scan(lens, torch.zeros(B, H, m["dim"], m["dim"], dtype=F64, device=dev), step)
        y = _rms(y + bonus, eps).reshape(B, T, -1) * w("norm") * F.silu(mix["g"] @ w("g").T)
        ends = torch.stack([h[b, n - 1] for b, n in enumerate(lens)])
        return y @ w("o").T, {"state": S, "prev": ends}
    a, b = s.sub("left", "").m, s.sub("right", "").m

    def att(q, k, v):
        q, k = (_turn(x, a["rot.dims"], a["rot.base"], False) for x in (q, k))
        return _attend(q, k, v, a["scale"], chunk=a["mask.size"], cap=a["softcap"])

    left = _each(lens, att, heads(h @ w("left.q").T, a["heads"]), *(heads(h @ w("left." + x).T, a["kv_heads"]) for x in "kv"))
    left = (left * torch.sigmoid(h @ w("left.g").T)) @ w("left.o").T
    H, Gk, dk, dv = b["heads"], b["kv_heads"], b["dim"], b["vdim"]
    q, k = (heads(_conv(h @ w("right." + x).T, w(f"right.{x}.conv")), Gk) for x in "qk")
    q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    q, k = (x.repeat_interleave(H // Gk, 2) for x in (q * dk ** -0.5, k))
    v = heads(_conv(h @ w("right.v").T, w("right.v.conv")), H)
    beta = torch.sigmoid(h @ w("right.b").T)
    g = torch.exp(-torch.exp(w("right.A_log")) * F.softplus(h @ w("right.a").T + w("right.dt_bias")))

    def step(t, S):  # [value, key]
        S.mul_(g[:, t, :, None, None])
        u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, None, :]).sum(-1))
        S.addcmul_(u[..., None], k[:, t, :, None, :])
        return (S * q[:, t, :, None, :]).sum(-1)

    S, y = _scan(lens, torch.zeros(B, H, dv, dk, dtype=F64, device=dev), step)
    y = (_rms(y, eps) * w("right.norm")).reshape(B, T, -1) * F.silu(h @ w("right.g").T)
    right = y @ w("right.o").T
    return 0.5 * (_rms(left, eps) * w("left.out") + _rms(right, eps) * w("right.out")), {"right": {"state": S}}


def _exact_layers(case, seed, device):
    cfg = _config(case["model"], case["width"])
    weights, ids = _Weights(cfg, seed, device), _tokens(case, seed)
    lens = [len(t) for t in ids]
    T, eps = max(lens), cfg.norm_eps
    W = lambda name: weights[name].double()  # noqa: E731
    tok = torch.tensor([t + [0] * (T - len(t)) for t in ids], device=device)
    x = W("embed")[tok] * cfg.embed_scale
    if cfg.arch == "dunesun":
        x = x + W("pos")[:T]

    def norm(name, y):
        if cfg.arch == "dunesun":
            return _rms(y, eps) * (1.0 + W(name))
        if cfg.arch == "bitonex":
            return _rms(y, eps) * W(name)
        return F.layer_norm(y, (cfg.d_model,), W(name), W(name + ".b"), eps)

    kept, states = {}, []
    for i, s in enumerate(cfg.layers):
        L = f"l{i}."
        h = norm(L + "norm1", x)
        y, st = _mixer(cfg, s, h, lambda n: W(L + "mix." + n), lens, kept, i)
        states.append(st)
        if cfg.arch == "dunesun":
            flat, p = h.reshape(-1, cfg.d_model), L + "mlp."
            top, idx = (flat @ W(p + "router").T + W(p + "router.b")).topk(s.mlp.top, -1)
            wt = torch.softmax(top, -1)
            x = x + y
            for e in range(s.mlp.experts):
                at, slot = torch.nonzero(idx == e, as_tuple=True)
                he = flat[at]
                ye = (F.silu(he @ W(f"{p}e{e}.gate").T) * (he @ W(f"{p}e{e}.up").T)) @ W(f"{p}e{e}.down").T
                x.view(-1, cfg.d_model).index_add_(0, at, ye * wt[at, slot][:, None])
        elif cfg.arch == "bitonex":
            x = x + cfg.residual_mult * y * torch.sigmoid(h @ W(L + "rg1").T + W(L + "rg1.b"))
            h = norm(L + "norm2", x)
            y = (F.gelu(h @ W(L + "mlp.gate").T, approximate="tanh") * (h @ W(L + "mlp.up").T)) @ W(L + "mlp.down").T
            x = x + cfg.residual_mult * y * torch.sigmoid(h @ W(L + "rg2").T + W(L + "rg2.b"))
        else:
            x = x + norm(L + "norm1b", y)
            y = torch.relu(norm(L + "norm2", x) @ W(L + "mlp.up").T) ** 2
            x = x + norm(L + "norm2b", y @ W(L + "mlp.down").T)
        del y, h
    z = norm("final.norm", torch.stack([x[b, n - 1] for b, n in enumerate(lens)])) @ W("head").T
    if cfg.logit_softcap:
        z = cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap)
    return {"logits": z, "kv": states}


def _exact_llama(case, seed, device):
    c = get_config(LLAMA)
    d, D, Hq, Hk = c.d_model, c.head_dim, c.n_heads, c.n_kv_heads

    def W(name, n, k, std=0.02):  # a random-init model's tensors: normal values seeded per name
        s = int.from_bytes(hashlib.blake2b(f"{seed}:{name}".encode(), digest_size=8).digest(), "little") & 0x7FFFFFFFFFFFFFFF
        g = torch.Generator(device=device).manual_seed(s)
        return torch.empty(n, k, dtype=torch.bfloat16, device=device).normal_(0.0, std, generator=g).double()

    ids = _tokens(case, seed)
    lens = [len(t) for t in ids]
    V = c.vocab_size_padded(1)
    x = W("embed", V, d)[torch.tensor([t for s in ids for t in s], device=device)]
    out_std = 0.02 / math.sqrt(2 * c.n_layers)
    for i in range(c.n_layers):
        p = f"layers.{i}."
        h = _rms(x, c.norm_eps)
        q, k, v = ((h @ W(p + n, m * D, d).T).view(-1, m, D) for n, m in (("wq", Hq), ("wk", Hk), ("wv", Hk)))
        o = [_attend(_turn(a, D, c.rope_theta, False), _turn(b, D, c.rope_theta, False), e, D ** -0.5)
             for a, b, e in zip(q.split(lens), k.split(lens), v.split(lens))]
        x = x + torch.cat(o) @ W(p + "wo", d, Hq * D, out_std).T
        h = _rms(x, c.norm_eps)
        h = F.silu(h @ W(p + "w1", c.ffn_dim, d).T) * (h @ W(p + "w3", c.ffn_dim, d).T)
        x = x + h @ W(p + "w2", d, c.ffn_dim, out_std).T
    ends = torch.tensor(lens, device=device).cumsum(0) - 1
    return {"logits": (_rms(x[ends], c.norm_eps) @ W("lm_head", V, d).T)[:, :c.vocab_size]}


def exact(case: dict, seed: int, device: str = "cuda:0"):
    """The step's logits and recurrent states as whole sequences in float64 give them; the pages of the attention
    layers have a layout of their own and are left out."""
    tokens = sum(c + n for c, n in _rows(case))
    with torch.no_grad():
        if case["model"] == LLAMA:
            return _exact_llama(case, seed, device) if tokens <= 20000 else None  # 64 sequences would take a minute
        return _exact_layers(case, seed, device)
