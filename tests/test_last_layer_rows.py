"""A prefill step that returns few rows' logits goes on with these rows alone behind its last mixer: logits, pages and states against a step
that returns every row's."""
import dataclasses

import pytest
import torch

from k8s_llm_monitor_amd import ops
from k8s_llm_monitor_amd.engine.block_manager import BlockManager
from k8s_llm_monitor_amd.engine.runner import ModelRunner, RunnerConfig
from k8s_llm_monitor_amd.engine.sequence import SamplingParams, Sequence
from k8s_llm_monitor_amd.models import HybridLM, build_model, get_config
from k8s_llm_monitor_amd.models.hybrid import _take

PRESETS = ["dunesun-tiny", "kisutar-tiny", "bitonex-tiny", "levovik-tiny", "dopivik-tiny", "zifisun-tiny"]


@pytest.fixture(autouse=True)
def _small_steps(monkeypatch):
    """Steps of these sizes too pick rows that do not lie together."""
    real = HybridLM._wanted

    def wanted(self, meta, T):
        w = real(self, meta, T)
        few = meta.is_prefill and meta.logits_idx is not None and 0 < 2 * meta.logits_idx.numel() <= T
        return meta.logits_idx if w is None and few else w

    monkeypatch.setattr(HybridLM, "_wanted", wanted)


def _step(model, every, cuts, lens=(37, 5, 50, 9), blocks=40):
    """Logits of the last rows and the caches after one prompt (the last of ``lens``), then the others in portions, the last of them beside
    its running sequence."""
    runner = ModelRunner(model, RunnerConfig(max_num_seqs=4, max_model_len=blocks * 16 // 5, num_blocks=blocks, keep_logits=True, use_graphs=False))
    manager = BlockManager(blocks, watermark=0.0, prefix_caching=False, state_slots=getattr(runner, "num_state_slots", 0))
    g = torch.Generator().manual_seed(5)
    ids = [torch.randint(3, model.cfg.vocab_size, (n,), generator=g).tolist() for n in lens]
    seqs = [Sequence(prompt_ids=t, params=SamplingParams(temperature=0.0, ignore_eos=True)) for t in ids]
    out = []
    for q in seqs:
        assert manager.allocate(q)

    def go(pro, dec):
        with torch.no_grad():
            rows = [[0] for _ in dec] + [list(range(q.chunk)) for q in pro]
            h = runner.prefill_launch(pro, dec, logit_rows=rows if every else None)
        z = h.logits if every else runner.last_logits
        last = torch.tensor([len(r) for r in rows]).cumsum(0) - 1
        out.append((z[last.to(z.device)] if every else z).float().cpu())

    run = seqs[3]
    run.num_computed, run.chunk = 0, len(ids[3]) - 1
    go([run], [])
    run.prompt_ids, run.output_ids = ids[3][:-1], ids[3][-1:]
    run.num_computed, run.chunk, run.prefilled = len(ids[3]) - 1, 1, True
    for a, b in zip(cuts, cuts[1:]):
        pro = [q for q in seqs[:3] if len(q.prompt_ids) > int(len(q.prompt_ids) * a)]
        for q in pro:
            q.num_computed = int(len(q.prompt_ids) * a)
            q.chunk = int(len(q.prompt_ids) * b) - q.num_computed
        go(pro, [run] if b == 1 else [])

    def flat(c):
        return [t for v in c.values() for t in (flat(v) if isinstance(v, dict) else [v])]

    return out, [t.float().cpu() for c in runner.kv for t in (flat(c) if isinstance(c, dict) else c)]


def _compare(model, tol, *sizes):
    for cuts in ((0, 1), (0, 0.4, 1)):
        (a, ca), (b, cb) = _step(model, False, cuts, *sizes), _step(model, True, cuts, *sizes)
        for x, y in zip(a, b):
            assert x.shape == y.shape and float((x - y).norm() / y.norm()) < tol
        for x, y in zip(ca, cb):  # what the last mixer wrote does not depend on whose logits are wanted
            torch.testing.assert_close(x, y, rtol=0, atol=0)


def _models(name, device, dtype, make=get_config):
    cfg = make(name)
    for k in range(1, len(cfg.layers) + 1):  # every layer as the last one
        yield HybridLM(dataclasses.replace(cfg, name=f"{name}-{k}", layers=cfg.layers[:k], loop=None), device=device, dtype=dtype, seed=3)


def _odd(name):
    """The preset with a width and mixer results that are not a multiple of 8 columns."""
    cfg, new = get_config(name), []
    for s in cfg.layers:
        m = dict(s.mixer)
        for k in ("vdim", "right.vdim"):
            if k in m and s.kind != "latent_attention":
                m[k] = m[k] // 2 | 1
        if s.kind == "wkv":
            m["dim"] = 14
        new.append(dataclasses.replace(s, mixer=tuple(sorted(m.items()))))
    return dataclasses.replace(cfg, d_model=cfg.d_model + 12, layers=tuple(new))


def test_take_keeps_whole_rows():
    """Rows of whole tensors come whole, whatever their width: the kernels want residuals, normed rows and fp32 results contiguous.  Columns of
    wider rows stay a multiple of 8 values apart."""
    idx = torch.tensor([2, 5])
    for x in (torch.randn(7, 100), torch.randn(7, 45), torch.randn(7, 90).bfloat16(), torch.randn(7, 3, 10)):
        (y,) = _take(idx, x)
        assert y.is_contiguous() and torch.equal(y, x[idx])
    wide = torch.randn(7, 64)
    for a, b in ((0, 20), (8, 45), (16, 32)):
        (y,) = _take(idx, wide[:, a:b])
        assert torch.equal(y, wide[idx, a:b]) and y.stride() == (-(a - b) + (a - b) % 8, 1)


@pytest.mark.parametrize("name", PRESETS)
def test_last_layer_on_wanted_rows(name):
    for m in _models(name, "cpu", torch.float32):
        _compare(m, 1e-4)  # fp32 sums of other shapes


def test_wanted_rows_llama_of_small_steps():
    """Below 1024 rows (and on the CPU) Llama takes every row to the final norm."""
    _compare(build_model(get_config("llama-tiny"), device="cpu", dtype=torch.float32, seed=3), 1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 3e-2)])  # bf16: one layer's roundings, each 2^-9
@pytest.mark.parametrize("name", PRESETS)
def test_gpu_last_layer_on_wanted_rows(name, dtype, tol):
    for m in _models(name, "cuda:0", dtype):
        _compare(m, tol)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["dunesun-tiny", "bitonex-tiny", "levovik-tiny", "dopivik-tiny"])
def test_gpu_last_layer_on_wanted_rows_odd_widths(name):
    for m in _models(name, "cuda:0", torch.float32, _odd):
        _compare(m, 1e-4)


@pytest.mark.gpu
def test_gpu_wanted_rows_llama_of_small_steps():
    _compare(build_model(get_config("llama-tiny-d128"), device="cuda:0", dtype=torch.bfloat16, seed=3), 1e-2)


@pytest.mark.gpu
def test_gpu_last_layer_on_wanted_rows_llama(monkeypatch):
    """Steps of 1024 rows and more, several prompts and a running sequence's token: behind the last attention only the wanted rows go on,
    through the same tile kernels, which give a row the same bits whatever rows lie beside it."""
    rows, real = [], ops.gemm_tile_resid
    monkeypatch.setattr(ops, "gemm_tile_resid", lambda x, *a, **k: rows.append(x.shape[0]) or real(x, *a, **k))
    model = build_model(get_config("llama-tiny-d128"), device="cuda:0", dtype=torch.bfloat16, seed=3)
    n, lens = len(model.layers), (1300, 1111, 1500, 1200)
    _compare(model, 1e-2, lens, 500)
    per = 2 * n - 1  # out-projections and all but the last down-projection
    steps = [rows[i:i + per] for i in range(0, len(rows), per)]
    few, total = [1, 4, 1, 3, 4], [1199, 3912, 1199, 1564, 2348]  # of one cut, and of a cut at 0.4 (its rows all in such steps)
    cut = [int(0.4 * t) for t in lens[:3]]
    assert total[3] == sum(cut) and total[4] == sum(lens[:3]) + 1 - sum(cut)
    want = [[t] * (per - 1) + [k] for t, k in zip(total, few)]
    every = [[t] * per for t in total]
    assert steps == want[:2] + every[:2] + want[2:] + every[2:]
