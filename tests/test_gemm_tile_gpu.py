"""The 256 x 256 MFMA prefill GEMM (ops/csrc/gemm_tile.hip): dense and expert-grouped, plain and
SwiGLU epilogues, against plain PyTorch fp32 references of the same op."""
import pytest
import torch

from k8s_llm_monitor_amd import ops
from k8s_llm_monitor_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
F_ = torch.nn.functional


@pytest.fixture(autouse=True, scope="module")
def _native_loaded():
    ops.native()
    torch.manual_seed(0)


def _close(a, b, atol, rtol=0.0, what=""):
    err = (a.float() - b.float()).abs()
    tol = atol + rtol * b.float().abs()
    bad = (err > tol).sum().item()
    assert bad == 0, f"{what}: {bad} elements out of tolerance, max err {err.max().item():.4g}"


ALGOS = [0, 1]  # the 4-wave kernel: 0 one barrier per k-tile, 1 two
DENSE_ALGOS = ALGOS


@pytest.mark.parametrize("algo", DENSE_ALGOS)
@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (255, 512, 128), (300, 256, 192), (1000, 1536, 1024),
                                   (2048, 768, 4096), (513, 512, 14336 // 4), (4096, 1024, 640)])
def test_gemm_tile_dense(M, N, K, algo):
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) * 0.05).to(torch.bfloat16)
    y = ops.gemm_tile(x, w, algo=algo)
    _close(y.cpu(), F_.linear(x.cpu().float(), w.cpu().float()), atol=3e-2, rtol=2e-2, what=f"dense {M}x{N}x{K}")


@pytest.mark.parametrize("M,N", [(77, 400), (600, 16), (257, 1296)])
def test_gemm_tile_w4_n_tail(M, N):
    """The 4-wave kernel takes any N % 16 == 0 (partial last n-tile: clamped DMA rows, masked stores)."""
    K = 320
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) * 0.05).to(torch.bfloat16)
    for algo in ALGOS:
        y = ops.gemm_tile(x, w, algo=algo)
        _close(y.cpu(), F_.linear(x.cpu().float(), w.cpu().float()), atol=3e-2, rtol=2e-2, what=f"tail {M}x{N}")


def test_gemm_tile_w4_asymmetric_identity():
    """A = I with an asymmetric B: a transposed C-write or a swapped fragment map cannot pass."""
    K = 256
    x = torch.zeros(256, K, device=DEV, dtype=torch.bfloat16)
    x[:, :] = torch.eye(256, K, device=DEV, dtype=torch.bfloat16)
    n = torch.arange(512, device=DEV).float()[:, None]
    k = torch.arange(K, device=DEV).float()[None, :]
    w = ((n * 3 + k * 7) % 61 - 30).to(torch.bfloat16)  # small integers: exact in bf16
    for algo in ALGOS:
        y = ops.gemm_tile(x, w, algo=algo)
        assert torch.equal(y.float().cpu(), w.float().t().cpu()[:256])


@pytest.mark.parametrize("algo", DENSE_ALGOS)
@pytest.mark.parametrize("M", [7, 700])
def test_gemm_tile_swiglu(M, algo):
    K, F = 512, 768
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w13 = (torch.randn(2 * F, K, device=DEV) * 0.05).to(torch.bfloat16)
    y = ops.gemm_tile(x, ops.interleave_gate_up(w13).contiguous(), swiglu=True, algo=algo)
    r = ref.silu_mul(F_.linear(x.cpu().float(), w13.cpu().float()).to(torch.bfloat16))
    _close(y.cpu(), r, atol=3e-2, rtol=2e-2, what="swiglu")


@pytest.mark.parametrize("algo", ALGOS)
@pytest.mark.parametrize("counts", [[300, 0, 129, 1], [256, 512, 5, 700, 0, 0, 33, 64], [1]])
@pytest.mark.parametrize("swiglu", [False, True])
def test_gemm_tile_grouped(counts, swiglu, algo):
    E, K, N = len(counts), 512, 512
    rows = sum(counts)
    x = torch.randn(rows, K, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(E, N, K, device=DEV) * 0.05).to(torch.bfloat16)
    if swiglu:
        w = torch.stack([ops.interleave_gate_up(we) for we in w]).contiguous()
    off = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    y = ops.gemm_tile(x, w, off, swiglu=swiglu, algo=algo)
    o = 0
    for e, n in enumerate(counts):
        if n:
            r = F_.linear(x[o:o + n].cpu().float(), w[e].cpu().float()).to(torch.bfloat16)
            if swiglu:
                r = ref.silu_mul(r, interleaved=True)
            _close(y[o:o + n].cpu(), r, atol=3e-2, rtol=2e-2, what=f"expert {e}")
        o += n


def test_gemm_tile_grouped_local_slice():
    """A rank's slice of the offsets: other experts' rows stay as allocated (zero)."""
    counts = [200, 150, 90, 310]
    E, K, N = 4, 256, 256
    x = torch.randn(sum(counts), K, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(E, N, K, device=DEV) * 0.05).to(torch.bfloat16)
    off = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    y = ops.gemm_tile(x, w[1:3].contiguous(), off[1:4])
    assert int(y[:200].abs().sum()) == 0 and int(y[440:].abs().sum()) == 0
    for e, (a, b) in ((1, (200, 350)), (2, (350, 440))):
        _close(y[a:b].cpu(), F_.linear(x[a:b].cpu().float(), w[e].cpu().float()), atol=3e-2, rtol=2e-2,
               what=f"local expert {e}")


def test_gemm_tile_in_graph_matches_eager():
    x = torch.randn(600, 1024, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(1024, 1024, device=DEV) * 0.03).to(torch.bfloat16)
    y0 = ops.gemm_tile(x, w)
    out = torch.empty_like(y0)
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        ops.gemm_tile(x, w, out=out)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, y0)


@pytest.mark.parametrize("algo", ALGOS)
@pytest.mark.parametrize("M,N,K", [(300, 256, 192), (1000, 1536, 1024), (257, 1296, 640), (2048, 768, 4096)])
def test_gemm_tile_packed_weights_bit_identical(M, N, K, algo):
    """W in the decode GEMMs' fragment-packed layout (pack_skinny) gives the same bits as W
    row-major: only the DMA source / LDS image of W change, not the MFMA operands or their order -
    plain, SwiGLU, grouped, RoPE + row scale and the residual epilogue."""
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) * 0.05).to(torch.bfloat16)
    assert torch.equal(ops.gemm_tile(x, ops.pack_skinny(w), algo=algo), ops.gemm_tile(x, w, algo=algo))
    if N % 256 == 0:
        wi = ops.interleave_gate_up(w).contiguous()
        assert torch.equal(ops.gemm_tile(x, ops.pack_skinny(wi), swiglu=True, algo=algo),
                           ops.gemm_tile(x, wi, swiglu=True, algo=algo))
    counts = [M // 3, 0, M - M // 3]
    off = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    we = torch.stack([w, w.flip(0), w * 0.5]).contiguous()
    wep = torch.stack([ops.pack_skinny(e) for e in we]).contiguous()
    assert torch.equal(ops.gemm_tile(x, wep, off, algo=algo), ops.gemm_tile(x, we, off, algo=algo))
    if algo == 1 and K >= 192 and K % 128 == 0 and N % 128 == 0:
        pos = torch.arange(M, device=DEV, dtype=torch.int32)
        cs = ref.rope_cos_sin(4096, 128, 500000.0).to(DEV).float().contiguous()
        ss = (torch.rand(M, K // 128, device=DEV) * 64 + 16).contiguous()
        kw = dict(algo=1, rope=(pos, cs, N // 128), rowscale=(ss, 1e-5))
        assert torch.equal(ops.gemm_tile(x, ops.pack_skinny(w), **kw), ops.gemm_tile(x, w, **kw))
        resid = torch.randn(M, N, device=DEV, dtype=torch.bfloat16)
        nw = (torch.rand(N, device=DEV) + 0.5).to(torch.bfloat16)
        r1, r2 = resid.clone(), resid.clone()
        h1, s1 = ops.gemm_tile_resid(x, ops.pack_skinny(w), r1, nw)
        h2, s2 = ops.gemm_tile_resid(x, w, r2, nw)
        assert torch.equal(r1, r2) and torch.equal(h1, h2) and torch.equal(s1, s2)


@pytest.mark.parametrize("M", [7, 700, 1500])
@pytest.mark.parametrize("rowscale", [False, True])
def test_gemm_tile_swiglu8_matches_fp32_and_decode_layout(M, rowscale):
    """SwiGLU over the decode GEMMs' gate/up copy (interleave_gate_up8, fragment-packed): the
    features silu(gate) * up against fp32, row-major vs packed bit for bit, dense and grouped -
    the one weight copy prefill and decode share."""
    K, F = 512, 768
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w13 = (torch.randn(2 * F, K, device=DEV) * 0.05).to(torch.bfloat16)
    w8 = ops.interleave_gate_up8(w13).contiguous()
    kw = {}
    xs = x.cpu().float()
    if rowscale:
        ss = (torch.rand(M, K // 128, device=DEV) * 64 + 16).contiguous()
        kw = dict(algo=1, rowscale=(ss, 1e-5))
        xs = xs * torch.rsqrt(ss.cpu().sum(1, keepdim=True) / K + 1e-5)
    y = ops.gemm_tile(x, ops.pack_skinny(w8), swiglu=8, **kw)
    assert torch.equal(y, ops.gemm_tile(x, w8, swiglu=8, **kw))
    gu = F_.linear(xs, w13.cpu().float()).to(torch.bfloat16).float()
    r = F_.silu(gu[:, :F]) * gu[:, F:]
    _close(y.cpu(), r, atol=3e-2, rtol=2e-2, what="swiglu8")
    if not rowscale:
        counts = [M // 2, M - M // 2]
        off = torch.tensor([0, counts[0], M], dtype=torch.int32, device=DEV)
        we = torch.stack([ops.pack_skinny(w8), ops.pack_skinny(w8.flip(1).contiguous())]).contiguous()
        yg = ops.gemm_tile(x, we, off, swiglu=8)
        assert torch.equal(yg[: counts[0]], y[: counts[0]])


@pytest.mark.parametrize("m_tiles,n_tiles,last,K,swiglu", [
    (1, 1, 1, 192, False), (5, 13, 64, 192, True), (8, 8, 65, 256, True), (9, 8, 129, 256, False), (13, 20, 200, 192, True),
    (16, 20, 256, 192, False), (16, 21, 3, 192, False), (17, 15, 193, 640, True),
])
def test_gemm_tile_last_round(m_tiles, n_tiles, last, K, swiglu):
    """Tiles beyond whole rounds of 256 as strips of 64 rows (up to 64 of them), dense, grouped (with an empty expert and short ones) and
    ended by a gated unit: the bits of the schedule that has whole tiles only."""
    g = torch.Generator().manual_seed(5)
    M, N = 256 * (m_tiles - 1) + last, 256 * n_tiles
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(2, N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    assert torch.equal(ops.gemm_tile(x, w[0], swiglu=swiglu, algo=1), ops.gemm_tile(x, w[0], swiglu=swiglu, algo=0))
    w3 = torch.cat([w, w[:1]])
    for cut in (M // 3, M - M // 5, M):
        off = torch.tensor([0, cut, cut, M], dtype=torch.int32, device="cuda")
        assert torch.equal(ops.gemm_tile(x, w3, off, swiglu=swiglu, algo=1), ops.gemm_tile(x, w3, off, swiglu=swiglu, algo=0))
    f = N // 2 - 64  # the unit's last tile is short; 128 more columns stand behind it
    y, y2 = torch.empty(M, f, dtype=torch.bfloat16, device="cuda"), torch.empty(M, 128, dtype=torch.bfloat16, device="cuda")
    ops.native().gemm_tile_unit(y, y2, x, w[1], 6)  # SiLU
    z = ops.gemm_tile(x, w[1], algo=0)
    up, gate = z[:, f:2 * f].float(), z[:, :f].float()
    torch.testing.assert_close(y.float(), torch.nn.functional.silu(gate) * up, rtol=2 ** -7, atol=2 ** -7)
    assert torch.equal(y2, z[:, 2 * f:])


@pytest.mark.parametrize("M,N,K,f", [  # 32 and 33 tiles, one behind a round, none of the second half's columns, a unit's half without features
    (1000, 2048, 256, 960), (1000, 2128, 192, 1056), (4097, 4096, 192, 1984), (300, 128, 640, 48), (300, 400, 192, 80), (8100, 2064, 256, 1000 // 16 * 16),
])
def test_gemm_tile_last_round_in_fine_strips(M, N, K, f):
    """Up to 32 tiles beyond whole rounds of 256 as strips of 64 rows x 128 columns: the bits of whole tiles, weights packed or not; a gated unit with other
    columns behind it."""
    g = torch.Generator().manual_seed(6)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    z = ops.gemm_tile(x, w, algo=0)
    off = torch.tensor([0, M], dtype=torch.int32, device="cuda")  # (dense products of few tiles have strips of their own)
    assert torch.equal(ops.gemm_tile(x, w[None], off, algo=1), z)
    assert torch.equal(ops.gemm_tile(x, w, algo=1), z)
    assert torch.equal(ops.gemm_tile(x, ops.pack_skinny(w)[None], off, algo=1), z)
    y, y2 = torch.empty(M, f, dtype=torch.bfloat16, device="cuda"), torch.empty(M, N - 2 * f, dtype=torch.bfloat16, device="cuda")
    ops.native().gemm_tile_unit(y, y2, x, w, 7)  # ReLU: exact but for the product's rounding
    assert torch.equal(y, (z[:, :f].float().clamp(min=0) * z[:, f:2 * f].float()).to(torch.bfloat16))
    assert torch.equal(y2, z[:, 2 * f:])


def _form(M, N, K, f=0, epi=0, rowscale=False):
    """(rows of a tile, tiles, tiles beyond whole rounds of 256) of a dense product, by the launcher's own rule."""
    rows, cols, n = ops.native().gemm_tile_form(M, N, K, f, epi, rowscale)
    return (rows, n, n % 256) if cols == 256 else (rows, n, None)


@pytest.mark.parametrize("M,N,K,f,form", [  # the last tile of 1, 33, 131, 150 and 224 rows; behind whole rounds 1, 8, 32, 33, 48 and 64 tiles in strips, none, and too many
    (224 * 28 + 1, 4096, 192, 1984, (224, 493, 237)), (224 * 14 + 33, 4096, 256, 2048, (224, 240, 240)), (6403, 4096, 320, 2000, (224, 493, 237)),
    (7830, 13312, 192, 5632, (256, 1612, 76)), (224 * 16, 8192 - 128, 640, 3072, (224, 512, 0)), (200, 65792, 192, 128, (224, 257, 1)),
    (1281, 11264, 192, 5632, (224, 264, 8)), (2561, 6144, 320, 2048, (224, 288, 32)), (2688, 6144, 192, 3072, (224, 288, 32)), (200, 73984, 192, 128, (224, 289, 33)),
    (1025, 28672, 192, 14336, (224, 560, 48)), (1119, 16384, 256, 8192, (224, 320, 64)), (4097, 4096, 192, 1984, (256, 289, 33)),
])
def test_gemm_tile_units_of_224_rows(M, N, K, f, form):
    """Units and squared ReLU on tiles of 224 rows where those are fewer rounds, whole ones beside strips among them: the bits of the other schedule's whole tiles."""
    assert _form(M, N, K, f, 7) == form
    g = torch.Generator().manual_seed(7)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    z = ops.gemm_tile(x, w, algo=0)
    y, y2 = torch.empty(M, f, dtype=torch.bfloat16, device="cuda"), torch.empty(M, N - 2 * f, dtype=torch.bfloat16, device="cuda")
    ops.native().gemm_tile_unit(y, y2, x, w, 7)  # ReLU: exact but for the product's rounding
    assert torch.equal(y, (z[:, :f].float().clamp(min=0) * z[:, f:2 * f].float()).to(torch.bfloat16))
    assert torch.equal(y2, z[:, 2 * f:])
    q = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ops.native().gemm_tile_unit(q, None, x, w, 8)
    assert torch.equal(q, (z.float().clamp(min=0) ** 2).to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K,form", [  # behind whole rounds 1, 16, 17, 32, 33, 48, 59 and 64 tiles, none, too many; a last tile of one row and of all
    (4097, 4096, 512, (256, 272, 16)), (4608, 4096, 512, (256, 288, 32)), (3073, 5376, 1024, (256, 273, 17)), (5120, 4096, 512, (256, 320, 64)),
    (1636, 28672, 512, (256, 784, 16)), (3585, 4096, 512, (256, 240, 240)), (700, 6144, 1536, (224, 96, 96)), (257, 1024, 512, (224, 8, 8)),
    (200, 65792, 512, (224, 257, 1)), (2610, 6144, 512, (224, 288, 32)), (1537, 28672, 512, (224, 784, 16)), (224, 73984, 512, (224, 289, 33)),
    (1085, 28672, 512, (224, 560, 48)), (3329, 5376, 1024, (224, 315, 59)), (1120, 16384, 512, (224, 320, 64)), (6945, 4096, 512, (224, 512, 0)),
    (5121, 4096, 512, (224, 368, 112)),
])
def test_gemm_tile_fused_ends_of_strips(M, N, K, form):
    """Residual, rotation and row scale at the end of strips and of tiles of 224 rows: the bits of the plain product on whole tiles, finished here.  (Scales are
    powers of two, so that they commute with every rounding.)"""
    assert _form(M, N, K, epi=3) == form and _form(M, N, K, epi=2, rowscale=True) == form and _form(M, N, K, epi=4, rowscale=True) == form
    g = torch.Generator().manual_seed(8)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    wr = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    w = ops.pack_skinny(wr)
    z = ops.gemm_tile(x, wr, algo=0)
    if _form(M, N, K) == form:
        assert torch.equal(ops.gemm_tile(x, w, algo=1), z)
    r, nw = torch.randn(M, N, generator=g).to(torch.bfloat16).cuda(), (torch.rand(N, generator=g) + 0.5).to(torch.bfloat16).cuda()
    h = (z.float() + r.float()).to(torch.bfloat16)
    hw, ss = ops.gemm_tile_resid(x, w, r, nw)
    assert torch.equal(r, h)
    assert torch.equal(hw, (h.float() * nw.float()).to(torch.bfloat16))
    torch.testing.assert_close(ss, (h.float() ** 2).view(M, N // 128, 128).sum(2), rtol=1e-5, atol=1e-5)  # 128 fp32 terms
    row = torch.arange(M, device=DEV)
    scale = (2.0 ** (row % 5 - 2)).float()[:, None]
    part = torch.zeros(M, K // 128, device=DEV)
    part[:, 1:2] = K / scale ** 2  # 1 / rms = scale
    pos, cs = (row % 97).to(torch.int32), torch.rand(97, 128, generator=g).cuda()
    heads = N // 128 - 3
    want = ops.gemm_tile(x, wr, algo=0, rope=(pos, cs, heads))
    assert torch.equal(ops.gemm_tile(x, w, algo=1, rope=(pos, cs, heads)), want)
    assert torch.equal(ops.gemm_tile(x, w, algo=1, rope=(pos, cs, heads), rowscale=(part, 0.0)), (want.float() * scale).to(torch.bfloat16))
    big = (x.float() * scale).to(torch.bfloat16)
    assert torch.equal(ops.gemm_tile(x, w, swiglu=8, algo=1, rowscale=(part, 0.0)), ops.gemm_tile(big, wr, swiglu=8, algo=0))


@pytest.mark.parametrize("M,N,K,form", [  # tiles of 224 and of 256 rows, alone, in 64 x 256 strips and in 64 x 128 ones, and whole ones beside those
    (1, 128, 192, (224, 1, 1)), (300, 384, 192, (224, 4, 4)), (4097, 384, 320, (224, 38, 38)), (9000, 384, 192, (224, 82, 82)), (4097, 4224, 192, (256, 289, 33)),
    (7937, 4224, 192, (256, 544, 32)), (10240, 4224, 192, (256, 680, 168)), (4609, 4224, 256, (224, 357, 101)), (1025, 28544, 192, (224, 560, 48)),
    (1537, 28544, 192, (224, 784, 16)),
])
def test_gemm_tile_residual_behind_half_a_tile(M, N, K, form):
    """N % 256 == 128: the last tile's second 128 columns are not there.  Every row's residual, weighted row and sums of squares are the plain product's,
    finished here, and nothing behind the buffers' ends is written."""
    assert _form(M, N, K, epi=3) == form
    g = torch.Generator().manual_seed(9)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    nw = (torch.rand(N, generator=g) + 0.5).to(torch.bfloat16).cuda()
    z, r = ops.gemm_tile(x, w, algo=0), torch.randn(M, N, generator=g).to(torch.bfloat16).cuda()
    h = (z.float() + r.float()).to(torch.bfloat16)
    bufs = [torch.full((M * n + 512,), 7.0, dtype=dt, device=DEV) for n, dt in ((N, torch.bfloat16), (N, torch.bfloat16), (N // 128, torch.float32))]
    res, hw, ss = (b[:-512].view(M, -1) for b in bufs)
    for wt in (w, ops.pack_skinny(w)):
        res.copy_(r)
        ops.gemm_tile_resid(x, wt, res, nw, hw, ss)
        assert torch.equal(res, h) and torch.equal(hw, (h.float() * nw.float()).to(torch.bfloat16))
        torch.testing.assert_close(ss, (h.float() ** 2).view(M, N // 128, 128).sum(2), rtol=1e-5, atol=1e-5)  # 128 fp32 terms
        assert all(bool((b[-512:] == 7.0).all()) for b in bufs)


@pytest.mark.parametrize("M,N,K,packed", [
    (1, 128, 192, False), (65, 4096, 4096, True), (43, 6144, 4096, True), (257, 1024, 8192, False), (512, 512, 1088, False), (80, 28672, 4096, True),
    (600, 6144, 2112, True), (1000, 1024, 4096, False), (70, 320, 512, False), (260, 4096, 2048, True),  # (64 columns: one round of strips, and more)
    (385, 6144, 192, False), (400, 6144, 1088, True), (113, 28672, 320, True), (1000, 4096, 1024, True), (128, 16640, 2048, False),  # (128 rows)
    (2300, 1536, 192, True), (2300, 1408, 192, False), (1300, 2304, 320, True), (4000, 768, 192, False),  # (columns over the XCDs: two rounds, and one)
])
def test_gemm_tile_narrow_strips(M, N, K, packed):
    """Products of few tiles as strips of 64 x 128, 64 x 64 or 128 x 128: plain, turned, gated in both pairings.  The bits of the schedule that has whole tiles
    only."""
    g = torch.Generator().manual_seed(6)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    w = ops.pack_skinny(w) if packed else w
    assert torch.equal(ops.gemm_tile(x, w, algo=1), ops.gemm_tile(x, w, algo=0))
    if N % 128:
        return
    pos = torch.randint(0, 300, (M,), generator=g, dtype=torch.int32).cuda()
    rope = (pos, torch.randn(300, 128, generator=g).cuda(), max(N // 128 - 2, 0))
    assert torch.equal(ops.gemm_tile(x, w, algo=1, rope=rope), ops.gemm_tile(x, w, algo=0, rope=rope))
    if N % 256 == 0:
        for kind in (True, 8):
            assert torch.equal(ops.gemm_tile(x, w, swiglu=kind, algo=1), ops.gemm_tile(x, w, swiglu=kind, algo=0))
