"""Which kernel takes a projection, by its sizes: points on both sides of each rule, with the times beside the rules."""
import pytest

from k8s_llm_monitor_amd.ops import hybrid as hops


@pytest.mark.parametrize("M,N,K,f,takes", [
    (7830, 13312, 2048, 5632, True), (3749, 13312, 2048, 5632, True), (256, 53248, 2048, 26624, True), (1300, 53248, 2048, 0, True),
    (1, 53248, 2048, 26624, False), (64, 102400, 1024, 0, False), (128, 57344, 8192, 28672, False),  # a decode step's rows
    (300, 53248, 2048, 26624, False),  # two row tiles, little more than half full
    (50000, 288, 1024, 144, False),  # the same of features
    (6403, 4096, 1024, 0, True), (1300, 13312, 2048, 0, False),  # a last round that is half full, mostly empty
])
def test_tile_gemm_with_a_unit(M, N, K, f, takes):
    assert hops._tile_form(M, N, K, f) is takes


@pytest.mark.parametrize("end,M,N,K,form", [
    ("glu", 16, 8192, 4096, "own"), ("glu", 33, 8192, 4096, None), ("glu", 64, 8192, 2048, "own"), ("glu", 32, 13312, 2048, None),
    ("glu", 64, 16384, 4096, None), ("glu", 4, 32768, 4096, "own"), ("glu", 16, 32768, 4096, "shared"), ("glu", 1, 10240, 5632, None),
    ("", 16, 8192, 4096, None), ("", 16, 10240, 4096, "shared"), ("", 4, 8192, 4096, "own"), ("", 16, 2048, 2048, "own"),
    ("", 64, 2048, 2048, "own"), ("", 64, 4096, 4096, None), ("", 4, 65536, 1024, "shared"), ("", 1, 128256, 4096, "own"),
    ("", 16, 128256, 4096, None), ("", 3, 6144, 6144, None), ("", 4, 4096, 6144, "own"), ("", 1, 2048, 6176, None),
    ("act", 64, 8192, 4096, None), ("act", 64, 12288, 4096, "shared"), ("act", 64, 24576, 2048, None), ("act", 32, 24576, 2048, "shared"),
    ("act", 65, 2048, 2048, None),
])
def test_projections_of_few_rows(end, M, N, K, form):
    assert hops._rows_form(M, N, K, end) == form


@pytest.mark.parametrize("end,M,N,K,form", [
    ("", 33, 56832, 256, None), ("", 48, 28672, 256, "shared"), ("", 64, 16384, 512, "own"), ("", 56, 54944, 2496, None), ("", 64, 32768, 4096, "shared"),
    ("", 28, 10368, 1056, "shared"), ("", 28, 8192, 2048, "own"), ("act", 48, 35136, 256, "shared"), ("act", 56, 52000, 2688, None),
    ("act", 56, 45056, 2688, "shared"), ("act", 33, 9920, 2048, "shared"), ("act", 56, 51072, 5056, None), ("act", 56, 45056, 5056, "shared"),
    ("glu", 16, 29952, 64, "shared"), ("glu", 8, 28672, 1024, "shared"), ("glu", 8, 28672, 1056, "own"), ("glu", 48, 13248, 256, "own"),
    ("glu", 48, 23824, 160, "shared"), ("glu", 28, 11840, 192, "shared"), ("glu", 28, 11840, 1024, "own"), ("glu", 28, 24576, 4096, "shared"),
])
def test_projections_of_few_rows_and_small_k(end, M, N, K, form):
    assert hops._rows_form(M, N, K, end) == form


@pytest.mark.parametrize("M,N,K,takes", [
    (6403, 5648, 1024, True), (1024, 5648, 1024, False), (7830, 3104, 2048, True), (5400, 3104, 2048, False), (8000, 11296, 2048, False),
    (7830, 5632, 1024, False), (7830, 5640, 1024, False), (7830, 5648, 1056, False), (7830, 5648, 128, False), (8000, 1040, 192, False), (8000, 1040, 512, True),
    (1023, 60016, 1024, False), (1024, 60016, 1024, True), (1024, 1 << 19 | 16, 1024, False), (8000, 4080, 2048, True), (8000, 4112, 2048, False),
])
def test_tile_gemm_of_plain_products(M, N, K, takes):
    assert hops._tile_plain(M, N, K) is takes


@pytest.mark.parametrize("T,H,R,pages,window,want", [
    (0, 8, 128, 512, 0, (1, 1)), (1, 8, 128, 15, 0, (1, 16)), (1, 8, 128, 16, 0, (2, 16)), (1, 8, 128, 512, 0, (16, 16)), (8, 16, 256, 512, 0, (16, 16)),
    (15, 8, 128, 512, 0, (8, 16)), (16, 8, 128, 39, 0, (1, 40)), (16, 8, 128, 40, 0, (5, 40)), (16, 16, 256, 39, 0, (5, 16)), (16, 20, 256, 512, 0, (4, 16)),
    (17, 20, 256, 512, 0, (3, 40)), (64, 16, 256, 512, 0, (3, 40)), (65, 16, 256, 512, 0, (1, 1)), (33, 20, 256, 512, 0, (1, 1)), (1, 8, 128, 512, 200, (1, 16)),
    (1, 8, 128, 512, 1024, (9, 16)),
])
def test_parts_of_latent_rows(T, H, R, pages, window, want):
    assert hops.latent_parts(T, H, R, pages, window) == want


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2304, 5648, 1024), (7937, 3104, 2048), (2048, 8000, 192), (2049, 5680, 512)])
def test_plain_product_on_the_tile_gemm(M, N, K):
    """Column counts that end inside a tile, row counts that end behind one and in front of one, few k-tiles.  A sum of K products of bf16 in fp32
    is within K 2^-24 of the sum of their absolute values, and is rounded once (2^-8)."""
    import torch

    assert hops._tile_plain(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = (torch.randn(r, K, generator=g, device="cuda").to(torch.bfloat16) for r in (M, N))
    want, most = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((hops.linear(x, w).double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * most).all())
    xg = x.clone().requires_grad_()  # the library's product has a backward
    hops.linear(xg, w).sum().backward()
    assert xg.grad is not None
    wide = torch.cat([x, x], 1)[:, :K]  # rows of another stride
    assert torch.equal(hops.linear(wide, w), torch.nn.functional.linear(wide, w))


def test_transforms_and_tangents_are_seen():
    import torch
    import torch.autograd.forward_ad as fw

    x, w, seen = torch.randn(3, 4), torch.randn(2, 4), []
    f = lambda v: seen.append(hops._transformed(v, w)) or v * 2.0  # noqa: E731
    f(x)
    torch.func.vmap(f)(x)
    torch.func.jvp(f, (x,), (x,))
    with fw.dual_level():
        f(fw.make_dual(x, x))
        f(x)
    torch.jit.trace(f, (x,), check_trace=False)
    assert seen == [False, True, True, True, False, True]


@pytest.mark.gpu
def test_large_products_keep_tangents():
    """A product that the tile GEMM takes otherwise: torch's own where a tangent goes through it."""
    import torch
    import torch.autograd.forward_ad as fw

    M, N, K = 2304, 5648, 1024
    assert hops._tile_plain(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w, t = (torch.randn(r, K, generator=g, device="cuda").to(torch.bfloat16) for r in (M, N, M))
    with fw.dual_level():
        y = fw.unpack_dual(hops.linear(fw.make_dual(x, t), w))
    assert torch.equal(y.primal, torch.nn.functional.linear(x, w)) and torch.equal(y.tangent, torch.nn.functional.linear(t, w))
    y, dy = torch.func.jvp(lambda v: hops.linear(v, w), (x,), (t,))
    assert torch.equal(dy, torch.nn.functional.linear(t, w))
