"""The automatic choice's residue route against the plain kernel over every operand form it accepts: the depths
where the rule switches, both tile sizes and their edges, orders, strides, unaligned bases and ops."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _draw(p, m, n, seed, form):
    """An m x n residue matrix: row-major, column-major, a window of a wider matrix (unaligned base), every
    second column."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda a, b: torch.randint(0, p, (a, b), generator=g, device="cuda").to(torch.int32)
    if form == "row":
        return r(m, n)
    if form == "col":
        return r(n, m).t()
    if form == "window":
        return r(m + 2, n + 5)[1:1 + m, 3:3 + n]
    return r(m, 2 * n)[:, ::2]


@pytest.mark.parametrize("p,n,k,route", [(2147483629, 2048, 767, 4), (2147483629, 2048, 768, 6), (4278124259, 1500, 1000, 6),
                                         (65521, 2048, 1535, 4), (65521, 1500, 1536, 6), (61001, 700, 2000, 4),
                                         (2147483629, 500, 1535, 4), (2147483629, 500, 1536, 6), (65521, 500, 2559, 4),
                                         (65521, 500, 2560, 6), (2147483629, 1024, 5000, 4), (65521, 256, 2000, 4),
                                         (65521, 256, 8192, 6), (65521, 256, 8193, 0)])
def test_auto_route_rule(p, n, k, route):
    from hacs_amd import engine as E
    assert E.gemm_route(E.ModCtx(p), n, n, k, E.HX_GEMM_AUTO) == route


@pytest.mark.parametrize("p", [251, 61001, 65521, 2147483629, 4278124259])
@pytest.mark.parametrize("m,n,k", [(200, 300, 129), (64, 64, 1000), (65, 129, 1023), (1000, 700, 500)])
def test_narrow_limb_tiles(hx_gpu, p, m, n, k):
    """Limb kernel 4 on 64 x 64 tiles (the default up to 128 wide tiles) against the wide ones (tile 4)."""
    from hacs_amd import engine as E
    ctx = E.ModCtx(p)
    A, B = _draw(p, m, k, 1, "row"), _draw(p, k, n, 2, "row")
    for op in (E.GemmOp.Set, E.GemmOp.Sub):
        C, D = _draw(p, m, n, 3, "row"), _draw(p, m, n, 3, "row")
        E.gemm(ctx, A, B, C, op, variant=E.HX_GEMM_LIMB)
        E.gemm(ctx, A, B, D, op, variant=E.HX_GEMM_LIMB, tile=4)
        assert torch.equal(C, D), op


@pytest.mark.parametrize("fa,fb,fc", [("row", "row", "row"), ("col", "col", "col"), ("window", "row", "window"),
                                      ("row", "window", "row"), ("step", "col", "step"), ("col", "step", "row")])
@pytest.mark.parametrize("p,m,n,k", [(2147483629, 515, 700, 1540), (65521, 640, 513, 2561), (1000003, 1025, 257, 2600),
                                     (2147483647, 1793, 2049, 833)])      # the last: 256 x 256 tiles
def test_auto_route_equals_plain(hx_gpu, p, m, n, k, fa, fb, fc):
    from hacs_amd import engine as E
    ctx = E.ModCtx(p)
    assert E.gemm_route(ctx, m, n, k, E.HX_GEMM_AUTO) == 6
    A, B = _draw(p, m, k, 1, fa), _draw(p, k, n, 2, fb)
    for op in (E.GemmOp.Set, E.GemmOp.Add, E.GemmOp.Sub):
        C, D = _draw(p, m, n, 3, fc), _draw(p, m, n, 3, fc)
        E.gemm(ctx, A, B, C, op)
        E.gemm(ctx, A, B, D, op, variant=E.HX_GEMM_PLAIN, splits=1)
        assert torch.equal(C, D), (fa, fb, fc, op)
    E.gemm_nt(ctx, A, _draw(p, k, n, 2, fb).t(), C)
    E.gemm(ctx, A, B, D, variant=E.HX_GEMM_PLAIN, splits=1)
    assert torch.equal(C, D)


@pytest.mark.parametrize("p", [251, 61001, 65521, 2147483629])
@pytest.mark.parametrize("m,n,k", [(16, 16, 15000), (16, 16, 16000), (8, 8, 60000), (4, 4, 140000), (16, 16, 8192), (3, 5, 300)])
def test_auto_deep_products_of_few_tiles(hx_gpu, p, m, n, k):
    """Both sides of the depth where few tiles are split over K, and of 4e6 multiply-adds."""
    from hacs_amd import engine as E
    ctx = E.ModCtx(p)
    A, B = _draw(p, m, k, 1, "row"), _draw(p, k, n, 2, "row")
    for op in (E.GemmOp.Set, E.GemmOp.Sub):
        C, D = _draw(p, m, n, 3, "row"), _draw(p, m, n, 3, "row")
        E.gemm(ctx, A, B, C, op)
        E.gemm(ctx, A, B, D, op, variant=E.HX_GEMM_PLAIN, splits=1)
        assert torch.equal(C, D), op


def test_residue_blocks_of_c(hx_gpu):
    """Planes past 8 GiB: C in blocks (ragged at both edges), the stream's scratch bounded, the limb kernel's bytes."""
    from hacs_amd import engine as E
    p, m, n, k = 2147483629, 31001, 29999, 801
    ctx = E.ModCtx(p)
    assert E.gemm_route(ctx, m, n, k, E.HX_GEMM_AUTO) == 6
    assert E.residue_moduli(p, k) * (m * n + (m + n) * k) > 8 << 30
    A, B = _draw(p, m, k, 1, "col"), _draw(p, k, n, 2, "row")
    s = torch.cuda.Stream()
    g = torch.Generator(device="cuda").manual_seed(3)
    C = torch.randint(0, p, (m, n), generator=g, device="cuda", dtype=torch.int32)
    D = C.clone()
    torch.cuda.synchronize()
    live = E.arena_stats()["live_bytes"]
    E.gemm(ctx, A, B, C, E.GemmOp.Sub, stream=s.cuda_stream)
    assert E.arena_stats()["live_bytes"] - live <= (8 << 30) + (260 << 20)
    s.synchronize()
    E.gemm(ctx, A, B, D, E.GemmOp.Sub, variant=E.HX_GEMM_LIMB, tile=4)
    assert torch.equal(C, D)
    del A, B, C, D
    torch.cuda.empty_cache()
