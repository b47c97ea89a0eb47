"""The automatic choice of the product's kernel, by its public queries (host arithmetic, no device)."""
import pytest

from hacs_amd import engine as E

P = {1: 251, 2: 61001, 3: 65521, 4: 2147483629}          # a modulus of each limb count


@pytest.mark.parametrize("limbs", [1, 2, 3, 4])
def test_deep_products_of_few_tiles_split(limbs):
    """The few tiles of a deep narrow product would run all of K in series: it splits over K on the plain kernel
    past k = 8192 from 4e6 multiply-adds on, below past k = 12288 (not with one limb), past the residue route's
    depth too."""
    c = E.ModCtx(P[limbs])
    for m, n, k in [(16, 16, 16000), (256, 256, 16384), (200, 100, 140000), (32, 32, 8193)]:
        assert E.gemm_route(c, m, n, k, E.HX_GEMM_AUTO) == 0, (m, n, k)
    for m, n, k in [(16, 16, 15000), (8, 8, 60000), (4, 4, 200000), (1, 1, 12289)]:
        assert E.gemm_route(c, m, n, k, E.HX_GEMM_AUTO) == (4 if limbs == 1 else 0), (m, n, k)
    for m, n, k in [(16, 16, 8192), (1, 1, 12288), (1, 1, 300), (8, 8, 257), (64, 64, 8192)]:
        assert E.gemm_route(c, m, n, k, E.HX_GEMM_AUTO) in (4, 6), (m, n, k)


@pytest.mark.parametrize("limbs", [1, 2, 3, 4])
def test_workspace_follows_the_route(limbs):
    """hx_gemm_workspace_bytes(AUTO) is zero exactly where the reported kernel needs no planes, and else serves
    that kernel."""
    c = E.ModCtx(P[limbs])
    for m, n, k in [(8, 8, 8), (40, 40, 500), (40, 40, 257), (40, 40, 256), (300, 300, 64), (300, 300, 65),
                    (16, 16, 15000), (1024, 1024, 1024), (2048, 2048, 2048), (256, 256, 16384), (4096, 34, 2000)]:
        route = E.gemm_route(c, m, n, k, E.HX_GEMM_AUTO)
        got = E.gemm_workspace_bytes(c, m, n, k, E.HX_GEMM_AUTO)
        if route in (0, 7):
            assert got == 0, (m, n, k)
        elif route == 6:
            assert got == E.gemm_workspace_bytes(c, m, n, k, E.HX_GEMM_LIMB, tile=6), (m, n, k)
        else:
            assert got == E.gemm_workspace_bytes(c, m, n, k, E.HX_GEMM_LIMB, tile=4) > 0, (m, n, k)


@pytest.mark.parametrize("p,m,n,k,route", [
    # long narrow products: the residue planes' passes and padding cost more than the multiply-adds they save
    (2147483629, 34, 8192, 2000, 4), (2147483629, 8192, 34, 3000, 4), (2147483629, 20000, 34, 3000, 4),
    (2147483629, 34, 40000, 3000, 4), (2147483629, 1, 8192, 3000, 4), (2147483629, 64, 4096, 5000, 4),
    (2147483629, 129, 20000, 1600, 4), (65521, 129, 20000, 1600, 4), (65521, 34, 40000, 3000, 4),
    (2147483629, 300, 7000, 4096, 4), (2147483629, 384, 20000, 2048, 4),
    # and where they do not
    (2147483629, 100, 2000, 3000, 6), (2147483629, 1000, 34, 5000, 6), (2147483629, 512, 4200, 2048, 6),
    (2147483629, 1677, 1419, 2049, 6), (2147483629, 700, 3000, 2560, 6), (16777213, 20000, 200, 8192, 6),
    (65521, 8192, 8192, 4096, 6), (2147483629, 8192, 8192, 1024, 6)])
def test_residue_route_by_shape(p, m, n, k, route):
    assert E.gemm_route(E.ModCtx(p), m, n, k, E.HX_GEMM_AUTO) == route


def test_residue_planes_are_bounded():
    """The default and the automatic choice run C in blocks of at most 8 GiB of residue planes; a tile the caller
    asks for keeps its one-piece formula."""
    c = E.ModCtx(P[4])
    for m, n, k in [(32768, 32768, 1024), (60000, 60000, 5000), (2000000, 2000, 800), (1500, 3000000, 1536), (100000, 100000, 133000)]:
        for variant in (E.HX_GEMM_AUTO, E.HX_GEMM_LIMB):
            if E.gemm_route(c, m, n, k, variant) == 6:
                assert 0 < E.gemm_workspace_bytes(c, m, n, k, variant) <= 8 << 30, (m, n, k)
        assert E.gemm_route(c, m, n, k, E.HX_GEMM_AUTO) == 6
    assert E.gemm_workspace_bytes(c, 16384, 16384, 16384, E.HX_GEMM_AUTO) == 10 * 3 * 16384 * 16384
    N = E.residue_moduli(c.p, 1024)
    assert E.gemm_workspace_bytes(c, 32768, 32768, 1024, E.HX_GEMM_LIMB, tile=6) == N * (2 * 32768 * 1024 + 32768 * 32768)
