"""Products of small depth and small products (hx_thin.hip, the automatic choice) against the plain kernel: the
edges of its 32-row blocks, 128-column workgroups and 32 / 64-deep k-steps, every limb count, the largest
balanced entries, the largest digits (test_thin_largest_digits: the anti-diagonals at their bounds), orders, strides
and ops."""
import pytest
import torch

pytestmark = pytest.mark.gpu

P = [2, 251, 257, 65279, 65521, 16711423, 16777213, 1000003, 2147483629, 2147483647]


def _draw(p, m, n, seed, form="row", extreme=False):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def r(a, b):
        if extreme:      # p // 2 and p // 2 + 1: balanced +-p/2
            return ((p // 2 + torch.randint(0, 2, (a, b), generator=g, device="cuda")) % p).to(torch.int32)
        return torch.randint(0, p, (a, b), generator=g, device="cuda").to(torch.int32)
    if form == "row":
        return r(m, n)
    if form == "col":
        return r(n, m).t()
    if form == "window":
        return r(m + 2, n + 5)[1:1 + m, 3:3 + n]
    return r(m, 2 * n)[:, ::2]


def _check(E, ctx, A, B, C, what):
    for op in (E.GemmOp.Set, E.GemmOp.Add, E.GemmOp.Sub):
        X, D = C(), C()
        E.gemm(ctx, A, B, X, op)
        E.gemm(ctx, A, B, D, op, variant=E.HX_GEMM_PLAIN, splits=1)
        assert torch.equal(X, D), (what, op)


@pytest.mark.parametrize("p", P)
@pytest.mark.parametrize("m,n,k", [(32, 32, 1), (33, 127, 31), (31, 129, 32), (100, 200, 33), (1, 4096, 64), (4096, 1, 63),
                                   (65, 128, 65), (70, 90, 129), (40, 50, 500), (2050, 2111, 40), (140001, 20, 31)])
def test_thin_shapes(hx_gpu, p, m, n, k):
    from hacs_amd import engine as E
    ctx = E.ModCtx(p)
    assert (E.gemm_route(ctx, m, n, k, E.HX_GEMM_AUTO) == 7) == (k <= 256)       # (past it: the limb kernel)
    for extreme in (False, True):
        A, B = _draw(p, m, k, 1, extreme=extreme), _draw(p, k, n, 2, extreme=extreme)
        if extreme:
            A[:, ::2] = p // 2              # sums of one sign along the depth
            B[:, ::2] = p // 2
        _check(E, ctx, A, B, lambda: _draw(p, m, n, 3), (p, m, n, k, extreme))


@pytest.mark.parametrize("fa,fb,fc", [("col", "col", "col"), ("window", "row", "window"), ("row", "window", "step"),
                                      ("step", "col", "row"), ("col", "step", "col")])
@pytest.mark.parametrize("p,m,n,k", [(2147483629, 150, 301, 30), (65521, 301, 150, 64), (1000003, 61, 75, 200)])
def test_thin_forms(hx_gpu, p, m, n, k, fa, fb, fc):
    from hacs_amd import engine as E
    assert E.gemm_route(E.ModCtx(p), m, n, k, E.HX_GEMM_AUTO) == 7
    _check(E, E.ModCtx(p), _draw(p, m, k, 1, fa), _draw(p, k, n, 2, fb), lambda: _draw(p, m, n, 3, fc), (fa, fb, fc))


def _digits(v, p):
    """The balanced base-256 digits of the residue v."""
    v, out = v - p if v > (p - 1) // 2 else v, []
    for _ in range(4):
        d = (v + 128) % 256 - 128
        out.append(d)
        v = (v - d) // 256
    assert v == 0
    return out


@pytest.mark.parametrize("k", [31, 32, 63, 64, 200])
@pytest.mark.parametrize("p,pos,neg", [
    (2147483647, 0x3F7F7F7F, 0x3F808080),        # digits 127, 127, 127, 63 and -128, -128, -128, -63
    (2147483629, 0x3F7F7F7F, 0x3F808080),
    (16777259, 0x7F7F7F, 0x7E8080),              # four limbs at their smallest modulus
    (16711423, 0x7F7F7F, 0x7E8080), (65279, 0x7F7F, 0x7E80), (251, 125, 125)])
def test_thin_largest_digits(hx_gpu, p, pos, neg, k):
    """Every digit at the end of its range, all products of one anti-diagonal with one sign: the sums and the
    pairs of sums of the kernel (and of the eliminations' updates, the same reduction) at their bounds."""
    from hacs_amd import engine as E
    ctx, m, n = E.ModCtx(p), 40, 70
    assert E.gemm_route(ctx, m, n, k, E.HX_GEMM_AUTO) == 7
    vals = (pos, p - neg)
    if p > 251:                              # (the digits that the modulus leaves free)
        assert set(_digits(vals[0], p)[:ctx.c.limbs - 1]) == {127}
        assert set(_digits(vals[1], p)[:min(2, ctx.c.limbs - 1)]) == {-128}
    for x in vals:
        for y in vals:
            A = torch.full((m, k), x, dtype=torch.int64, device="cuda").to(torch.int32)
            B = torch.full((k, n), y, dtype=torch.int64, device="cuda").to(torch.int32)
            C = torch.zeros((m, n), dtype=torch.int32, device="cuda")
            E.gemm(ctx, A, B, C)
            assert (C == k * x * y % p).all(), (x, y)
            E.gemm(ctx, A, B, C, E.GemmOp.Sub)
            assert (C == 0).all(), (x, y)
