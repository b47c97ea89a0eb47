"""GEMM mod p on 64-bit residues (hx_gemm_u64) against the oracle's exact unsigned __int128 product
(itself equal to the reference's kernels::gemm<uint64_t>, tests/test_oracle.py): the moduli of the
reference's u64 gates (2^61 - 1, KernelBitIdentityValidation.cpp:520-604) and 2^64 - 59, moduli just
above 2^32 and 2^63, an even modulus (the long-division epilogue), every op, ragged and strided
views, k = 0, and the all-(p-1) worst case over a K that fills the 160-bit accumulator's top word."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

PRIMES = [2305843009213693951, 18446744073709551557, 4294967311, 9223372036854775837, (1 << 64) - 2, 7]


def _draw(rng, p, shape):
    return ((rng.integers(0, 1 << 32, shape, dtype=np.uint64) << np.uint64(32)) |
            rng.integers(0, 1 << 32, shape, dtype=np.uint64)) % np.uint64(p)


@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 17, 33), (64, 64, 64), (65, 129, 300), (130, 70, 17), (3, 5, 0)])
def test_gemm_u64_matches_oracle(hx_gpu, O, p, shape):
    from hacs_amd import engine as E
    ctx = E.ModCtx64(p)
    m, n, k = shape
    rng = np.random.default_rng((p ^ (m * 1000003 + n * 1009 + k)) & 0xFFFFFFFF)
    A, B, C0 = _draw(rng, p, (m, k)), _draw(rng, p, (k, n)), _draw(rng, p, (m, n))
    dA, dB = E.to_device64(A), E.to_device64(B)
    for op in (0, 1, 2):
        dC = E.to_device64(C0)
        E.gemm_u64(ctx, dA, dB, dC, op)
        torch.cuda.synchronize()
        want = O.gemm_u64(p, A, B, C0, op, 16) if k else (np.zeros_like(C0) if op == 0 else C0)
        assert np.array_equal(E.from_device64(dC), want), f"op {op}"


def test_gemm_u64_strided_views(hx_gpu, O):
    """A transposed (column-major) A, a strided window of B and C."""
    from hacs_amd import engine as E
    p = 18446744073709551557
    ctx = E.ModCtx64(p)
    rng = np.random.default_rng(5)
    m, n, k = 90, 75, 130
    At = _draw(rng, p, (k, m))
    Bbig = _draw(rng, p, (k + 3, n + 9))
    Cbig = _draw(rng, p, (m + 4, n + 6))
    dAt, dBbig, dCbig = E.to_device64(At), E.to_device64(Bbig), E.to_device64(Cbig)
    E.gemm_u64(ctx, dAt.t(), dBbig[2:2 + k, 5:5 + n], dCbig[1:1 + m, 3:3 + n], 2)
    torch.cuda.synchronize()
    want = Cbig.copy()
    want[1:1 + m, 3:3 + n] = O.gemm_u64(p, At.T.copy(), Bbig[2:2 + k, 5:5 + n].copy(), Cbig[1:1 + m, 3:3 + n].copy(), 2)
    assert np.array_equal(E.from_device64(dCbig), want)


@pytest.mark.parametrize("p", [18446744073709551557, (1 << 64) - 2, 2305843009213693951])
def test_gemm_u64_worst_case_carries(hx_gpu, O, p):
    """Every entry p - 1 over K = 70000: each product is nearly 2^128, so the sum's top word counts up to
    K; the result is the closed form K (p - 1)^2 = K mod p."""
    from hacs_amd import engine as E
    ctx = E.ModCtx64(p)
    K = 70000
    dA = E.to_device64(np.full((8, K), p - 1, np.uint64))
    dB = E.to_device64(np.full((K, 72), p - 1, np.uint64))
    dC = torch.zeros((8, 72), dtype=torch.int64, device="cuda")
    E.gemm_u64(ctx, dA, dB, dC, 0)
    torch.cuda.synchronize()
    assert (E.from_device64(dC) == np.uint64(K % p)).all()


@pytest.mark.parametrize("p", [2305843009213693951, 18446744073709551557, (1 << 64) - 2, 4294967311])
@pytest.mark.parametrize("shape", [(128, 128, 64), (129, 127, 65), (255, 300, 129), (1, 700, 1000), (700, 1, 1000),
                                   (1400, 1500, 70),                               # 256 x 256 tiles
                                   (10, 20001, 64), (10, 20001, 96), (34, 4097, 64), (1001, 999, 40)])   # either side of the rule below k = 96
def test_gemm_u64_residue_route(hx_gpu, O, p, shape):
    """The matrix-core route at the edges of its tiles, row- and column-major operands, every op."""
    from hacs_amd import engine as E
    ctx = E.ModCtx64(p)
    m, n, k = shape
    rng = np.random.default_rng((p ^ (m * 1000003 + n * 1009 + k)) & 0xFFFFFFFF)
    A, B, C0 = _draw(rng, p, (m, k)), _draw(rng, p, (k, n)), _draw(rng, p, (m, n))
    A[0, :] = p - 1
    B[:, 0] = p // 2
    want = [O.gemm_u64(p, A, B, C0, op, 16) for op in (0, 1, 2)]
    At = E.to_device64(np.ascontiguousarray(A.T)).t()
    Bt = E.to_device64(np.ascontiguousarray(B.T)).t()
    for dA, dB, op in ((E.to_device64(A), E.to_device64(B), 0), (At, Bt, 1), (At, E.to_device64(B), 2)):
        dC = E.to_device64(C0)
        E.gemm_u64(ctx, dA, dB, dC, op)
        torch.cuda.synchronize()
        assert np.array_equal(E.from_device64(dC), want[op]), f"op {op}"


@pytest.mark.parametrize("p", [18446744073709551557, 2305843009213693951])
@pytest.mark.parametrize("m,n,k", [(40, 200, 133056 + 77), (1500, 300, 133000)])
def test_gemm_u64_residue_chunks(hx_gpu, p, m, n, k):
    """K past one chunk of int32 sums; C in blocks (planes past the workspace bound).  B holds three entries
    per column, so every result is three products."""
    from hacs_amd import engine as E
    rng = np.random.default_rng(m + n)
    dA = torch.randint(0, 1 << 62, (m, k), device="cuda", dtype=torch.int64) % (p >> 3)
    rows = np.stack([rng.choice(k, 3, replace=False) for _ in range(n)])
    coef = _draw(rng, p, (n, 3))
    B = np.zeros((k, n), np.uint64)
    for e in range(3):
        B[rows[:, e], np.arange(n)] = coef[:, e]
    cols = E.from_device64(dA[:, torch.from_numpy(rows.reshape(-1)).cuda()]).reshape(m, n, 3)
    want = np.array([sum(int(cols[i, j, e]) * int(coef[j, e]) for e in range(3)) % p
                     for i in range(m) for j in range(n)], np.uint64).reshape(m, n)
    dC = torch.zeros((m, n), dtype=torch.int64, device="cuda")
    E.gemm_u64(E.ModCtx64(p), dA, E.to_device64(B), dC, 1)
    torch.cuda.synchronize()
    assert np.array_equal(E.from_device64(dC), want)


def test_gemm_u64_captured(hx_gpu, O):
    """A captured product (the plain kernel: no library scratch in a graph) replayed on new operands."""
    from hacs_amd import engine as E
    p, m, n, k = 2305843009213693951, 150, 140, 160
    ctx = E.ModCtx64(p)
    rng = np.random.default_rng(3)
    dA, dB = (torch.zeros(s, dtype=torch.int64, device="cuda") for s in ((m, k), (k, n)))
    dC = torch.zeros((m, n), dtype=torch.int64, device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        E.gemm_u64(ctx, dA, dB, dC)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        E.gemm_u64(ctx, dA, dB, dC)
    for _ in range(3):
        A, B = _draw(rng, p, (m, k)), _draw(rng, p, (k, n))
        dA.copy_(E.to_device64(A))
        dB.copy_(E.to_device64(B))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(E.from_device64(dC), O.gemm_u64(p, A, B, np.zeros((m, n), np.uint64), 0, 16))
