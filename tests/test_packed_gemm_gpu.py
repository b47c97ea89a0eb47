"""The matrix-core product over F_2 / F_3 (hx_packed_gemm.hip) at the edges of its tiles, stages and K chunks,
against torch's float32 product of the unpacked entries (integers below 2^24: exact in any order)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pack(bits):
    m, n = bits.shape
    w = (n + 63) // 64
    full = torch.zeros((m, w * 64), dtype=torch.bool, device="cuda")
    full[:, :n] = bits
    full = full.view(m, w, 64)
    out = torch.zeros((m, w), dtype=torch.int64, device="cuda")
    for j in range(64):
        out |= full[:, :, j].to(torch.int64) << j
    return out


def _words(p, x):
    return _pack(x == 1) if p == 2 else torch.cat([_pack(x == 1), _pack(x == 2)], dim=1)


def _entries(p, m, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0, p, (m, n), generator=g, device="cuda", dtype=torch.int8)


def _product(p, a, b):
    signed = (lambda x: torch.where(x == 2, -1, x).float()) if p == 3 else (lambda x: x.float())
    return torch.remainder((signed(a) @ signed(b)).to(torch.int64), p).to(torch.int8)


@pytest.mark.parametrize("p", [2, 3])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (127, 65, 127), (128, 128, 128), (129, 129, 129), (130, 700, 385),
                                   (257, 383, 641), (200, 64, 1000),
                                   (4096, 4096, 200), (4100, 3841, 897),      # 256 x 256 tiles
                                   (100, 64, 4194304 + 77),                   # more than one K chunk
                                   (199800, 70, 64), (199900, 70, 64), (60, 210000, 33)])   # one word of k, long operands
def test_packed_gemm_edges(hx_gpu, p, m, n, k):
    from hacs_amd import engine as E
    mul = E.f2_gemm if p == 2 else E.f3_gemm
    print(f"F{p} product {m}x{n}x{k}", flush=True)
    a, b, c = _entries(p, m, k, 1), _entries(p, k, n, 2), _entries(p, m, n, 3)
    want = _product(p, a, b)
    A, B = _words(p, a), _words(p, b)
    C = _words(p, c)
    mul(A, B, C, k, n)
    assert torch.equal(C, _words(p, want))
    C = _words(p, c)
    mul(A, B, C, k, n, accumulate=True)
    assert torch.equal(C, _words(p, (want + c) % p))


@pytest.mark.parametrize("p", [2, 3])
def test_packed_gemm_captured(hx_gpu, p):
    """Inside a capture the table kernel runs (no library scratch in a graph): every replay on new operands."""
    from hacs_amd import engine as E
    mul = E.f2_gemm if p == 2 else E.f3_gemm
    m, n, k = 300, 200, 500
    A, B = _words(p, _entries(p, m, k, 1)), _words(p, _entries(p, k, n, 2))
    C = torch.zeros((m, B.shape[1]), dtype=torch.int64, device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        mul(A, B, C, k, n)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        mul(A, B, C, k, n)
    for seed in (5, 6, 7):
        a, b = _entries(p, m, k, seed), _entries(p, k, n, seed + 10)
        A.copy_(_words(p, a))
        B.copy_(_words(p, b))
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, _words(p, _product(p, a, b)))


def test_packed_gemm_past_the_grid_limit(hx_gpu):
    """An F_2 product of 2^23 tiles of 256 x 256 (69 GB of C): one launch cannot hold its threads, the table
    kernel runs it."""
    from hacs_amd import engine as E
    m, n, k = 1 << 20, 1 << 19, 70
    a, b = _entries(2, m, k, 1), _entries(2, k, n, 2)
    A, B = _words(2, a), _words(2, b)
    C = torch.zeros((m, n // 64), dtype=torch.int64, device="cuda")
    E.f2_gemm(A, B, C, k, n)
    for i0 in (0, 300000, m - 128):
        assert torch.equal(C[i0:i0 + 128], _words(2, _product(2, a[i0:i0 + 128], b)))
    del a, b, A, B, C
    torch.cuda.empty_cache()
