"""Two host threads queue products with operands of their own on one stream, so both use that stream's library
scratch (split, product, product's read-back each a launch), and their growing sizes replace it in between: every
result is the one that the same call gives alone."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

ROUNDS = 24


def _residues(p, m, n, g):
    return torch.randint(0, p, (m, n), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)


def _words(P, m, n, g):
    """Random bit-packed rows (P = 2) or one-hot planes (P = 3); n is a multiple of 64."""
    w = torch.randint(-(1 << 63), (1 << 63) - 1, (m, n // 64), generator=g, device="cuda", dtype=torch.int64)
    if P == 2:
        return w
    v = torch.randint(-(1 << 63), (1 << 63) - 1, (m, n // 64), generator=g, device="cuda", dtype=torch.int64)
    return torch.cat([w & ~v, v & ~w], dim=1)


def _calls(E, kind, seed):
    """One thread's calls: [(call, the output it writes)], sizes growing."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for i in range(ROUNDS):
        s = 64 * (1 + i // 2) + 64 * (seed % 2)
        if kind in ("f2", "f3"):
            P = 2 if kind == "f2" else 3
            A, B = _words(P, s, 2 * s, g), _words(P, 2 * s, s, g)
            C = torch.zeros((s, s // 64 * (P - 1)), dtype=torch.int64, device="cuda")
            mul = E.f2_gemm if P == 2 else E.f3_gemm
            out.append((lambda st, A=A, B=B, C=C, k=2 * s, n=s, mul=mul: mul(A, B, C, k, n, stream=st), C))
        elif kind == "u64":
            p = 2305843009213693951
            A, B = (torch.randint(0, p, sh, generator=g, device="cuda", dtype=torch.int64) for sh in ((s, 2 * s), (2 * s, s)))
            C = torch.zeros((s, s), dtype=torch.int64, device="cuda")
            out.append((lambda st, A=A, B=B, C=C, c=E.ModCtx64(p): E.gemm_u64(c, A, B, C, stream=st), C))
        else:
            p = 2147483629
            m, k = (40, 400 + 20 * i) if kind == "gemm_small" else (s, 800 + 100 * i)      # limb planes; also residue planes
            A, B = _residues(p, m, k, g), _residues(p, k, m, g)
            C = torch.zeros((m, m), dtype=torch.int32, device="cuda")
            out.append((lambda st, A=A, B=B, C=C, c=E.ModCtx(p): E.gemm(c, A, B, C, stream=st), C))
    return out


@pytest.mark.parametrize("kind", ["f2", "f3", "u64", "gemm_small", "gemm"])
def test_two_threads_one_stream(hx_gpu, kind):
    from hacs_amd import engine as E
    work = [_calls(E, kind, seed) for seed in (1, 2)]
    torch.cuda.synchronize()
    alone = []
    for calls in work:                       # on the default stream, one after the other
        for call, C in calls:
            call(0)
        torch.cuda.synchronize()
        alone.append([C.clone() for _, C in calls])
        for _, C in calls:
            C.fill_(-1)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()             # its scratch grows as the calls below do
    start, errors = threading.Barrier(2), []

    def run(calls):
        try:
            start.wait()
            for call, _ in calls:
                call(stream.cuda_stream)
        except Exception as e:               # noqa: BLE001  (shown by the test's thread)
            errors.append(e)

    threads = [threading.Thread(target=run, args=(calls,)) for calls in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    stream.synchronize()
    assert not errors, errors
    for t, (calls, want) in enumerate(zip(work, alone)):
        for i, ((_, C), W) in enumerate(zip(calls, want)):
            assert torch.equal(C, W), f"{kind}: thread {t}, call {i}"
