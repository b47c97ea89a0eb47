"""Automatic products inside a capture: where the plain kernel needs no scratch none is recorded, so the graph
stays good when a later, larger call on the stream replaces the library's planes."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

PR = 2147483629


def _rnd(m, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0, PR, (m, n), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)


def _capture(E, h, call):
    from hacs_amd import _lib
    g = C.c_void_p()
    _lib.check(_lib.lib().hx_graph_begin(h))
    call()
    _lib.check(_lib.lib().hx_graph_end(h, C.byref(g)))
    return g


@pytest.mark.parametrize("m,n,k", [(40, 40, 500), (3, 200, 1000), (64, 64, 257)])
def test_captured_auto_product_keeps_no_scratch(hx_gpu, m, n, k):
    from hacs_amd import _lib
    from hacs_amd import engine as E
    L, ctx = _lib.lib(), E.ModCtx(PR)
    A, B = _rnd(m, k, 1), _rnd(k, n, 2)
    X = torch.zeros((m, n), dtype=torch.int32, device="cuda")
    want = torch.zeros_like(X)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        h = s.cuda_stream
        E.gemm(ctx, A, B, want, stream=h)                        # grows this stream's planes
        s.synchronize()
        before = E.launch_stats()["limb_launches"]
        g = _capture(E, h, lambda: E.gemm(ctx, A, B, X, stream=h))
        assert E.launch_stats()["limb_launches"] == before       # the plain kernel: nothing of the library's kept
        big = _rnd(600, 2000, 3)
        out = torch.zeros((600, 600), dtype=torch.int32, device="cuda")
        E.gemm_nt(ctx, big, big, out, stream=h)                  # replaces the planes
        s.synchronize()
        ref = out.clone()
        for rep in range(3):
            X.fill_(-1)
            _lib.check(L.hx_graph_launch(g, h))
            s.synchronize()
            assert torch.equal(X, want), rep
            E.gemm_nt(ctx, big, big, out, stream=h)              # eager work between replays
            s.synchronize()
            assert torch.equal(out, ref), rep
        _lib.check(L.hx_graph_destroy(g))


def test_captured_auto_product_with_a_workspace(hx_gpu):
    """With a workspace of the caller's the captured product runs the reported kernel in it."""
    from hacs_amd import _lib
    from hacs_amd import engine as E
    L, ctx = _lib.lib(), E.ModCtx(PR)
    for m, n, k in [(40, 40, 500), (500, 500, 1600)]:
        assert E.gemm_route(ctx, m, n, k, E.HX_GEMM_AUTO) in (4, 6)
        A, B = _rnd(m, k, 1), _rnd(k, n, 2)
        X = torch.zeros((m, n), dtype=torch.int32, device="cuda")
        want = torch.zeros_like(X)
        E.gemm(ctx, A, B, want, variant=E.HX_GEMM_PLAIN, splits=1)
        ws = torch.empty(E.gemm_workspace_bytes(ctx, m, n, k, E.HX_GEMM_AUTO), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            h = s.cuda_stream
            before = E.launch_stats()["limb_launches"]
            g = _capture(E, h, lambda: E.gemm(ctx, A, B, X, stream=h, workspace=ws))
            assert E.launch_stats()["limb_launches"] == before + 1
            for rep in range(3):
                X.fill_(-1)
                _lib.check(L.hx_graph_launch(g, h))
                s.synchronize()
                assert torch.equal(X, want), rep
            _lib.check(L.hx_graph_destroy(g))
