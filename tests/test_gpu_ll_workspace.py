"""The device memory that the likelihood and adjoint calls keep between calls:
it goes back on request and where an engine's allocation fails."""
import pytest
import torch

import cudamica_amd as ca
from tests.test_gpu_ll_nan import _model

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _forward(n, T, M=1, m=2):
    p = _model(n, M, m, n)
    x = torch.randn((T, n), device="cuda")
    ll = torch.empty(T, dtype=torch.float64, device="cuda")
    ca.ll_forward(32, x.data_ptr(), T, n, M, m, {k: v.data_ptr() for k, v in p.items()}, 0.0, ll.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()


def test_the_kept_workspace_goes_back_on_request(built):
    print("[ll workspace] release", flush=True)
    n, T = 64, 400_000                      # b alone is 98 MiB; the runtime's own memory moves by a few
    _forward(n, T)
    kept = torch.cuda.mem_get_info()[0]
    ca.ll_release_workspace()
    assert torch.cuda.mem_get_info()[0] - kept >= 90 * MIB
    _forward(n, T)                          # and is taken again where needed


def test_the_kept_workspace_goes_back_for_an_engine(built):
    """An engine that does not fit (whitened data of 1.4 times the GPU's memory) fails,
    but not for the sake of an idle workspace."""
    print("[ll workspace] engine allocation", flush=True)
    n, T = 64, 400_000
    _forward(n, T)
    kept, total = torch.cuda.mem_get_info()
    with pytest.raises(ca.EngineError, match="hipMalloc") as err:
        ca.Engine(ca.options(n, int(1.4 * total) // (4 * n), 1, 2))
    print(" ", err.value, flush=True)
    assert torch.cuda.mem_get_info()[0] - kept >= 90 * MIB


def test_threads_and_streams_share_the_pool(built):
    """Four threads on a stream each, more than the pool has blocks, with calls of
    different sizes in turn: the bits of the same calls one after another."""
    import threading
    print("[ll workspace] threads", flush=True)
    n, M, m = 48, 2, 3
    p = _model(n, M, m, n)
    addr = {k: v.data_ptr() for k, v in p.items()}
    xs = [torch.randn((20_000 + 7001 * k, n), device="cuda", dtype=torch.float64) for k in range(4)]
    dll = torch.ones(60_000, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()

    def calls(k, stream):
        out = []
        for r in range(3):
            x = xs[(k + r) % 4]
            ll = torch.empty(x.shape[0], dtype=torch.float64, device="cuda")
            g = {q: torch.empty_like(v) for q, v in p.items()}
            torch.cuda.synchronize()
            ca.ll_adjoint(64, x.data_ptr(), x.shape[0], n, M, m, addr, 0.0, dll.data_ptr(),
                          {q: v.data_ptr() for q, v in g.items()}, ll.data_ptr(), stream.cuda_stream)
            out += [ll, *g.values()]
        return out

    want = [calls(k, torch.cuda.current_stream()) for k in range(4)]
    got = [None] * 4

    def work(k):
        got[k] = calls(k, torch.cuda.Stream())

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(want, got):
        assert b is not None and all(torch.equal(u, v) for u, v in zip(a, b))


def _adjoint_block(n, T, M):
    """Device memory an adjoint call (FP64, one component) leaves in the pool."""
    p = _model(n, M, 1, n)
    x = torch.randn((T, n), device="cuda", dtype=torch.float64)
    dll = torch.ones(T, device="cuda", dtype=torch.float64)
    g = {k: torch.empty_like(v) for k, v in p.items()}
    ca.ll_release_workspace()
    before = torch.cuda.mem_get_info()[0]
    ca.ll_adjoint(64, x.data_ptr(), T, n, M, 1, {k: v.data_ptr() for k, v in p.items()}, 0.0, dll.data_ptr(),
                  {k: v.data_ptr() for k, v in g.items()}, 0, torch.cuda.current_stream().cuda_stream)
    return before - torch.cuda.mem_get_info()[0]


def test_the_workspace_does_not_grow_with_the_samples(built):
    """One chunk of 8000 samples (250 MiB of b and g), and eight of them: the
    sums of a chunk (16 MiB of them here) are not kept beside each other."""
    print("[ll workspace] chunks", flush=True)
    n, M = 1024, 2
    one = _adjoint_block(n, 8000, M)
    assert one >= 250 * MIB
    assert _adjoint_block(n, 8 * 8000, M) <= one + 2 * MIB
