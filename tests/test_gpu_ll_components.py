"""The adjoint with five to eight components, whose tiles hold one or two
samples, against FP64 autograd of the plain formula; and allocation-free calls
whose ranges of samples take more than one 16-sample tile and end inside one."""
import numpy as np
import pytest
import torch

import cudamica_amd as ca
from tests.test_gpu_ll_nan import _model

pytestmark = pytest.mark.gpu

LOG2 = 0.693147180559945


def _plain(x, p, M):
    L = []
    for h in range(M):
        W = p["W"][h].T                                       # column-major
        b = (x - p["c"][h]) @ W.T
        y = (p["beta"][h].sqrt() * (b[:, None, :] - p["mu"][h])).abs()
        Q = (p["alpha"][h].log() + 0.5 * p["beta"][h].log() - LOG2 - torch.lgamma(1.0 + 1.0 / p["rho"][h])
             - y.pow(p["rho"][h]))
        L.append(p["gm"][h].log() + torch.linalg.slogdet(W)[1] + torch.logsumexp(Q, 1).sum(1))
    return torch.logsumexp(torch.stack(L), 0)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,T,M,m", [(16, 1501, 2, 5), (70, 1202, 1, 6), (33, 1003, 3, 7), (64, 1001, 1, 8),
                                     (130, 907, 3, 6), (200, 803, 3, 8)])
def test_adjoint_of_many_components(built, bits, n, T, M, m):
    print(f"[ll components] n={n} T={T} M={M} m={m} FP{bits}", flush=True)
    p = _model(n, M, m, 31 * n + m)
    x = torch.tensor(np.random.default_rng(n * m).laplace(size=(T, n)).astype(np.float32), device="cuda")
    x = x.double() if bits == 64 else x
    dll = torch.tensor(np.random.default_rng(m).uniform(0.5, 1.5, T), device="cuda")
    ll = torch.empty(T, dtype=torch.float64, device="cuda")
    g = {k: torch.empty_like(v) for k, v in p.items()}
    ca.ll_adjoint(bits, x.data_ptr(), T, n, M, m, {k: v.data_ptr() for k, v in p.items()}, 0.0, dll.data_ptr(),
                  {k: v.data_ptr() for k, v in g.items()}, ll.data_ptr(), torch.cuda.current_stream().cuda_stream)
    leaf = {k: v.cpu().requires_grad_() for k, v in p.items()}
    ref = _plain(x.cpu().double(), leaf, M)
    (dll.cpu() * ref).sum().backward()
    # the bars the FP64 and FP32 variants have against the oracle and each other
    tol, ll_tol = (1e-10, 1e-12) if bits == 64 else (1e-4, 1e-5)
    ref = ref.detach()
    assert float(((ll.cpu() - ref) / ref).abs().max()) <= ll_tol
    for k in p:
        err = float(torch.linalg.vector_norm(g[k].cpu() - leaf[k].grad) / torch.linalg.vector_norm(leaf[k].grad))
        print(f"  d{k}: {err:.1e}", flush=True)
        assert err <= tol, k


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,M,ranges,extra", [(40, 1, 4096, 37), (64, 8, 512, 21), (100, 2, 1024, 18)])
def test_allocation_free_ranges_of_several_tiles(built, bits, n, M, ranges, extra):
    """`ranges` is the most ranges a call of these shapes is cut into on 256 CUs (16
    waves per CU); `extra` samples each leave the second or third 16-sample tile of
    a range partly filled."""
    T, m = ranges * extra - 5, 2
    print(f"[ll noalloc ranges] n={n} T={T} M={M} FP{bits}", flush=True)
    p = _model(n, M, m, n)
    addr = {k: v.data_ptr() for k, v in p.items()}
    gen = torch.Generator("cuda").manual_seed(n)
    x = torch.randn((T, n), generator=gen, device="cuda", dtype=torch.float64 if bits == 64 else torch.float32)
    out = []
    stream = torch.cuda.current_stream().cuda_stream
    for call in (ca.ll_forward_noalloc, ca.ll_forward):
        ll = torch.full((T,), float("nan"), dtype=torch.float64, device="cuda")
        call(bits, x.data_ptr(), T, n, M, m, addr, 0.0, ll.data_ptr(), stream)
        torch.cuda.synchronize()
        out.append(ll)
    rel = float(((out[0] - out[1]) / out[1]).abs().max())
    print(f"  max per-sample relative difference {rel:.2e}", flush=True)
    assert rel <= (1e-12 if bits == 64 else 2e-6)
