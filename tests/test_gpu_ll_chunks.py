"""The likelihood and its adjoint over more than one chunk of samples: the
per-sample values of separate calls on slices that are cut elsewhere, and the
sums of their gradients.  The last chunk is neither full nor a multiple of 64
samples; shapes within one workgroup, through the three-pass split and with
padded channels."""
import pytest
import torch

import cudamica_amd as ca
from tests.test_gpu_ll_nan import _model

pytestmark = pytest.mark.gpu


def _call(bits, x, dll, p, n, M, m):
    T = x.shape[0]
    addr = {k: v.data_ptr() for k, v in p.items()}
    stream = torch.cuda.current_stream().cuda_stream
    fwd = torch.full((T,), float("nan"), dtype=torch.float64, device="cuda")
    ll = torch.full((T,), float("nan"), dtype=torch.float64, device="cuda")
    g = {k: torch.full_like(v, float("nan")) for k, v in p.items()}
    ca.ll_forward(bits, x.data_ptr(), T, n, M, m, addr, 0.1, fwd.data_ptr(), stream)
    ca.ll_adjoint(bits, x.data_ptr(), T, n, M, m, addr, 0.1, dll.data_ptr(), {k: v.data_ptr() for k, v in g.items()},
                  ll.data_ptr(), stream)
    return fwd, ll, g


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,T,M,m", [(128, 140_003, 4, 2), (64, 600_001, 1, 3), (1000, 23_001, 2, 2),
                                     (50, 300_007, 3, 1)])
def test_chunks_add_up(built, bits, n, T, M, m):
    # samples per chunk of the adjoint: 256 MiB of b, g and (n < NP) padded x; at least 4096
    NP = (n + 63) // 64 * 64
    most = max(4096, (256 << 20) // (bits // 8 * (2 * M * NP + (NP if n < NP else 0))))
    assert T > most
    print(f"[ll chunks] n={n} T={T} M={M} m={m} FP{bits}", flush=True)
    p = _model(n, M, m, n + T)
    gen = torch.Generator("cuda").manual_seed(T)
    s = torch.randn((T, n), generator=gen, device="cuda", dtype=torch.float64)
    x = (torch.sign(s) * s.abs().pow(1.4)).to(torch.float64 if bits == 64 else torch.float32)
    dll = 0.5 + torch.rand(T, generator=gen, device="cuda", dtype=torch.float64)
    fwd, ll, g = _call(bits, x, dll, p, n, M, m)
    cut = [0, 1, *range(1 + 7 * most // 10, T, 7 * most // 10), T]       # one chunk each
    ref = {k: torch.zeros_like(v) for k, v in p.items()}
    size = dict.fromkeys(p, 0.0)
    fwds, lls = [], []
    for a, b in zip(cut, cut[1:]):
        f1, l1, g1 = _call(bits, x[a:b].clone(), dll[a:b].clone(), p, n, M, m)
        fwds.append(f1)
        lls.append(l1)
        for k in ref:
            ref[k] += g1[k]
            size[k] += float(torch.linalg.vector_norm(g1[k]))
    # the rounding of b, which the forward has against the allocation-free call
    ll_tol = 1e-12 if bits == 64 else 2e-6
    assert float(((torch.cat(fwds) - fwd) / fwd).abs().max()) <= ll_tol
    assert float(((torch.cat(lls) - ll) / ll).abs().max()) <= ll_tol
    # the same terms in another grouping: the bars the variants have against
    # the oracle and against each other
    for k in ref:
        err = float(torch.linalg.vector_norm(g[k] - ref[k])) / size[k]
        print(f"  d{k}: {err:.1e}", flush=True)
        assert err <= (1e-10 if bits == 64 else 1e-4), k
