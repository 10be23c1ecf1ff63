"""A sample that holds a NaN has no likelihood: its ll_t is NaN and every other
sample's is what it is without it, in every form of the likelihood (one
workgroup with one and with several models, the three-pass split, the
allocation-free call)."""
import numpy as np
import pytest
import torch

import cudamica_amd as ca

pytestmark = pytest.mark.gpu


def _model(n, M, m, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(0.5, 1.5, (M, m, n))
    vals = dict(W=np.eye(n) + 0.3 / np.sqrt(n) * rng.standard_normal((M, n, n)), c=0.1 * rng.standard_normal((M, n)),
                alpha=a / a.sum(1, keepdims=True), mu=rng.standard_normal((M, m, n)),
                beta=rng.uniform(0.5, 1.5, (M, m, n)), rho=rng.uniform(1.1, 1.9, (M, m, n)), gm=np.full(M, 1.0 / M))
    return {k: torch.tensor(v, dtype=torch.float64, device="cuda").contiguous() for k, v in vals.items()}


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,M,noalloc", [(40, 1, False), (70, 3, False), (300, 2, False), (40, 1, True),
                                         (64, 4, True)])
def test_a_nan_sample_scores_nan(built, bits, n, M, noalloc):
    print(f"[ll nan] n={n} M={M} FP{bits} {'noalloc' if noalloc else ''}", flush=True)
    T, m = 203, 3
    p = _model(n, M, m, n + M)
    addr = {k: v.data_ptr() for k, v in p.items()}
    x = torch.tensor(np.random.default_rng(n).laplace(size=(T, n)), device="cuda",
                     dtype=torch.float64 if bits == 64 else torch.float32)
    call = ca.ll_forward_noalloc if noalloc else ca.ll_forward
    got = []
    bad = [6, 100, T - 1]
    for poison in (False, True):
        if poison:
            for t in bad:
                x[t, (7 * t) % n] = float("nan")
        ll = torch.zeros(T, dtype=torch.float64, device="cuda")
        call(bits, x.data_ptr(), T, n, M, m, addr, 0.0, ll.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got.append(ll.cpu().numpy())
    assert np.all(np.isfinite(got[0]))
    assert np.all(np.isnan(got[1][bad]))
    good = np.setdiff1d(np.arange(T), bad)
    np.testing.assert_array_equal(got[1][good], got[0][good])
