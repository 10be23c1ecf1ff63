"""The E-step that forms b itself (one model of up to 64 channels, FP32 path,
m <= 3), through an output of its own: g of every sample and channel against
FP64 from the same data and state.  A wrong fragment, row or transpose of its
unmixing would move g by its own size.  Sample counts end in the first or
second eight samples of a 16-sample tile; the longest has ranges of several
tiles."""
import numpy as np
import pytest

import cudamica_amd as ca
from tests.test_gpu_engine import _random_state

pytestmark = pytest.mark.gpu

L2E = 1.4426950408889634


@pytest.mark.parametrize("n,T,m", [(64, 1009, 3), (17, 1047, 1), (40, 1016, 2), (64, 1033, 1), (64, 2015, 2),
                                   (8, 33, 3), (33, 140_009, 3)])
def test_g_of_every_sample(built, n, T, m):
    print(f"[estep g] n={n} T={T} m={m}", flush=True)
    from scipy.special import gammaln
    x = np.random.default_rng(n + T).laplace(size=(T, n)).astype(np.float32).astype(np.float64)
    st = _random_state(n, 1, m, seed=n + m)
    with ca.Engine(ca.options(n, T, 1, m, precision=ca.PREC_FP32)) as eng:
        eng.load_white(x, 0.0)
        eng.set_state(st)
        eng.estep_stats()
        g = eng.debug_buffer("g", np.float32, (T, 64)).astype(np.float64)
    W = np.linalg.inv(st["A"].reshape(n, n).T)
    b = (x - st["c"]) @ W.T
    al, mu, be, rho = (st[k].reshape(m, n) for k in ("alpha", "mu", "beta", "rho"))
    y = np.sqrt(be) * (b[:, None, :] - mu)
    la = np.log2(np.maximum(np.abs(y), 2.0 ** -126))
    yr = np.exp2(rho * la)
    q2 = L2E * (np.log(al) + 0.5 * np.log(be) - np.log(2.0) - gammaln(1.0 + 1.0 / rho) - yr)
    e = np.exp2(q2 - q2.max(1, keepdims=True))
    terms = np.sqrt(be) * (e / e.sum(1, keepdims=True)) * rho * np.sign(y) * np.exp2((rho - 1.0) * la)
    # FP32 rounding, in units of 2^-23: |y|^(rho-2) takes the rounding of its
    # exponent p = (rho - 2) log2|y| and its logarithm, |y|^rho a few more, Q
    # that of |y|^rho at its own size, and u the spread of the Q's; every
    # hardware log2 and exp2 adds one
    p = np.abs((rho - 2.0) * la)
    rel = 2.0 * p + 8.0
    dq = (L2E * yr * rel + np.abs(q2) + 2.0).max(1, keepdims=True)
    bound = 2.0 ** -23 * (np.abs(terms) * (rel + 2.0 * dq + 8.0)).sum(1) + 1e-30
    worst = float((np.abs(g[:, :n] - terms.sum(1)) / bound).max())
    print(f"  largest error {worst:.3f} of its bound", flush=True)
    assert worst <= 1.0
    assert not g[:, n:].any()
