"""E-step statistics of the two-sample tiles (m = 4, FP32 b) with one sample
whose densities underflow in every component, which only part of the tiles'
code runs for: the mixed-precision paths and the plain FP32 one, one launch and
the split one, at the bars those paths have without such a sample.  phi is left
to the plain path: its bf16 operands round that one sample's product, which
dominates it, to 2^-9 each."""
import numpy as np
import pytest

import cudamica_amd as ca
from oracle import pyoracle as po
from tests.test_gpu_engine import _compare_stats, _random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["plain", "bf16", "fp8"])
@pytest.mark.parametrize("n,T,M", [(65, 2005, 2), (30, 2006, 8), (96, 2009, 3), (300, 2003, 2)])
def test_a_sample_far_from_every_component(built, prec, n, T, M):
    print(f"[estep far] {prec} n={n} T={T} M={M}", flush=True)
    m = 4
    x = np.random.default_rng(n + T).laplace(size=(T, n))
    x[T - 2] *= 50.0
    x32 = x.astype(np.float32).astype(np.float64)
    st = _random_state(n, M, m, seed=n + m)
    code = {"plain": ca.PREC_FP32_PLAIN, "bf16": ca.PREC_BF16, "fp8": ca.PREC_FP8}[prec]
    with ca.Engine(ca.options(n, T, M, m, precision=code)) as eng:
        eng.load_white(x32, 0.3)
        xh = eng.white().astype(np.float64)
        eng.set_state(st)
        gpu = eng.estep_stats()
    ora = po.estep(xh, 0.3, st["A"], st["c"], st["alpha"], st["mu"], st["beta"], st["rho"], st["gm"], M, m)
    if prec == "plain":
        _compare_stats(gpu, ora, n, m, M, tol=1e-4, ll_tol=1e-6, skip=("mu_denom",), vsum_tol=1e-5)
    else:
        _compare_stats(gpu, ora, n, m, M, tol=1e-3, ll_tol=1e-5, skip=("mu_denom", "phi"), vsum_tol=1e-4)
