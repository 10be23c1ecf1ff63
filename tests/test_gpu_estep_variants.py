"""E-step statistics against the FP64 oracle for the variants of the kernel that
follow from the components, the path and the number of waves in a workgroup:
two-sample tiles on the FP32 path at m = 3 (five waves and more, and the split
launch), one-sample tiles that keep or form again what the sums need (m = 4 on
the FP32 path, m >= 5; five to seven waves at m = 5 on the plain path), with a
last tile that is not full and one sample whose densities underflow in every
component."""
import numpy as np
import pytest

import cudamica_amd as ca
from oracle import pyoracle as po
from tests.test_gpu_engine import _compare_stats, _random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n,T,M,m", [
    ("fp32", 60, 1501, 5, 3), ("fp32", 100, 1502, 3, 3), ("fp32", 20, 1503, 7, 3), ("fp32", 300, 1505, 2, 3),
    ("fp32", 40, 1506, 2, 4), ("fp32", 64, 1507, 6, 4), ("fp32", 30, 1501, 3, 6), ("fp32", 200, 1502, 3, 6),
    ("fp32", 90, 1503, 2, 7), ("fp32", 60, 1505, 10, 8), ("plain", 60, 1506, 2, 5), ("plain", 100, 1507, 3, 5),
    ("plain", 30, 1501, 7, 5), ("plain", 64, 1502, 8, 6), ("plain", 300, 1503, 2, 5), ("plain", 30, 1505, 3, 8)])
def test_variants(built, prec, n, T, M, m):
    print(f"[estep variants] {prec} n={n} T={T} M={M} m={m}", flush=True)
    x = np.random.default_rng(n + T).laplace(size=(T, n))
    x[T - 2] *= 50.0
    x32 = x.astype(np.float32).astype(np.float64)
    st = _random_state(n, M, m, seed=n + m)
    ora = po.estep(x32, 0.3, st["A"], st["c"], st["alpha"], st["mu"], st["beta"], st["rho"], st["gm"], M, m)
    code = ca.PREC_FP32 if prec == "fp32" else ca.PREC_FP32_PLAIN
    with ca.Engine(ca.options(n, T, M, m, precision=code)) as eng:
        eng.load_white(x32, 0.3)
        eng.set_state(st)
        gpu = eng.estep_stats()
    # the bars of the two paths (test_gpu_engine, test_gpu_plain)
    if prec == "fp32":
        _compare_stats(gpu, ora, n, m, M, vsum_tol=2e-6)
    else:
        _compare_stats(gpu, ora, n, m, M, tol=1e-4, ll_tol=1e-6, skip=("mu_denom",), vsum_tol=1e-5)
