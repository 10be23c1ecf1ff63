"""E-step statistics against the FP64 oracle where a sample tile, an 8-sample
group or a wave's channels are not full, with one sample whose densities
underflow in every component."""
import numpy as np
import pytest

import cudamica_amd as ca
from oracle import pyoracle as po
from tests.test_gpu_engine import _compare_stats, _random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,T,M,m", [(33, 2001, 2, 1), (64, 2002, 3, 2), (70, 2003, 4, 3), (20, 2004, 8, 3),
                                     (65, 2005, 2, 4), (30, 2006, 8, 4), (40, 2007, 2, 5), (130, 2009, 4, 3)])
def test_tile_remainders(built, n, T, M, m):
    print(f"[estep tiles] n={n} T={T} M={M} m={m}", flush=True)
    x = np.random.default_rng(n + T).laplace(size=(T, n))
    x[T - 2] *= 50.0
    x32 = x.astype(np.float32).astype(np.float64)
    st = _random_state(n, M, m, seed=n + m)
    ora = po.estep(x32, 0.3, st["A"], st["c"], st["alpha"], st["mu"], st["beta"], st["rho"], st["gm"], M, m)
    with ca.Engine(ca.options(n, T, M, m, precision=ca.PREC_FP32)) as eng:
        eng.load_white(x32, 0.3)
        eng.set_state(st)
        gpu = eng.estep_stats()
    # posteriors are exponentials of FP32 sums of n log densities (|L| up to
    # about 4 n here): 2^-24 * 4 n * sqrt(4 n / 16) / sqrt(T) < 2e-6 of vsum
    _compare_stats(gpu, ora, n, m, M, vsum_tol=2e-6)


@pytest.mark.parametrize("n,T,m", [(64, 1009, 3), (17, 1041, 1), (40, 5007, 2), (64, 30_001, 3), (8, 2048, 3),
                                   (64, 1024, 4)])
def test_single_model_fp32(built, n, T, m):
    """One model of up to 64 channels: 16-sample tiles whose first or second
    eight samples the recording ends in, one or several ranges per workgroup,
    and b where the E-step formed it itself (m <= 3)."""
    print(f"[estep m1] n={n} T={T} m={m}", flush=True)
    x = np.random.default_rng(n + T).laplace(size=(T, n)).astype(np.float32).astype(np.float64)
    st = _random_state(n, 1, m, seed=n + m)
    ora = po.estep(x, 0.3, st["A"], st["c"], st["alpha"], st["mu"], st["beta"], st["rho"], st["gm"], 1, m)
    with ca.Engine(ca.options(n, T, 1, m, precision=ca.PREC_FP32)) as eng:
        eng.load_white(x, 0.3)
        eng.set_state(st)
        gpu = eng.estep_stats()
        b = eng.debug_buffer("b64", np.float64, (T, 64))
        W = eng.debug_buffer("Wg64", np.float64, (64, 64))
        wc = eng.debug_buffer("wc64", np.float64, (64,))
    _compare_stats(gpu, ora, n, m, 1)
    xp = np.zeros((T, 64))
    xp[:, :n] = x
    # 64 products and the subtraction, in any order
    assert np.all(np.abs(b - (xp @ W.T - wc)) <= 2 * 66 * 2.0 ** -53 * (np.abs(xp) @ np.abs(W).T + np.abs(wc)))
