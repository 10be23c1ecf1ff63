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
