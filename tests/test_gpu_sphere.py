"""Preprocessing on the GPU (mean, covariance, S = 2 C^-1/2, log-determinant,
whitened data) against numpy in FP64, at the sizes where its kernels change
shape: one channel, both sides of the 16- and 32-wide product tiles and of
the 64-channel padding, sample counts that end inside a tile, and covariances
from well conditioned to beyond what the Newton-Schulz products take, where
the eigensolver computes S."""
import numpy as np
import pytest

import cudamica_amd as ca

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _recording(n, T, cond, seed):
    """Correlated channels whose covariance has condition number ~cond, with offsets."""
    rng = np.random.default_rng(seed)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    s = rng.laplace(size=(T, n)) * np.logspace(0.0, -0.5 * np.log10(cond), n)
    return (s @ q.T + 3.0 * rng.standard_normal(n)).astype(np.float32)


@pytest.mark.parametrize("n,T,cond", [(1, 50, 1.0), (2, 64, 10.0), (15, 1000, 1e2), (16, 1025, 1e3),
                                      (17, 2049, 1e4), (63, 3001, 1e4), (64, 4096, 1e6), (65, 4099, 1e2),
                                      (130, 5003, 1e4), (192, 6000, 1e2), (193, 6007, 1e3), (260, 9001, 1e4),
                                      (300, 9000, 1e2), (704, 3000, 1e2), (1024, 4100, 1e1), (32, 4000, 1e11)])
def test_sphering_against_numpy(built, n, T, cond):
    print(f"[sphere] n={n} T={T} cond={cond:g}", flush=True)
    x = _recording(n, T, cond, 17 * n + T)
    xd = x.astype(np.float64)
    mean = xd.mean(0)
    C = (xd - mean).T @ (xd - mean) / T
    d, V = np.linalg.eigh(C)
    S = (V * (2.0 / np.sqrt(d))) @ V.T
    with ca.Engine(ca.options(n, T, 1, 1)) as eng:
        eng.load_raw(x)
        eng.preprocess(1)
        Sg, mg, lg = eng.sphere()
        w = eng.white()
    Sg = Sg.reshape(n, n)
    kappa = d[-1] / d[0]
    # C's own rounding (a few eps of its norm) moves C^-1/2 by about kappa
    # times as much, relative to its norm: n sums of it on either side
    tol = 8.0 * EPS * (np.sqrt(n) * kappa + 100.0)
    np.testing.assert_allclose(mg, mean, rtol=0, atol=64 * EPS * (np.abs(mean).max() + 1.0))
    assert np.linalg.norm(Sg - S) <= tol * np.linalg.norm(S)
    assert abs(lg + np.linalg.slogdet(S)[1]) <= n * tol + 1e-12 * (1.0 + abs(lg))
    # whitened data: FP64 products rounded to float32 once
    ref = (xd - mean) @ Sg.T
    np.testing.assert_allclose(w, ref, rtol=2e-7, atol=1e-12 * np.abs(ref).max() + 1e-30)


@pytest.mark.parametrize("n,M", [(1, 1), (16, 2), (17, 3), (65, 1), (193, 2), (260, 5)])
def test_output_transform_against_numpy(built, n, M):
    print(f"[output] n={n} M={M}", flush=True)
    T = 20 * n + 50
    x = _recording(n, T, 1e2, 31 * n + M)
    st = ca.synth_init(n, M, 2, n + M)
    with ca.Engine(ca.options(n, T, M, 2)) as eng:
        eng.load_raw(x)
        eng.preprocess(1)
        eng.set_state(st)
        S, mean, _ = eng.sphere()
        A, c = eng.output()
    Sinv = np.linalg.inv(S.reshape(n, n).T)
    # two inverses of S, each off by at most ~n eps cond(S)
    tol = 8.0 * n * EPS * np.linalg.cond(S.reshape(n, n)) + 1e-14
    for h in range(M):
        ref = Sinv @ st["A"].reshape(M, n, n)[h].T
        ref /= np.linalg.norm(ref, axis=0)
        got = A.reshape(M, n, n)[h].T
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
        ref = Sinv @ st["c"].reshape(M, n)[h] + mean
        assert np.linalg.norm(c.reshape(M, n)[h] - ref) <= tol * (np.linalg.norm(Sinv) * np.sqrt(n) + np.linalg.norm(ref))
