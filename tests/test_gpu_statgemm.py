"""The statistic GEMM G = sum_t g_t x_t^T against numpy in FP64 on the engine's
own g and x, where g's columns do not fill the last workgroup's waves."""
import numpy as np
import pytest

import cudamica_amd as ca

pytestmark = pytest.mark.gpu


def _bf16(u):
    return (u.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _operands(prec, n, M, T, seed):
    """g, x (FP64 values of what the engine holds) and its G."""
    NP = (n + 63) // 64 * 64
    x = np.random.default_rng(seed).laplace(size=(T, n))
    with ca.Engine(ca.options(n, T, M, 2, precision=prec)) as eng:
        eng.load_white(x, 0.0)
        eng.set_state(ca.synth_init(n, M, 2, 5))
        eng.estep_stats()
        if prec == ca.PREC_BF16:
            T32 = (T + 31) // 32 * 32
            g8 = eng.debug_buffer("g", np.uint16, (T32 // 8, M * NP, 8))
            g = _bf16(np.ascontiguousarray(g8.transpose(0, 2, 1).reshape(T32, M * NP)[:T]))
            xs = _bf16(eng.debug_buffer("xbf", np.uint16, (2, T, NP))[0])
        else:
            g = eng.debug_buffer("g", np.float32, (T, M * NP)).astype(np.float64)
            xs = eng.debug_buffer("x", np.float32, (T, NP)).astype(np.float64)
        G = eng.debug_buffer("gx", np.float64, (M * NP, NP))
    return g, xs, G


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("n,M,T", [(64, 9, 700), (100, 5, 333), (128, 6, 1000)])
def test_last_column_group_of_the_statistic_gemm(built, prec, n, M, T):
    print(f"[statgemm] {prec} n={n} M={M} T={T}", flush=True)
    g, x, G = _operands(ca.PREC_FP32 if prec == "fp32" else ca.PREC_BF16, n, M, T, T)
    # at most 512 samples (or all of these) per FP32 accumulation, four or more
    # products at a time
    bound = (1024 / 4 + 8) * 2.0 ** -24 * (np.abs(g).T @ np.abs(x))
    assert np.all(np.abs(G - g.T @ x) <= bound + 1e-300)


@pytest.mark.parametrize("n,M,T", [(16, 1, 33), (16, 1, 20_000), (64, 2, 1000), (64, 2, 4099), (64, 3, 2050),
                                   (64, 4, 5001), (100, 1, 3001), (100, 2, 3002), (128, 4, 4003), (200, 1, 2047),
                                   (200, 2, 1029)])
def test_fp32_statistic_gemm_sample_splits(built, n, M, T):
    """Sample counts that end inside a 4-sample step, a wave's range and a
    workgroup's range, for every width of g (waves that split a chunk's samples
    or not) and both column tilings of x."""
    print(f"[statgemm] n={n} M={M} T={T}", flush=True)
    g, x, G = _operands(ca.PREC_FP32, n, M, T, T)
    bound = (512 / 4 + 8) * 2.0 ** -24 * (np.abs(g).T @ np.abs(x))
    assert np.all(np.abs(G - g.T @ x) <= bound + 1e-300)
