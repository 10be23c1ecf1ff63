"""The FP32 statistic GEMM where the number of sample ranges decides its
workgroups (one range each, or several that meet in LDS) and the steps of loads a
wave has in flight, against numpy in FP64 on the engine's own g and x."""
import numpy as np
import pytest

import cudamica_amd as ca
from tests.test_gpu_statgemm import _operands

pytestmark = pytest.mark.gpu


# 512 samples a range on 256 CUs: a range to a workgroup, one per CU at most
# (65k samples of 128 x 256 columns), and with one step in flight where three
# (128-column x blocks) or five (64) waves a SIMD hold all ranges; widths of
# three and five waves with four, two and one step
@pytest.mark.parametrize("n,M,T", [(128, 2, 70_003), (100, 2, 131_070), (256, 1, 140_003), (64, 4, 530_001),
                                   (180, 1, 101), (180, 1, 180_001), (180, 1, 240_002), (64, 3, 66_005),
                                   (300, 1, 20_006), (300, 1, 30_007), (300, 1, 60_001), (64, 5, 200_002)])
def test_ranges_and_steps(built, n, M, T):
    print(f"[statgemm depth] n={n} M={M} T={T}", flush=True)
    g, x, G = _operands(ca.PREC_FP32_PLAIN, n, M, T, T)
    # 512 samples per FP32 accumulation, four products at a time
    bound = (512 / 4 + 8) * 2.0 ** -24 * (np.abs(g).T @ np.abs(x))
    assert np.all(np.abs(G - g.T @ x) <= bound + 1e-300)
