"""The blocked inverse where the rows a lane holds of a panel change, and where
the last panel is partial."""
import pytest

from tests.test_gpu_inverse import test_inverse_and_logdet as _inverse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,M,kind", [(255, 1, "permuted"), (257, 2, "random"), (320, 1, "graded"),
                                      (321, 1, "permuted"), (384, 2, "random"), (385, 1, "graded"),
                                      (448, 1, "permuted"), (449, 1, "random")])
def test_panel_rows(built, n, M, kind):
    _inverse(built, n, M, kind)
