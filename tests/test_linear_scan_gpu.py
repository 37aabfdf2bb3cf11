"""The decode scan of linear attention with 1024 threads: ragged rows, values that leave threads over, the edge of its rule."""
import pytest

from tests.test_fubapel_gpu import KINDS, check_lin, lin_case, run_lin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dt", ["bf16", "fp32"])
@pytest.mark.parametrize("H,D,V,n", [(1, 128, 132, 1), (2, 250, 260, 5), (1, 1000, 20, 2), (3, 65, 256, 7), (8, 129, 128, 64),
                                     (9, 129, 128, 57), (1, 220, 224, 1), (1, 2460, 20, 2), (3, 193, 256, 7), (8, 384, 128, 16),
                                     (8, 384, 128, 17), (2, 256, 188, 3)])
def test_decode(kind, dt, H, D, V, n):
    c = lin_case(kind, [1] * n, H, D, V, dt, [(5 * i) % 23 for i in range(n)], D - D % 2)
    check_lin(c, dt, run_lin(c, dt, None))
