"""GPU checks of the kernels that only a tuning key chooses, against the default
ones on the same frame (the bound of test_gpu_pass_shapes: 5e-6)."""
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_pass_shapes import _frame

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,W", [(2048, 2), (4096, 1), (4096, 2), (8192, 1)])
def test_column_elements(ctx, N, W):
    print(f"col_e N={N} W={W}", flush=True)
    want = _frame(ctx, N, W, 1, True, gap_passes=2)
    for keys in (dict(col_e=16), dict(col_e=32), dict(col_c=2)):
        assert rel_l2(_frame(ctx, N, W, 1, True, gap_passes=2, **keys), want) < 5e-6
