"""Putting key shares of many rows together: row counts that do not fill the last workgroup, or a thread's second row, fewer queries
than a workgroup has rows, a share without keys; the bar of the one-workgroup path against the oracle."""
import pytest

from test_gpu_attention import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('splits', [2, 3, 8])
@pytest.mark.parametrize('D', [64, 128])
@pytest.mark.parametrize('B,H,Lq,Lk', [
    (3, 7, 197, 200),       # 4137 rows
    (64, 65, 1, 130),       # 4160 rows of one query each
    (5, 103, 8, 60),        # 4120 rows over one tile: the other shares have no keys
    (2, 16, 128, 300),      # 4096 rows, the fewest
])
def test_rows_of_many_shares(dev, B, H, Lq, Lk, D, splits):
    _run(dev, B, H, Lq, Lk, D, 4, D, D, seed=B * Lq + D + splits, what='combine', splits=splits)
