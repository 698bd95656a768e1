"""Row blocks of matrices of more than 262,144 rows, whose segments hold 16,384
rows (4,096 up to there), against the oracle's greedy walk."""
import numpy as np
import pytest

import oracle
from gpu_cases import announce

pytestmark = pytest.mark.gpu

FEW = 1 << 18  # the largest number of rows with segments of 4,096
SEG = 16384


def _mixed(n, seed):
    return np.minimum(1 / (1 - np.random.default_rng(seed).random(n)), 5000).astype(np.int64)


BLOCK_ROWS = {
    "last with small segments": lambda: np.full(FEW, 3),
    "first with large ones": lambda: np.full(FEW + 1, 3),
    "one short of a segment": lambda: np.full(FEW + SEG - 1, 2),
    "whole segments": lambda: np.full(FEW + SEG, 2),
    "one past": lambda: np.full(FEW + SEG + 1, 1),
    # blocks of W + 1 empty rows pass over whole segments for W >= 32,768
    "empty rows over segments": lambda: np.concatenate([np.zeros(90000), [5], np.zeros(120000), [9] * 3,
                                                        np.zeros(80000)]).astype(np.int64),
    "all empty": lambda: np.zeros(300007, np.int64),
    "long rows": lambda: np.tile([700, 1, 0, 699, 513, 512, 511, 1], 34000),
    "a long row at each segment's edge": lambda: np.where(np.arange(300001) % SEG < 2, 3000, 1),
    "mixed": lambda: _mixed(301001, 8),
    "mixed, closed at the last row": lambda: np.append(_mixed(270000, 9), 60000),
}


@pytest.mark.parametrize("W", [1, 64, 512, 2040, 40000])
@pytest.mark.parametrize("rows", list(BLOCK_ROWS))
def test_row_blocks_of_many_rows(gpu, rows, W):
    announce(f"row blocks {rows} W={W}")
    rp = np.concatenate([[0], np.cumsum(BLOCK_ROWS[rows]())]).astype(np.uint32)
    assert np.array_equal(gpu.fill_row_blocks(rp.size - 1, rp, W), oracle.fill_row_blocks(rp, W))
