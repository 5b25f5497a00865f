"""Mode 10's lists that overflow past K = 16: queries whose nearest list holds fewer than K rows get no
threshold from it and list every row they probe."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search


@pytest.mark.gpu
@pytest.mark.parametrize("D", [30, 300])
@pytest.mark.parametrize("K", [17, 64, 65, 128])
@pytest.mark.parametrize("B", [1, 45])
def test_overflowed_lists(dev, D, K, B):
    """40 queries at a list of 5 rows, then lists of 12,600, 63 and 1: they list 12,669 rows where a list
    holds at most 4,096.  B = 45: more overflow than the 32 that are rescanned in parallel, and five
    queries that don't."""
    rng = np.random.default_rng([D, K])
    sizes = [5, 12600, 63, 1] + [4] * 28
    lid = np.repeat(np.arange(len(sizes)), sizes)
    cen = np.zeros((len(sizes), D), np.float32)
    cen[1, 0], cen[2, 1], cen[3, 2] = 3.0, 4.0, 5.0
    cen[4:, 3] = 100.0 + np.arange(28)
    xb = torch.as_tensor((cen[lid] + 0.1 * rng.normal(size=(len(lid), D))).astype(np.float32))
    b = build_index(xb, len(sizes), dev, list_ids=lid, centroids=cen, max_batch=64)
    xq = (0.1 * rng.normal(size=(B, D))).astype(np.float32)
    xq[40:] += cen[1]
    _, rd, ri = oracle_search(b, xq, 4, K)
    d, i = run_search(b, torch.as_tensor(xq).to(dev), 4, K, mode=10, route=2)
    assert_exact(d, i, rd, ri, f"D={D} K={K} B={B}")
