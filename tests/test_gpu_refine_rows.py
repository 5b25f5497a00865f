"""The staged float64 rows (refine_rows) at the edges of its steps: 16-dim runs of the chain, 128-dim
chunks, 16-row groups, rows of whole float4s or not, and the uint8 copy of a host base."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search


def _integer_base(n, D, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, 256, (n, D), generator=g).float()


@pytest.mark.gpu
@pytest.mark.parametrize("placement", ["device", "host"])
@pytest.mark.parametrize("D", [5, 15, 16, 17, 112, 127, 128, 129, 132, 144, 160, 257, 400])
def test_steps_and_remainders(dev, D, placement):
    """Integer rows: their float64 distances are exact in any order, ties and all.  K = 1, 17 and 100
    seeds leave groups of 1, 16 + 1 and 64 + 36 rows; mode 10 per pair takes 64-row batches of clusters."""
    xb = _integer_base(900, D, D)
    lid = np.repeat(np.arange(4), [100, 129, 191, 480])
    cen = torch.stack([xb[torch.as_tensor(lid == c)].mean(0) for c in range(4)]).numpy()
    b = build_index(xb, 4, dev, list_ids=lid, centroids=cen, max_batch=32, xb_placement=placement)
    xq = _integer_base(21, D, D + 1).numpy() + 0.25
    for K in (1, 17, 100):
        _, rd, ri = oracle_search(b, xq, 3, K)
        for mode, route in ((2, 2), (2, 1), (10, 1)):
            d, i = run_search(b, torch.as_tensor(xq).to(dev), 3, K, mode=mode, ub=1, route=route)
            assert_exact(d, i, rd, ri, f"D={D} K={K} mode={mode} route={route}")
