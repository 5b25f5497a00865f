"""Weight planes and pair records of the batched route: every width's split of the dimensions over
lanes, steps and waves, groups of 1 to 32 pairs and the group after, tiny, huge and constant weights."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search

pytestmark = pytest.mark.gpu


def _search(dev, xb, xq, nprobe, K, **kw):
    lid = np.arange(len(xb)) % 3
    xb = torch.as_tensor(xb)
    cen = np.stack([xb[torch.as_tensor(lid == c)].mean(0).numpy() for c in range(3)])
    b = build_index(xb, 3, dev, list_ids=lid, centroids=cen, max_batch=len(xq), use_pca=0, **kw)
    _, rd, ri = oracle_search(b, xq, nprobe, K)
    d, i = run_search(b, torch.as_tensor(xq).to(dev), nprobe, K, mode=2, route=2)
    assert_exact(d, i, rd, ri)


@pytest.mark.parametrize("D", [5, 64, 65, 128, 190, 256, 257, 321, 700, 960, 1024])
@pytest.mark.parametrize("B", [1, 4, 5, 16, 17, 32, 33, 95])
def test_group_sizes_and_widths(dev, D, B):
    rng = np.random.default_rng([D, B])
    xb = (rng.normal(size=(330, D)) * rng.uniform(0.1, 4.0, size=D)).astype(np.float32)
    xq = (rng.normal(size=(B, D)) * 1.5).astype(np.float32)
    _search(dev, xb, xq, 2, 7)


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1e12])
@pytest.mark.parametrize("D", [128, 320])
def test_weight_scales(dev, D, scale):
    rng = np.random.default_rng(D)
    xb = (rng.normal(size=(300, D)) * scale).astype(np.float32)
    xb[:, 3] = 0.0  # a constant dimension: weight 0 in every pair
    xq = (rng.normal(size=(20, D)) * scale).astype(np.float32)
    xq[5] *= np.float32(1000.0)  # one query sets its group's scale
    _search(dev, xb, xq, 3, 9)
