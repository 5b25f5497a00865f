"""The batched route's seeding lists at the edges of their lengths: K on both sides of the
per-lane list lengths (16, 64) and at 128, clusters shorter than K, duplicated rows (equal
bounds), and every probe seeding (lists past the 512 entries one wave holds in registers)."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search
from trident_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[96, 300])
def uneven(request, dev):
    """30 clusters: a few of 1 to 40 rows, one of 2,500, and 300 copies of one row."""
    D = request.param
    xb, xq = datagen.cfg1(N=9_000, D=D, B=70, n_centers=24, seed=5)
    xb[1000:1300] = xb[1000]
    g = torch.Generator().manual_seed(3)
    lid = torch.randint(8, 30, (9_000,), generator=g)
    lid[:2500] = 7
    for c, n in enumerate((1, 2, 15, 16, 17, 40)):
        lid[2500 + 50 * c:2500 + 50 * c + n] = c
    cen = torch.stack([xb[lid == c].mean(0) if bool((lid == c).any()) else xb[c] for c in range(30)])
    b = build_index(xb, 30, dev, list_ids=lid.numpy(), centroids=cen.numpy(), max_batch=128)
    return b, np.concatenate([xq.numpy(), xb[1000:1002].numpy()])


@pytest.mark.parametrize("K", [16, 17, 64, 65, 127, 128])
def test_seeding_lists_at_their_edges(uneven, dev, K):
    b, xq = uneven
    xqd = torch.as_tensor(xq).to(dev)
    for nprobe, ub in ((3, 1), (30, 1), (30, 2)):
        _, rd, ri = oracle_search(b, xq, nprobe, K)
        d, i = run_search(b, xqd, nprobe, K, mode=2, ub=ub, route=2)
        assert_exact(d, i, rd, ri, f"K={K} nprobe={nprobe} ub={ub}")
