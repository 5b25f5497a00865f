"""The front end's launches at the edges of their tiles: 16-query and 16-column rotation tiles
(dimensions and batches around them, rows not 16-byte aligned), the three-part coarse pass split
over the dimensions and not, and the grouping scan around its 4,096-cluster chunk and the LDS
counters' limit."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search
from trident_amd import datagen

pytestmark = pytest.mark.gpu


def _search(b, xq, nprobe, K, **kw):
    d, i, _ = b.ix.search(xq, nprobe, k=K, **kw)
    torch.cuda.synchronize()
    cids = b.ix.probe_cids_buf[:len(xq), :nprobe].cpu().numpy()
    return d.cpu().numpy(), i.cpu().numpy(), cids


@pytest.mark.parametrize("D", [2, 15, 17, 33, 130, 257, 960, 1030])
def test_rotation_and_coarse_tiles(dev, D):
    xb, xq = datagen.cfg1(N=1500, D=D, B=70, n_centers=12, seed=D)
    b = build_index(xb, 20, dev, max_batch=70)
    raw = torch.empty(70 * D + 1, device=dev)
    shifted = raw[1:].view(70, D)  # 4-byte aligned rows
    shifted.copy_(xq.to(dev))
    for B, q in ((1, shifted), (15, xq.to(dev)), (17, shifted), (70, xq.to(dev))):
        rc, rd, ri = oracle_search(b, xq.numpy()[:B], 7, 5)
        for mode, route in ((2, 1), (2, 0), (10, 0)):
            d, i, c = _search(b, q[:B], 7, 5, mode=mode, route=route)
            assert np.array_equal(c, rc), f"D={D} B={B} mode={mode}"
            assert_exact(d, i, rd, ri, f"D={D} B={B} mode={mode} route={route}")


@pytest.mark.parametrize("B", [63, 1023])
def test_wide_coarse_pass_split_and_whole(dev, B):
    """1,100 centroids in 200 dimensions: 63 queries split the dimensions over the waves, 1,023
    do not; the last centroid tile is partial in both."""
    xb, xq = datagen.cfg1(N=4000, D=200, B=B, n_centers=64, seed=9)
    b = build_index(xb, 1100, dev, max_batch=B, niter=2)
    rc, rd, ri = oracle_search(b, xq.numpy(), 20, 10)
    d, i, c = _search(b, xq.to(dev), 20, 10, mode=2, ub_seed=1)
    assert np.array_equal(c, rc)
    assert_exact(d, i, rd, ri)


@pytest.mark.parametrize("nlist", [1, 3, 4096, 4097, 8191, 8192])
def test_grouping_chunks(dev, nlist):
    g = torch.Generator().manual_seed(nlist)
    xb = torch.randn((2 * nlist + 500, 16), generator=g)
    xq = torch.randn((90, 16), generator=g)
    b = build_index(xb, nlist, dev, list_ids=(np.arange(len(xb)) % nlist), centroids=xb[:nlist].numpy(),
                    max_batch=90)
    nprobe = min(nlist, 40)
    _, rd, ri = oracle_search(b, xq.numpy(), nprobe, 10)
    for mode, route, ub in ((2, 2, 1), (2, 2, 2), (2, 1, 1), (10, 2, 0), (10, 1, 0)):
        d, i, _ = _search(b, xq.to(dev), nprobe, 10, mode=mode, route=route, ub_seed=ub)
        assert_exact(d, i, rd, ri, f"nlist={nlist} mode={mode} route={route} ub={ub}")
