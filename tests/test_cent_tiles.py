"""The centroids' tile layout (TridentIndexView.cent_tiles) is read by no kernel: an index does not keep
it, a search does not ask for it, and one that a caller still gives is ignored."""
import ctypes

import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search
from tests.test_route_rule import _view
from trident_amd import _lib, datagen, ext


def test_not_built():
    W = torch.randn(20, 5 + 32)
    rows, tiles, norms, nmax = ext.centroid_band_layouts(W, 5, tiles=False)
    full = ext.centroid_band_layouts(W, 5)
    assert tiles is None and torch.equal(rows, full[0]) and torch.equal(norms, full[2]) and nmax == full[3]


@pytest.mark.parametrize("norms,nmax,ok", [(256, 1.0, True), (None, 1.0, False), (256, -1.0, False),
                                           (256, float("inf"), False)])
def test_not_asked_for(norms, nmax, ok):
    v = _view(1000, 32, 10)
    v.num_blocks, v.rot_sq_min, v.rot_sq_max = 1, 1.0, 1.0
    v.W_combined = v.b_combined = v.cluster_vec_off = v.cluster_tile_off = v.xb_sorted = v.tile_orig_ids = 256
    v.cent_rows, v.cent_norms, v.cent_norm_max = 256, norms, nmax
    # B = 0 ends after the view's checks
    rc = _lib.lib().trident_coarse_probe(ctypes.byref(v), None, 0, 4, None, 0, 256, None, 4, None)
    assert (rc == 0) == ok


@pytest.mark.gpu
def test_ignored(dev):
    xb, xq = datagen.cfg1(N=8000, D=48, B=8, n_centers=16, seed=5)
    b = build_index(xb, 20, dev, max_batch=8)
    _, rd, ri = oracle_search(b, xq.numpy(), 8, 10)
    rows, tiles, norms, nmax = b.ix.cent_band
    assert tiles is None
    for t in (None, torch.full((32 * 48,), float("nan"), device=dev)):
        b.ix.cent_band = (rows, t, norms, nmax)
        d, i, _ = b.ix.search(xq.to(dev), 8, k=10)
        torch.cuda.synchronize()
        assert_exact(d.cpu().numpy(), i.cpu().numpy(), rd, ri)
    b.ix.cent_band = (rows, torch.zeros(7, device=dev), norms, nmax)
    with pytest.raises(_lib.TridentError):  # a wrong size is refused as before
        b.ix.search(xq.to(dev), 8, k=10)
