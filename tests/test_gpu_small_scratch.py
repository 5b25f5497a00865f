"""Scratch too small for the matrix-core coarse pass: many centroids of many dimensions take the float64
coarse pass instead, and answer the same."""
import ctypes

import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search
from tests.test_gpu_batched_lists import _call
from trident_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def wide(dev):
    """7,000 lists of one or two rows in 1,024 dims, lists 3 and 7 of the same centroid: the split
    operands take 43 MB, the centroids' rows 29, the fixed scratch is 67 MB (2^26 bytes)."""
    rng = np.random.default_rng(3)
    nlist, D = 7000, 1024
    cen = rng.normal(size=(nlist, D)).astype(np.float32)
    cen[7] = cen[3]
    lid = np.concatenate([np.arange(nlist), np.arange(0, nlist, 3)])
    xb = cen[lid] + (0.1 * rng.normal(size=(len(lid), D))).astype(np.float32)
    b = build_index(torch.as_tensor(xb), nlist, dev, list_ids=lid, centroids=cen, max_batch=2)
    xq = (cen[[3, 50]] + 0.1 * rng.normal(size=(2, D))).astype(np.float32)
    return b, xq


@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("nprobe", [1, 34, 100])
def test_fixed_scratch(dev, wide, nprobe, rows):
    b, xq = wide
    xqd = torch.as_tensor(xq).to(dev)
    keep = b.ix.cent_band
    try:
        if not rows:
            b.ix.cent_band = None
        need = _lib.lib().trident_workspace_bytes(ctypes.byref(b.ix.view()), 2, nprobe, 10)
        assert rows or need > _lib.NOALLOC_SCRATCH_BYTES
        _, rd, ri = oracle_search(b, xq, nprobe, 10)
        for ws in (need, need - 1, 16 << 20, None):
            rc, d, i = _call(b, xqd, nprobe, 10, ws)
            assert rc == 0, (ws, need)
            assert_exact(d, i, rd, ri, f"rows={rows} nprobe={nprobe} workspace={ws}")
        rc, _, _ = _call(b, xqd, nprobe, 10, 64 << 10)
        assert rc == 3, "64 KiB is refused"
    finally:
        b.ix.cent_band = keep
