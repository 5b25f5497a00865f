"""Mode 10's matrix-core products: the six bfloat16 products of three-part operands (h h in one
float32 accumulator, the other five in another) against the bound its scan uses,
    kappa = (Dp + 4) 2^-23 (1 + 2^-7) + (5 Dp + 4) 2^-30 (1 + 2^-5) + 4.2 2^-24,
and against float32 products; and on the GPU every width and unit size at its edges, values whose
squares overflow or vanish, and listed rows past a wave's queue."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search
from tests.test_band_split import _rows
from tests.test_front_end_split3 import _chain, _parts


@pytest.mark.parametrize("kind", ["gauss", "uniform", "coherent", "below_next"])
@pytest.mark.parametrize("D", [32, 256])
def test_six_products_within_bound_and_no_worse_than_float32(kind, D):
    kappa = (D + 4) * 2.0 ** -23 * (1 + 2.0 ** -7) + (5 * D + 4) * 2.0 ** -30 * (1 + 2.0 ** -5) + 4.2 * 2.0 ** -24
    err, ref = [], []
    for seed in range(12):
        rng = np.random.default_rng([seed, D])
        q, x = _rows(rng, kind, D)
        (qh, qm, ql), (xh, xm, xl) = _parts(q), _parts(x)
        prod = q.astype(np.float64) * x
        s = np.float32(_chain([(qh, xh)], rng) + _chain([(qh, xm), (qm, xh), (qh, xl), (qm, xm), (ql, xh)], rng))
        err.append(abs(float(s) - prod.sum()) / np.abs(prod).sum())
        ref.append(abs(float(_chain([(q, x)], rng)) - prod.sum()) / np.abs(prod).sum())
    assert max(err) <= kappa
    # the maxima of two samples of twelve float32 accumulations differ by less than a factor of two
    assert max(err) <= 2.0 * max(ref) + 2.0 ** -24, (max(err), max(ref))


def _lists(rng, sizes):
    return np.repeat(np.arange(len(sizes)), sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [8, 40, 61, 128, 130, 192, 224, 256])
@pytest.mark.parametrize("B", [1, 16, 17, 129])
def test_widths_and_unit_sizes(dev, D, B):
    """All queries probe the same clusters (units of 1, 16, 17 and 129 queries: one wave of eight, two,
    and a second unit), of 63, 64, 65 and 1,100 rows."""
    rng = np.random.default_rng(D)
    lid = _lists(rng, [63, 64, 65, 1100, 1])
    xb = torch.as_tensor(rng.normal(size=(len(lid), D)).astype(np.float32) + lid[:, None])
    cen = torch.stack([xb[torch.as_tensor(lid == c)].mean(0) for c in range(5)])
    b = build_index(xb, 5, dev, list_ids=lid, centroids=cen.numpy(), max_batch=129)
    xq = (rng.normal(size=(B, D)) + 1.5).astype(np.float32)
    for nprobe, K in ((1, 1), (5, 10), (5, 16), (5, 17), (4, 128)):
        _, rd, ri = oracle_search(b, xq, nprobe, K)
        d, i = run_search(b, torch.as_tensor(xq).to(dev), nprobe, K, mode=10, route=2)
        assert_exact(d, i, rd, ri, f"D={D} B={B} nprobe={nprobe} K={K}")


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-30, 1e-18, 3e18])
def test_extreme_scales(dev, scale):
    """Squares far below float32's range, and past it: bounds degenerate, results stay exact."""
    rng = np.random.default_rng(7)
    xb = torch.as_tensor((rng.normal(size=(600, 64)) * scale).astype(np.float32))
    lid = np.arange(600) % 3
    b = build_index(xb, 3, dev, list_ids=lid, centroids=xb[:3].numpy(), max_batch=32, use_pca=0)
    xq = (rng.normal(size=(20, 64)) * scale).astype(np.float32)
    _, rd, ri = oracle_search(b, xq, 3, 10)
    d, i = run_search(b, torch.as_tensor(xq).to(dev), 3, 10, mode=10, route=2)
    assert np.array_equal(i, ri)
    assert np.array_equal(d, rd.astype(np.float32))


@pytest.mark.gpu
def test_more_listed_rows_than_a_wave_queues(dev):
    """Every row is the same point: all are within the band of each other, so each block lists all of
    its rows for every query and the queues drain many times."""
    xb = torch.ones((3000, 32)) * 3.0
    lid = np.arange(3000) % 2
    b = build_index(xb, 2, dev, list_ids=lid, centroids=np.stack([np.full(32, 3.0), np.full(32, 2.0)]), max_batch=64)
    xq = np.full((40, 32), 2.5, np.float32)
    _, rd, ri = oracle_search(b, xq, 2, 12)
    d, i = run_search(b, torch.as_tensor(xq).to(dev), 2, 12, mode=10, route=2)
    assert_exact(d, i, rd, ri)
