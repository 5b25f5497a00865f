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


def _descending(D, u8, n_lists=20, rows=8192):
    """A list of 5 rows nearest to every query, then lists of eight slices whose rows come nearer one by
    one: with K > 5 no query has a threshold when the 160 units start, each lists its first 64 rows at
    least (10,240 where a list holds 4,096), and every later block holds rows nearer than all before."""
    rng = np.random.default_rng([D, u8])
    sizes = [5] + [rows] * n_lists
    lid = np.repeat(np.arange(len(sizes)), sizes)
    xb = (0.01 * rng.normal(size=(len(lid), D))).astype(np.float32)
    pos = np.concatenate([np.arange(s) % 1024 for s in sizes])
    xb[:, 0] += np.where(lid == 0, 9.0, 6.0 - 5.0 * pos / 1024)
    if u8:
        xb = np.clip(np.round(40.0 + 20.0 * xb), 0, 255).astype(np.float32)
    cen = np.zeros((len(sizes), D), np.float32)
    cen[1:, 1] = 300.0 + np.arange(n_lists)
    return torch.as_tensor(xb), lid, cen, len(sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("D,base", [(32, "device"), (50, "host"), (128, "host-u8"), (300, "device"), (320, "host-u8")])
def test_overflowed_lists_of_small_k(dev, D, base):
    """The same up to K = 16, where the scan keeps thresholds of its own, past the 32 queries of the
    cascade's slots, and (host base) that the rescan ran: every probed row is read a second time."""
    xb, lid, cen, nlist = _descending(D, base == "host-u8")
    b = build_index(xb, nlist, dev, list_ids=lid, centroids=cen, max_batch=64, xb_placement=base.split("-")[0],
                    within="id")
    rng = np.random.default_rng(D)
    q = (0.01 * rng.normal(size=(40, D))).astype(np.float32)
    xq = q if base != "host-u8" else np.round(40.0 + 20.0 * q).astype(np.float32)
    xqd = torch.as_tensor(xq).to(dev)
    hr = torch.zeros(1, dtype=torch.int64, device=dev)
    try:
        for B, K in ((1, 6), (1, 10), (40, 10), (3, 16), (40, 33), (2, 64)):
            _, rd, ri = oracle_search(b, xq[:B], nlist, K)
            d, i, _ = b.ix.search(xqd[:B], nlist, mode=10, k=K, route=2, host_rows_buf=hr if base != "device" else None)
            torch.cuda.synchronize()
            assert_exact(d.cpu().numpy(), i.cpu().numpy(), rd, ri, f"{base} D={D} B={B} K={K}")
            if base != "device":
                assert int(hr) >= len(lid) * (1 + B), f"no rescan: {int(hr)} host rows, B={B} K={K}"
    finally:
        torch.cuda.synchronize()
        if b.ix.storage._host_buf is not None:
            b.ix.storage._host_buf.free()


@pytest.mark.gpu
def test_a_short_first_list_costs_no_serial_rescan(dev):
    """One query whose nearest list holds fewer than K rows and overflows its list: the time stays near
    the per-pair scan's (one wave reading every probed row took 100 times that)."""
    import time
    xb, lid, cen, nlist = _descending(128, False)
    b = build_index(xb, nlist, dev, list_ids=lid, centroids=cen, max_batch=8, within="id")
    xqd = torch.zeros((1, 128), device=dev)
    ms = []
    for route in (1, 2):
        best = 1e9
        for _ in range(5):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            b.ix.search(xqd, nlist, mode=10, k=10, route=route)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        ms.append(best * 1e3)
    assert ms[1] < 12 * ms[0], ms
