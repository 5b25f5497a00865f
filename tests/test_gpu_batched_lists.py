"""The batched route's seeding lists at the edges of their lengths: K on both sides of the
per-lane list lengths (16, 64) and at 128, clusters shorter than K, duplicated rows (equal
bounds), and every probe seeding (lists past the 512 entries one wave holds in registers).  And its candidate
lists: deep enough for a few probes of long clusters, and the smaller ones that a workspace sized
without that depth still gets."""
import ctypes

import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search, run_search
from trident_amd import _lib, datagen
from trident_amd._lib import TridentSearchOutputs, TridentSearchParams

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


def _call(b, xqd, nprobe, K, ws_bytes):
    """trident_search (or, with ws_bytes None, trident_search_noalloc) on the batched route."""
    L, v = _lib.lib(), b.ix.view()
    td = torch.empty((len(xqd), K), dtype=torch.float32, device=xqd.device)
    ti = torch.empty((len(xqd), K), dtype=torch.int64, device=xqd.device)
    sp = TridentSearchParams(2, len(xqd), K, nprobe, 1, 0, -1, 2)
    out = TridentSearchOutputs()
    out.topk_d, out.topk_i = td.data_ptr(), ti.data_ptr()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if ws_bytes is None:
        rc = L.trident_search_noalloc(ctypes.byref(v), ctypes.byref(sp), ctypes.c_void_p(xqd.data_ptr()),
                                      ctypes.byref(out), st)
    else:
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=xqd.device)
        rc = L.trident_search(ctypes.byref(v), ctypes.byref(sp), ctypes.c_void_p(xqd.data_ptr()),
                              ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(ws_bytes), ctypes.byref(out), st)
    torch.cuda.synchronize()
    return rc, td.cpu().numpy(), ti.cpu().numpy()


@pytest.mark.parametrize("nprobe,K", [(1, 10), (2, 100), (4, 128)])
def test_few_probes_of_long_clusters(dev, nprobe, K):
    """1,250 rows a cluster: lists of 64 or K slots a probe overflow, lists of twice the visited
    rows do not.  A workspace one byte short of the stated size, and the fixed scratch of
    trident_search_noalloc, get the smaller lists: same results, through the rescan."""
    xb, xq = datagen.cfg1(N=20_000, D=128, B=2500, n_centers=16, seed=11)
    b = build_index(xb, 16, dev, max_batch=2500)
    xqd = xq.to(dev).contiguous()
    _, rd, ri = oracle_search(b, xq.numpy(), nprobe, K)
    need = _lib.lib().trident_workspace_bytes(ctypes.byref(b.ix.view()), 2500, nprobe, K)
    for ws in (need, need - 1):
        rc, d, i = _call(b, xqd, nprobe, K, ws)
        assert rc == 0
        assert_exact(d, i, rd, ri, f"nprobe={nprobe} K={K} workspace={ws - need}")
    if nprobe == 1:
        assert need > _lib.NOALLOC_SCRATCH_BYTES
        rc, d, i = _call(b, xqd, nprobe, K, None)
        assert rc == 0
        assert_exact(d, i, rd, ri, "fixed scratch")
