"""Which route AUTO takes for a few queries, on both sides of its lines (no GPU: the rule reads
sizes only), and on the GPU that the batched route answers small calls as the per-pair route does,
in every form a call can have."""
import ctypes

import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search
from trident_amd import _lib, datagen
from trident_amd._lib import TridentIndexView


def _view(N, D, nlist, layouts=True):
    v = TridentIndexView()
    v.N, v.D, v.D_pad, v.nlist, v.tile_size = N, D, (D + 31) // 32 * 32, nlist, 64
    v.sq8_packed = 256
    if layouts:
        v.vec_Ar = v.sq8_cells = v.orig_ids_sorted = 256
    return v


PAIR, BATCHED = _lib.ROUTE_PAIR, _lib.ROUTE_BATCHED


@pytest.mark.parametrize("N,D,nlist,B,K,nprobe,want", [
    (62_500, 128, 100, 2, 1, 8, BATCHED), (62_400, 128, 100, 2, 1, 8, PAIR),    # 80,000 / 79,872
    (62_500, 128, 100, 1, 1, 8, PAIR), (62_500, 128, 100, 1, 2, 8, BATCHED),    # one neighbour
    (50_000, 400, 100, 4, 10, 8, BATCHED), (49_900, 400, 100, 4, 10, 8, PAIR),  # past 256 dims
    (10_000, 32, 100, 100, 10, 8, BATCHED), (10_000, 32, 100, 99, 10, 8, PAIR),  # 8 pairs a cluster
    (62_500, 128, 100, 2, 129, 8, PAIR),                                        # K past the lists
])
def test_auto_route_lines(N, D, nlist, B, K, nprobe, want):
    L = _lib.lib()
    assert L.trident_route_for(ctypes.byref(_view(N, D, nlist)), B, K, nprobe, 0) == want
    # an index without the batched layouts keeps the per-pair route
    assert L.trident_route_for(ctypes.byref(_view(N, D, nlist, layouts=False)), B, K, nprobe, 0) == PAIR


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "l1", "global", "blocks", "host", "wide", "tile256"])
def test_small_calls_agree_with_the_pair_route(dev, form):
    D = 300 if form == "wide" else 100
    xb, xq = datagen.cfg1(N=14_000, D=D, B=6, n_centers=8, seed=31)
    b = build_index(xb, 10, dev, max_batch=8, per_cluster_sq8=0 if form == "global" else 1,
                    var_block=1 if form == "blocks" else 0, tile_size=256 if form in ("wide", "tile256") else 64,
                    xb_placement="host" if form == "host" else "device")
    xqd = xq.to(dev)
    try:
        for B, K, nprobe, ub, p_init in ((1, 10, 4, 1, -1), (1, 100, 1, 0, -1), (2, 1, 1, 1, -1), (6, 33, 9, 0, 0),
                                         (6, 128, 10, 2, -1), (5, 17, 10, 1, 7)):
            _, rd, ri = oracle_search(b, xq.numpy()[:B], nprobe, K)
            for mode in (2, 10):
                if mode == 2:
                    assert b.ix.route_for(B, nprobe, K) == BATCHED
                for route in (0, 1, 2):
                    d, i, _ = b.ix.search(xqd[:B], nprobe, mode=mode, k=K, ub_seed=ub if mode == 2 else 0, route=route,
                                          p_init=p_init, use_l1=1 if form == "l1" and mode == 2 else 0)
                    torch.cuda.synchronize()
                    assert_exact(d.cpu().numpy(), i.cpu().numpy(), rd, ri,
                                 f"{form} mode={mode} route={route} B={B} K={K} nprobe={nprobe}")
    finally:
        torch.cuda.synchronize()
        if b.ix.storage._host_buf is not None:
            b.ix.storage._host_buf.free()
