"""CostRouter's default rule: the cascade where the library runs it batched, where the base is in
host memory and from W0 on, else mode 10."""
import ctypes
import types

import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search
from tests.test_route_rule import _view
from trident_amd import _lib, datagen, router


class _Index:
    """An index by its sizes: the library's route needs no more."""

    def __init__(self, N, D, nlist, placement="device", layouts=True, packed=True):
        self.N, self.D, self.nlist, self.k = N, D, nlist, 10
        self.storage = types.SimpleNamespace(placement=placement)
        self.v = _view(N, D, nlist, layouts)
        if not packed:
            self.v.sq8_packed = None

    def route_for(self, B, nprobe, k=None, route=0, mode=2):
        r = _lib.lib().trident_route_for_mode(ctypes.byref(self.v), mode, B, k or self.k, nprobe, route)
        if r < 0:
            _lib.check(-r, "trident_route_for")
        return r


@pytest.mark.parametrize("N,D,nlist,nprobe,B,want", [
    (1_000_000, 128, 1024, 64, 1, 2), (1_000_000, 128, 1024, 64, 40, 2),       # long clusters: batched
    (200_000, 960, 512, 8, 1, 2), (1_000_000, 128, 1024, 1, 1, 10),
    (100_000, 128, 250, 16, 31, 10), (100_000, 128, 250, 16, 32, 2),           # W = 2.56e7 at 31.25
    (60_000, 100, 300, 300, 8, 2), (60_000, 100, 300, 300, 4, 10),             # 8 pairs a cluster
])
def test_rule(N, D, nlist, nprobe, B, want):
    ix = _Index(N, D, nlist)
    r = router.CostRouter(ix)
    assert r.rule == "route" and r.mode_for(B, nprobe) == want
    assert router.CostRouter(ix, rule="route").mode_for(B, nprobe) == want
    # the other rules stand as they were
    assert router.CostRouter(ix, rule="pairs").mode_for(B, nprobe) == router.choose_mode_pairs(B, nprobe, nlist)
    assert router.CostRouter(ix, W0=1.0).mode_for(B, nprobe) == 2


def test_rule_by_placement_layouts_and_neighbours():
    assert router.CostRouter(_Index(100_000, 128, 250, placement="host")).mode_for(1, 16) == 2
    assert router.CostRouter(_Index(100_000, 128, 250)).mode_for(1, 16) == 10
    bare = router.CostRouter(_Index(1_000_000, 128, 1024, layouts=False))      # per-pair: by the work
    assert bare.mode_for(1, 64) == 10 and bare.mode_for(4, 64) == 2
    # packing released and K past the batched route's lists: this cascade cannot run
    r = router.CostRouter(_Index(1_000_000, 128, 1024, packed=False))
    assert r.mode_for(40, 64, k=10) == 2 and r.mode_for(40, 64, k=129) == 10


@pytest.mark.gpu
@pytest.mark.parametrize("base", ["device", "host"])
def test_both_modes_answer_exactly(dev, base):
    xb, xq = datagen.cfg1(N=20_000, D=64, B=64, n_centers=30, seed=8)
    b = build_index(xb, 64, dev, max_batch=64, xb_placement=base)
    try:
        r = router.CostRouter(b.ix)
        for B, nprobe, K in ((1, 4, 10), (64, 32, 10), (7, 64, 50)):
            _, rd, ri = oracle_search(b, xq.numpy()[:B], nprobe, K)
            d, i, _, mode = r.search(xq[:B].to(dev), nprobe, k=K)
            torch.cuda.synchronize()
            assert mode == r.mode_for(B, nprobe, K) and (base != "host" or mode == 2)
            assert_exact(d.cpu().numpy(), i.cpu().numpy(), rd, ri, f"{base} B={B} nprobe={nprobe} K={K} mode={mode}")
    finally:
        torch.cuda.synchronize()
        if b.ix.storage._host_buf is not None:
            b.ix.storage._host_buf.free()
