"""AUTO's lines for a few queries on long clusters, modes 2 and 10, on both sides of each (no GPU: the
rules read sizes only)."""
import ctypes

import pytest

from tests.test_route_rule import BATCHED, PAIR, _view
from trident_amd import _lib


def _route(mode, rows, D, B, K, nprobe, nlist=1000):
    v = _view(rows * nlist, D, nlist)
    r = _lib.lib().trident_route_for_mode(ctypes.byref(v), mode, B, K, nprobe, 0)
    assert r in (PAIR, BATCHED)
    return r


# rows of an average cluster, dims, queries, neighbours, probes; rows x dims is the line's c
@pytest.mark.parametrize("rows,D,B,K,nprobe,want", [
    (625, 128, 2, 10, 2, BATCHED), (624, 128, 2, 10, 2, PAIR),          # 80,000
    (625, 128, 1, 10, 2, BATCHED), (624, 128, 1, 17, 64, PAIR),
    (1000, 100, 1, 1, 2, BATCHED), (999, 100, 1, 1, 64, PAIR),          # one neighbour: 100,000
    (1250, 96, 2, 10, 1, BATCHED), (1249, 96, 2, 10, 1, PAIR),          # one probe: 120,000 ...
    (1000, 100, 4, 10, 1, BATCHED), (1000, 100, 3, 10, 1, PAIR),        # ... or B c = 400,000
    (1249, 96, 1, 10, 1, PAIR), (4000, 100, 1, 10, 1, BATCHED), (4000, 100, 1, 1, 1, PAIR),
    (625, 128, 1, 17, 1, BATCHED), (625, 128, 1, 16, 1, PAIR),          # past K = 16
    (625, 320, 2, 1, 2, BATCHED), (624, 320, 2, 10, 2, PAIR),           # past 256 dims: 200,000
    (1000, 350, 1, 10, 2, BATCHED), (999, 350, 1, 10, 2, PAIR),         # one query: 350,000
    (999, 350, 1, 17, 1, BATCHED), (4000, 350, 1, 1, 64, PAIR),
    (1000, 350, 2, 10, 1, BATCHED), (999, 350, 2, 10, 1, PAIR),         # one probe
    (1000, 300, 4, 10, 1, BATCHED), (999, 300, 4, 10, 1, PAIR),         # ... or 1,200,000
])
def test_cascade_lines(rows, D, B, K, nprobe, want):
    assert _route(2, rows, D, B, K, nprobe) == want


@pytest.mark.parametrize("rows,D,B,K,nprobe,want", [
    (600, 100, 1, 16, 1, BATCHED), (544, 110, 1, 16, 1, PAIR),          # 60,000 (59,840: under 550 rows)
    (600, 100, 1, 17, 1, PAIR), (600, 100, 1, 1, 1, BATCHED),           # past K = 16 only from 4 a cluster
    (600, 80, 1, 10, 1, BATCHED), (599, 80, 1, 10, 1, PAIR),            # 48,000 ...
    (550, 96, 1, 10, 1, BATCHED), (549, 96, 1, 10, 1, PAIR),            # ... from 550 rows
    (400, 125, 50, 10, 10, BATCHED), (400, 125, 49, 10, 10, PAIR),      # ... or P c = 2.5e7
    (300, 125, 399, 10, 10, PAIR), (300, 125, 400, 10, 10, BATCHED),    # 4 queries a cluster
    (1000, 320, 1, 10, 2, BATCHED), (999, 320, 1, 10, 2, PAIR),         # past 256 dims: 320,000
    (500, 400, 40, 10, 10, BATCHED), (500, 400, 39, 10, 10, PAIR),      # 200,000 while P c >= 8e7
    (499, 400, 60, 10, 10, PAIR), (240, 400, 157, 10, 10, BATCHED), (240, 400, 156, 10, 10, PAIR),  # 96,000: 1.5e8
    (500, 400, 6, 10, 1, BATCHED), (500, 400, 5, 10, 1, PAIR), (499, 400, 60, 10, 1, PAIR),        # one probe
    (4000, 960, 1, 17, 64, PAIR),
])
def test_exact_scan_lines(rows, D, B, K, nprobe, want):
    assert _route(10, rows, D, B, K, nprobe) == want


@pytest.mark.parametrize("mode", [2, 10])
def test_what_the_batched_route_cannot_take_stays_per_pair(mode):
    assert _route(mode, 4000, 128, 8, 129, 8) == PAIR
    assert _route(mode, 4000, 1200, 8, 10, 8) == PAIR
