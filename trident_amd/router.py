"""Cost router between the cluster-major exact scan (mode 10) and the cascade (mode 2).

Reference: benchmarks/phase4a_suite.py:1063-1079 (per-batch choice) and :999-1035
(calibration).  The work measure is W = B * nprobe * (N / nlist) * D; the route is mode 10
when W < W0, else mode 2.  The calibration sweeps batch sizes, times both routes with the
reference's methodology (warmup, back-to-back calls, one synchronise) and sets W0 to the
smallest work at which the cascade is at least as fast (the reference's rule);
``stable_crossover`` gives the smallest work from which the cascade wins at every larger
measured work, which ignores an isolated win at a tiny batch.

W0 is hardware-specific.  The reference's A100 value is 946,811,200 (README rounds it to
9.0e8); W0_MI355X = 2.56e7.

No W0 alone fits, because the cascade has two routes here.  Where the library takes its batched
int8 matrix-core route (clusters shared by 8 queries on average, or long ones: trident_route_for)
it wins at any work: 1e6 rows, D = 128, nlist 1024, 64 probes, K = 10, 1 / 16 / 40 / 200 queries take
114 / 138 / 148 / 176 us against mode 10's 152 / 260 / 269 / 365; at D = 960, nlist 512, 260 - 373 against
717 - 1589.  So it does for a base in host memory, of which mode 10 reads every probed row (147 -
285 us against 335 - 4316).  On its per-pair route, short clusters, the crossing follows the work
as in the reference: 311 searches on twelve indexes (33 to 960 dims, 1 to 256 queries, K 1 to 50)
cross between 1.5e7 (up to 256 dims) and 4e7 (past them).  ``choose_mode_route`` is that rule, and
``CostRouter`` uses it unless it is given a W0: on those searches 1.03 times the faster mode in the
geometric mean, at worst 2.3 (one query at D = 768).  ``choose_mode_pairs``, the rule by pairs per
probed cluster alone, stands at 1.27 there, at worst 15.
"""
import time
from typing import Dict, List, Optional, Sequence, Tuple

import torch

from . import _lib

W0_REFERENCE_A100 = 946_811_200.0
# Work from which the cascade's per-pair route is at least as fast as mode 10 on MI355X.
W0_MI355X = 2.56e7
# Pairs per cluster from which the cascade takes its batched route whatever the clusters' length
# (capi.hip, choose_route).
BATCHED_PAIRS_PER_CLUSTER = 8.0

MODE_CM_EXACT = 10
MODE_CASCADE = 2


def work_measure(B: int, nprobe: int, N: int, nlist: int, D: int) -> float:
    """W = B * nprobe * (N / nlist) * D (reference :1018, :1063)."""
    return float(B) * float(nprobe) * (float(N) / float(nlist)) * float(D)


def choose_mode(work: float, W0: float) -> int:
    """mode 10 (exact cluster-major scan) below W0, else mode 2 (cascade) (reference :1079)."""
    return MODE_CM_EXACT if work < W0 else MODE_CASCADE


def choose_mode_pairs(B: int, nprobe: int, nlist: int) -> int:
    """MI355X rule: mode 2 (cascade) once B * nprobe >= 8 nlist (its batched route), else
    mode 10."""
    return MODE_CASCADE if float(B) * nprobe >= BATCHED_PAIRS_PER_CLUSTER * nlist else MODE_CM_EXACT


def choose_mode_route(index, B: int, nprobe: int, k: Optional[int] = None, route: int = 0) -> int:
    """MI355X rule: mode 2 (cascade) where it takes its batched route, where the base lives in host
    memory, and from W0_MI355X on; else mode 10.  Where the index cannot run this cascade, as
    choose_mode_pairs (mode 10 below 8 pairs per cluster)."""
    try:
        batched = index.route_for(B, nprobe, k, route=route, mode=MODE_CASCADE) == _lib.ROUTE_BATCHED
    except _lib.TridentError:
        return choose_mode_pairs(B, nprobe, index.nlist)
    if batched or getattr(index.storage, "placement", "device") == "host":
        return MODE_CASCADE
    return choose_mode(work_measure(B, nprobe, index.N, index.nlist, index.D), W0_MI355X)


def _time_ms(fn, warmup: int, iters: int) -> float:
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(iters):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) * 1000.0 / iters


def calibrate_w0(index, xq_pool: torch.Tensor, nprobe: int,
                 batches: Sequence[int] = (1, 4, 8, 16, 32, 64, 128, 256, 512, 1024),
                 warmup: int = 5, iters: int = 20, ub_seed: int = 0) -> Tuple[float, List[Dict]]:
    """Times mode 10 and mode 2 per batch size; W0 = min work where mode 2 is at least as fast
    (reference :999-1035).  Returns (W0, rows); W0 is +inf if mode 10 always wins."""
    rows, crossings = [], []
    N, nlist, D = index.N, index.nlist, index.D
    for b in batches:
        if b > xq_pool.shape[0] or b > index.max_batch:
            break
        q = xq_pool[:b].contiguous()
        w = work_measure(b, nprobe, N, nlist, D)
        # mode 10 on each of its routes (1: float64 per pair, 2: matrix cores), the
        # faster of them standing for mode 10
        ms_routes = {}
        for rt in (1, 2):
            try:
                ms_routes[rt] = _time_ms(lambda: index.search(q, nprobe, mode=MODE_CM_EXACT, route=rt),
                                         warmup, iters)
            except RuntimeError:  # the matrix-core route does not apply (K, D or placement)
                pass
        ms_cm = min(ms_routes.values())
        ms_k2 = _time_ms(lambda: index.search(q, nprobe, mode=MODE_CASCADE, ub_seed=ub_seed), warmup, iters)
        rows.append({"batch": b, "nprobe": nprobe, "work": w, "ms_cm": ms_cm, "ms_cascade": ms_k2,
                     "ms_cm_pair": ms_routes.get(1), "ms_cm_matrix": ms_routes.get(2),
                     "qps_cm": b * 1000.0 / ms_cm, "qps_cascade": b * 1000.0 / ms_k2,
                     "cascade_faster": ms_k2 <= ms_cm})
        if ms_k2 <= ms_cm:
            crossings.append(w)
    return (min(crossings) if crossings else float("inf")), rows


def stable_crossover(rows: List[Dict]) -> float:
    """Smallest work from which the cascade is at least as fast at every larger measured work
    (+inf when mode 10 wins the largest)."""
    w0 = float("inf")
    for r in sorted(rows, key=lambda r: r["work"], reverse=True):
        if not r["cascade_faster"]:
            break
        w0 = r["work"]
    return w0


class CostRouter:
    """Routes each batch of an index to mode 10 or mode 2: ``rule="work"`` by the reference's
    work measure against W0 (W0_MI355X unless given), ``rule="pairs"`` by choose_mode_pairs,
    ``rule="route"`` by choose_mode_route; ``rule="auto"`` (the default) is "work" when a W0 is
    given, else "route" ("pairs" for an index without ``route_for``)."""

    def __init__(self, index, W0: Optional[float] = None, rule: str = "auto"):
        if rule not in ("auto", "work", "pairs", "route"):
            raise ValueError(f"rule must be 'auto', 'work', 'pairs' or 'route', not {rule!r}")
        if rule == "auto":
            rule = "work" if W0 is not None else "route" if hasattr(index, "route_for") else "pairs"
        self.index = index
        self.rule = rule
        self.W0 = W0_MI355X if W0 is None else float(W0)

    def mode_for(self, B: int, nprobe: int, k: Optional[int] = None, route: int = 0) -> int:
        ix = self.index
        if self.rule == "route":
            return choose_mode_route(ix, B, nprobe, k, route)
        if self.rule == "pairs":
            return choose_mode_pairs(B, nprobe, ix.nlist)
        return choose_mode(work_measure(B, nprobe, ix.N, ix.nlist, ix.D), self.W0)

    def search(self, xq: torch.Tensor, nprobe: int, **kw):
        mode = self.mode_for(int(xq.shape[0]), nprobe, kw.get("k"), kw.get("route", 0))
        return self.index.search(xq, nprobe, mode=mode, **kw) + (mode,)
