"""What a user of this framework has it do, as cases that can be timed and checked.

A case is one index of a stated size and one call into it: ``TridentV4Index.search`` on a batch of
queries (the cascade, mode 2, or the exhaustive exact scan, mode 10), ``CostRouter.search`` (the
mode chosen per batch) or ``SearchPipeline.run`` (queries and results in host memory).  The base
is either resident in HBM or in device-mapped host memory (out of core).

Sizes are those of the benchmark's configurations, taken at the scale where an index is built in a
second or two, and odd ones between them.  Every result is a top-K list whose ids and float32
distances are fixed by the data: the K smallest (float64 distance, id) of the probed lists, the
probes being the nprobe smallest (float64 distance, cluster).  So the tolerance is "exact".
"""
import math

import numpy as np
import torch

from trident_amd import SharedClusterStorage, TridentV4Index, choose_tile
from trident_amd.pipeline import SearchPipeline
from trident_amd.router import CostRouter

DEV = "cuda:0"


def _case(name, data, N, D, nlist, nprobe, B, K, mode=2, call="search", base="device", ub_seed=1, batch=0):
    c = dict(data=data, N=N, D=D, nlist=nlist, nprobe=nprobe, B=B, K=K, mode=mode, call=call, base=base,
             ub_seed=ub_seed, batch=batch)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one interactive query: latency and launches
        _case("single_query", "hist", 1_000_000, 128, 1024, 64, 1, 10),
        # an online server's small batch, clusters shared by few queries
        _case("few_queries", "hist", 1_000_000, 128, 1024, 64, 16, 10),
        # the same in many dimensions (GIST-like descriptors)
        _case("wide_few", "aniso", 200_000, 960, 512, 32, 24, 10),
        # a batch on a small index: fixed costs count
        _case("small_index", "gmm", 100_000, 128, 256, 16, 1000, 10),
        # the ordinary large batch on integer descriptors (SIFT-like)
        _case("batch", "hist", 1_000_000, 128, 1024, 64, 10_000, 10),
        # nothing round: rows, dimensions, lists, probes, queries, neighbours
        _case("ragged", "norm", 700_001, 100, 777, 37, 1237, 33),
        # a batch in many dimensions
        _case("wide_batch", "aniso", 300_000, 960, 512, 48, 1000, 10),
        # normalised float descriptors, many neighbours per query
        _case("deep_k100", "norm", 2_000_000, 96, 2048, 64, 5000, 100),
        # a small batch through the cost router, which sends it to the exhaustive exact scan
        _case("routed_few", "hist", 1_000_000, 128, 1024, 64, 40, 10, call="router", ub_seed=0),
        # the exhaustive exact scan of a large batch of float descriptors
        _case("exact_batch", "gmm", 1_000_000, 128, 1024, 32, 4000, 10, mode=10, ub_seed=0),
        # the base in host memory, bounds in HBM, exact rows over PCIe
        _case("out_of_core", "hist", 3_000_000, 128, 4096, 128, 10_000, 10, base="host"),
        # a query stream in host memory, two batches in flight
        _case("pipeline", "hist", 1_000_000, 128, 1024, 32, 20_000, 10, call="pipeline", batch=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the listed ones' ranges: an index of 50,000 to 2,000,000 rows in 33 to 960
    dimensions, batches of 1 to 10,000, each call, mode and placement."""
    kind = rng.choice(["search"] * 5 + ["router", "exact", "host", "pipeline"])
    wide = kind in ("search", "exact", "router") and rng.random() < 0.25
    data = "aniso" if wide else rng.choice(["hist", "gmm", "norm"])
    D = rng.choice([320, 384, 500, 768, 960]) if wide else rng.choice([33, 64, 96, 100, 128, 128, 160, 200])
    N = _log_int(rng, 50_000, 250_000 if wide else 2_000_000)
    nlist = int(math.sqrt(N) * rng.uniform(0.6, 1.6))
    nprobe = min(nlist // 2, _log_int(rng, 6, 160))
    B = _log_int(rng, 1, 10_000)
    K = rng.choice([1, 5, 10, 10, 10, 20, 50, 100])
    mode = 10 if kind == "exact" else 2
    batch = 0
    if kind == "router":
        B = _log_int(rng, 1, 200)
    if kind == "pipeline":
        B = _log_int(rng, 1000, 20_000)
        batch = max(1, B // rng.randint(2, 6))
    # no dearer than the largest listed case: rows visited times dimensions
    most = 1.2e10 if mode == 10 else 4e10
    B = max(1, min(B, int(most / (nprobe * (N / nlist) * D))))
    batch = min(batch, B)
    return _case(None, data, N, D, nlist, nprobe, B, K, mode=mode,
                 call=kind if kind in ("router", "pipeline") else "search",
                 base="host" if kind == "host" else "device", ub_seed=rng.choice([0, 1]), batch=batch)


def _rows(data, n, mu, basis, g):
    """n rows of a mixture around the centres mu: integer histograms in [0, 255], isotropic or
    anisotropic Gaussians, or anisotropic Gaussians normalised to length 1."""
    D = mu.shape[1]
    out = torch.empty((n, D), device=DEV)
    for s in range(0, n, 1 << 18):
        m = min(n, s + (1 << 18)) - s
        z = torch.randint(0, mu.shape[0], (m,), generator=g, device=DEV)
        if data == "hist":
            u = torch.randn((m, D), generator=g, device=DEV)
            x = torch.clamp(torch.round(mu[z] + 20.0 * u * u), 0.0, 255.0)  # gamma(1/2, 40)
        elif data == "gmm":
            x = mu[z] + 8.0 * torch.randn((m, D), generator=g, device=DEV)
        else:
            power = 0.6 if data == "aniso" else 0.5
            sl = torch.arange(1, D + 1, device=DEV, dtype=torch.float32).pow(-power)
            x = (torch.randn((m, D), generator=g, device=DEV) * sl) @ basis
            x = mu[z] + (x if data == "aniso" else 0.35 * x)
            if data == "norm":
                x = x / x.norm(dim=1, keepdim=True)
        out[s:s + m] = x
    return out


def _assign(x, cen):
    cn, ct = (cen.double() ** 2).sum(1).float(), cen.t().contiguous()
    return torch.cat([torch.argmin(cn - 2.0 * (x[s:s + (1 << 18)] @ ct), dim=1)
                      for s in range(0, x.shape[0], 1 << 18)])


def _data(case, seed):
    """Base, queries, centroids and the list of every row, from the seed alone (the sums of the
    k-means steps are taken in integers, so that they do not depend on their order)."""
    N, D, nlist, data = case["N"], case["D"], case["nlist"], case["data"]
    g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)
    n_mu = min(nlist, 1024)
    if data in ("hist", "gmm"):
        mu = (64.0 if data == "hist" else 100.0) * torch.rand((n_mu, D), generator=g, device=DEV)
    else:
        mu = (0.1 if data == "aniso" else 1.0) * torch.randn((n_mu, D), generator=g, device=DEV)
    basis = None
    if data in ("aniso", "norm"):
        h = torch.Generator().manual_seed(seed * 7919 + 19)
        basis = torch.linalg.qr(torch.randn((D, D), generator=h))[0].to(DEV)
    x = _rows(data, N, mu, basis, g)
    q = _rows(data, case["B"], mu, basis, g)
    train = x[torch.randperm(N, generator=g, device=DEV)[:min(N, 48 * nlist)]]
    cen = train[:nlist].clone()
    scale = 2.0 ** 24
    fixed = torch.round(train.double() * scale).long()
    for _ in range(4):
        a = _assign(train, cen)
        sums = torch.zeros((nlist, D), dtype=torch.int64, device=DEV).index_add_(0, a, fixed)
        cnt = torch.bincount(a, minlength=nlist)
        mean = (sums.double() / (cnt.clamp(min=1).double().unsqueeze(1) * scale)).float()
        cen = torch.where((cnt > 0).unsqueeze(1), mean, cen)
    return x, q, cen.contiguous(), _assign(x, cen)


class _HostBase:
    """Gives the mapped host memory of an out-of-core base back with the state that used it."""

    def __init__(self, storage):
        self.storage = storage

    def __del__(self):
        buf = getattr(self.storage, "_host_buf", None)
        if buf is not None:
            torch.cuda.synchronize()
            buf.free()
            self.storage._host_buf = None


def prepare(case, seed):
    x, q, cen, lid = _data(case, seed)
    N, D, nlist = case["N"], case["D"], case["nlist"]
    r = torch.empty(N, device=DEV)
    for s in range(0, N, 1 << 18):
        r[s:s + (1 << 18)] = (x[s:s + (1 << 18)] - cen[lid[s:s + (1 << 18)]]).norm(dim=1)
    # PCA of the residuals of a sample, as the index's rotation
    n = min(N, 20_000)
    res = (x[:n] - cen[lid[:n]]).double()
    mean = res.mean(0)
    cov = ((res - mean).t() @ (res - mean) / (n - 1)).cpu()
    rot = torch.linalg.eigh(cov)[1].flip(1).contiguous()
    st = SharedClusterStorage(x, lid, r, nlist, device=DEV, xb_placement=case["base"])
    del x, lid, r, res
    batch = case["batch"] or case["B"]
    ix = TridentV4Index(st, cen, mean.cpu(), rot, tile_size=choose_tile(D), device=DEV, max_batch=batch,
                        max_nprobe=max(case["nprobe"], 1), k=case["K"])
    state = dict(case=case, ix=ix, xq=q)
    if case["call"] == "router":
        state["router"] = CostRouter(ix)
    elif case["call"] == "pipeline":
        state["xq"] = q.cpu().numpy()
        state["pipe"] = SearchPipeline(ix, case["nprobe"], case["K"], batch, depth=2, ub_seed=case["ub_seed"])
    if case["base"] == "host":
        state["host"] = _HostBase(st)
    return state


def run(state):
    case, ix = state["case"], state["ix"]
    if case["call"] == "pipeline":
        d, i = state["pipe"].run(state["xq"])
    elif case["call"] == "router":
        d, i = state["router"].search(state["xq"], case["nprobe"], ub_seed=case["ub_seed"])[:2]
    else:
        d, i = ix.search(state["xq"], case["nprobe"], mode=case["mode"], ub_seed=case["ub_seed"])[:2]
    return {"distances": d, "ids": i}


def work(case):
    """Every probed list read once (a byte per dimension for the cascade, which reads codes; four
    for the exact scan), centroids, queries, the K exact rows of each query, results; one product
    per (query, probed row) and (query, centroid) and dimension, and the cascade's rotation."""
    N, D, nlist, nprobe, B, K = (case[k] for k in ("N", "D", "nlist", "nprobe", "B", "K"))
    pairs = B * nprobe * (N / nlist)
    rows = N * (1.0 - (1.0 - nprobe / nlist) ** B)  # rows of the lists that some query probes
    exact = case["mode"] == 10 or (case["call"] == "router" and B * nprobe < 8 * nlist)
    by = rows * D * (4 if exact else 1) + 4 * nlist * D + 4 * B * D + 12 * B * K
    fl = 2.0 * D * (pairs + B * nlist)
    if not exact:
        by += 4.0 * B * K * D + 4 * D * D
        fl += 2.0 * B * D * D
    return {"bytes": int(by), "flops": int(fl)}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The K nearest rows of the probed lists in float64: distances, and ids by (distance, id)."""
    x, q, cen, lid = _data(case, seed)
    B, K, nprobe, nlist = case["B"], case["K"], case["nprobe"], case["nlist"]
    q64, c64 = q.double(), cen.double()
    probes = torch.empty((B, nprobe), dtype=torch.int64, device=DEV)
    for s in range(0, B, 1024):
        d = (q64[s:s + 1024] ** 2).sum(1, keepdim=True) + (c64 ** 2).sum(1) - 2.0 * (q64[s:s + 1024] @ c64.t())
        probes[s:s + 1024] = torch.topk(d, nprobe, dim=1, largest=False).indices
    order = torch.argsort(lid, stable=True)
    off = [0] + torch.cumsum(torch.bincount(lid, minlength=nlist), 0).tolist()
    flat = torch.argsort(probes.reshape(-1), stable=True)
    poff = [0] + torch.cumsum(torch.bincount(probes.reshape(-1), minlength=nlist), 0).tolist()
    # integer data ties often: its distances are integers below 2^24, so distance 2^27 + id is
    # exact in float64 and orders by both
    tied = 2.0 ** 27 if case["data"] == "hist" else 0.0
    key = torch.full((B * nprobe, K), math.inf, dtype=torch.float64, device=DEV)
    ids = torch.full((B * nprobe, K), -1, dtype=torch.int64, device=DEV)
    for c in range(nlist):
        rows, pairs = order[off[c]:off[c + 1]], flat[poff[c]:poff[c + 1]]
        if rows.numel() == 0 or pairs.numel() == 0:
            continue
        xc, qc = x[rows].double(), q64[pairs // nprobe]
        d = (qc ** 2).sum(1, keepdim=True) + (xc ** 2).sum(1) - 2.0 * (qc @ xc.t())
        if tied:
            d = torch.round(d) * tied + rows.double()
        top = torch.topk(d, min(K, rows.numel()), dim=1, largest=False)
        key[pairs, :top.values.shape[1]] = top.values
        ids[pairs, :top.values.shape[1]] = rows[top.indices]
    best = torch.topk(key.view(B, nprobe * K), K, dim=1, largest=False)
    dist = torch.floor(best.values / tied) if tied else best.values
    out = {"distances": dist, "ids": torch.gather(ids.view(B, nprobe * K), 1, best.indices)}
    return {k: v.cpu().numpy() for k, v in out.items()} if case["call"] == "pipeline" else out
