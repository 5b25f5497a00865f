"""Mode 10's thresholds (K <= 16) are float32 bounds without a loss: which rows a search lists is
computed here from the kernel's definition."""
import math

import numpy as np
import pytest
import torch

from tests.helpers import assert_exact, build_index, oracle_search

D = 32


def _row(norm2):
    """Integers whose squares sum to norm2 (every product and sum of them is exact in float32)."""
    x = np.zeros(D, np.float32)
    for d in range(D):
        x[d] = math.isqrt(norm2)
        norm2 -= math.isqrt(norm2) ** 2
    assert norm2 == 0
    return x


def _bounds(n2):
    """(lb, ub) of a row with |x|^2 = n2 from the query 0: base = S = n2, E = fma(2^-20, S, D 2^-100)
    (1 + 2^-20), every operation rounded to float32 (fma: the sum of two values 2^20 apart and more)."""
    f = np.float32
    E = f(f(2.0 ** -20 * n2 + D * 2.0 ** -100) * f(1.0 + 2.0 ** -20))
    return max(f(f(n2) - E), f(0.0)), f(f(n2) + E)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [16, 5, 1])
@pytest.mark.parametrize("tie", [0, 3])
def test_listed_rows(dev, K, tie):
    """The nearest list's 16 rows set the threshold, the K-th smallest ub of them (the last 1 + tie of
    its K smallest equal); of the second list, whose norms go up by one, the rows with lb <= it are listed."""
    X = 1 << 23
    first = sorted([X - 40 * i for i in range(max(K - 1 - tie, 0))] + [X] * (min(tie, K - 1) + 1) +
                   [X + 5000 + i for i in range(16 - K)])
    second = [X + i for i in range(1, 65)]
    xb = torch.as_tensor(np.stack([_row(n) for n in first + second]))
    lid = np.repeat([0, 1], [16, 64])
    cen = np.zeros((2, D), np.float32)
    cen[1, 0] = 1.0
    b = build_index(xb, 2, dev, list_ids=lid, centroids=cen, max_batch=8)
    xq = np.zeros((1, D), np.float32)
    t = _bounds(first[K - 1])[1]
    want = sum(_bounds(n)[0] <= t for n in first + second)
    assert 16 >= sum(n <= X for n in first) >= K and 10 <= want < 60
    stats = torch.zeros(4, dtype=torch.int64, device=dev)
    d, i, _ = b.ix.search(torch.as_tensor(xq).to(dev), 2, mode=10, k=K, route=2, stats_buf=stats)
    torch.cuda.synchronize()
    _, rd, ri = oracle_search(b, xq, 2, K)
    assert_exact(d.cpu().numpy(), i.cpu().numpy(), rd, ri, f"K={K}")
    assert int(stats[2]) == want, (int(stats[2]), want)
