"""The three-part bfloat16 form of the coarse pass (more than 128 dimensions), restated in numpy:
x = h + m + l + r, six products a dimension in three float32 accumulators (h h; h m, m h; h l, l h,
m m), against the bound the probe selection uses,
    |s' - q.c| <= kappa sum |q_d c_d|,
    kappa = (Dp + 6) 2^-23 (1 + 2^-7) + (2 Dp + 6) 2^-30 (1 + 2^-5) + (10 Dp + 20) 2^-39 + 4.2 2^-24,
and against float32 products summed the same way, which it must not be worse than.  Leaving out the
h m products must break the bound."""
import numpy as np
import pytest

from tests.test_band_split import _rows, bf16_rne


def _kappa(Dp):
    return ((Dp + 6) * 2.0 ** -23 * (1 + 2.0 ** -7) + (2 * Dp + 6) * 2.0 ** -30 * (1 + 2.0 ** -5)
            + (10 * Dp + 20) * 2.0 ** -39 + 4.2 * 2.0 ** -24)


def _parts(x):
    h = bf16_rne(x)
    m = bf16_rne((x - h).astype(np.float32))
    return h, m, bf16_rne((x - h - m).astype(np.float32))


def _chain(pairs, rng):
    """One float32 accumulator: each 32-dim step adds its products (exact in float64 for bfloat16
    parts, rounded to float32 for float32 values) in a random order."""
    acc = np.float32(0.0)
    Dp = pairs[0][0].size
    for s in range(0, Dp, 32):
        for a, b in pairs:
            for t in rng.permutation((a[s:s + 32].astype(np.float64) * b[s:s + 32]).astype(np.float32)):
                acc = np.float32(acc + t)
    return acc


def _errors(kind, D, seed, drop_mid=False):
    rng = np.random.default_rng([seed, D])
    Dp = 32 * ((D + 31) // 32)
    rows = np.zeros((2, Dp), np.float32)
    rows[:, :D] = _rows(rng, kind, D)
    q, c = rows
    (qh, qm, ql), (ch, cm, cl) = _parts(q), _parts(c)
    prod = q.astype(np.float64) * c
    den = np.abs(prod).sum()
    mid = _chain([(ch, qm), (cm, qh)], rng) if not drop_mid else np.float32(0.0)
    s = np.float32(_chain([(ch, qh)], rng) + np.float32(mid + _chain([(ch, ql), (cm, qm), (cl, qh)], rng)))
    f = _chain([(c, q)], rng)
    return abs(float(s) - prod.sum()) / den, abs(float(f) - prod.sum()) / den


@pytest.mark.parametrize("kind", ["gauss", "uniform", "coherent", "below_next"])
@pytest.mark.parametrize("D", [130, 960])
def test_three_parts_within_bound_and_no_worse_than_float32(kind, D):
    e = np.array([_errors(kind, D, s) for s in range(12)])
    assert e[:, 0].max() <= _kappa(32 * ((D + 31) // 32))
    # both are float32 accumulations of the same length: the same error up to chance (12 draws of
    # each; the maxima of two such samples differ by less than a factor of two)
    assert e[:, 0].max() <= 2.0 * e[:, 1].max() + 2.0 ** -24, (e[:, 0].max(), e[:, 1].max())


def test_dropped_products_break_the_bound():
    assert max(_errors("coherent", 130, s, drop_mid=True)[0] for s in range(4)) > _kappa(160)
