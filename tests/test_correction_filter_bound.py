"""The error bound of the correction's nearest-element filter (gg_correct.hip), its arithmetic restated: a
barycenter's row is three BF16 pieces of each of -2q' and R, a voxel's column its small integer offsets and 1,
and the matrix product adds their 12 products in an order and with a rounding that are the hardware's.  Whatever
they are, as long as each rounding is within one unit of the last place, the filter's value may be no further
from the exact one than kFilterEps times the bound S of the terms' sum.  Every box side, near and far from the
plane x = y, truncating and away-from-zero adders, added one after the other in several orders, pairwise, and
as blocks of aligned terms.
"""
import os
import re

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gragles_3d_amd", "csrc",
                   "gg_correct.hip")


def filter_eps():
    m = re.search(r"constexpr float kFilterEps = (\d+)\.0f / (\d+)\.0f;", open(SRC).read())
    return int(m.group(1)) / int(m.group(2))


def bf16(x):
    b = np.asarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000
    return b.astype(np.uint32).view(np.float32).astype(np.float64)


def pieces(v):
    out, rest = [], v
    for _ in range(3):
        p = bf16(rest)
        out.append(p)
        rest = rest - p
    return out, rest


def ulp(x):
    return 2.0 ** (np.floor(np.log2(np.maximum(np.abs(x), 1e-300))) - 23)


def cut(x, unit, away):
    """x as a multiple of unit, toward zero or away from it."""
    f = np.ceil if away else np.floor
    return np.sign(x) * f(np.abs(x) / unit) * unit


def add_chain(t, away):
    s = t[0]
    for x in t[1:]:
        s = s + x
        s = cut(s, ulp(s), away)
    return s


def add_pairs(t, away):
    while len(t) > 1:
        t = [cut(a + b, ulp(a + b), away) for a, b in zip(t[::2], t[1::2])] + ([t[-1]] if len(t) % 2 else [])
    return t[0]


def add_aligned(t, block, away):
    """Blocks of terms and the accumulator cut at the last place of the largest, then the sum cut."""
    acc = np.zeros_like(t[0])
    for k in range(0, len(t), block):
        part = t[k:k + block] + ([acc] if k else [])
        unit = ulp(np.max(np.abs(part), axis=0))
        acc = np.sum([cut(x, unit, away) for x in part], axis=0)
        acc = cut(acc, ulp(acc), away)
    return acc


def rows_and_columns(side, dx, rng, n=4000):
    half = side // 2
    q = rng.uniform(-half - 1, half + 1, size=(n, 3))
    d = np.array([dx, -dx, 0.0])
    r = np.sum(q * q, axis=1) + 2.0 * q @ d
    p = rng.integers(-half, half + 1, size=(n, 3)).astype(np.float64)
    rho = np.sqrt(np.max(np.sum(q * q, axis=1)))
    s = rho * rho + 2.0 * rho * (np.sqrt(2.0) * abs(dx) + np.sqrt(np.sum(p * p, axis=1)))
    return q, r, p, s


@pytest.mark.parametrize("dx", [0, 3, 40, 400, 1100])
@pytest.mark.parametrize("side", [8, 16, 24, 32, 33, 48, 64, 96])
def test_filter_error_is_below_its_bound(side, dx):
    rng = np.random.default_rng(1000 * side + dx)
    q, r, p, s = rows_and_columns(side, dx, rng)
    terms, left = [], 0.0
    for a in range(3):
        ps, rest = pieces(-2.0 * q[:, a])
        terms += [x * p[:, a] for x in ps]
        left = left + np.abs(rest * p[:, a])
    ps, rest = pieces(r)
    terms += ps
    left = left + np.abs(rest)
    exact = r - 2.0 * np.sum(q * p, axis=1)
    assert np.all(np.sum(np.abs(terms), axis=0) <= 1.01 * s)
    assert np.all(left <= 2.0 ** -24 * s)
    by_size = list(np.take_along_axis(np.array(terms), np.argsort(-np.abs(terms), axis=0), axis=0))
    worst = 0.0
    for away in (False, True):
        for got in (add_chain(terms, away), add_chain(terms[::-1], away), add_chain(by_size, away),
                    add_pairs(terms, away), add_aligned(terms, 4, away), add_aligned(terms, 8, away),
                    add_aligned(terms, 12, away)):
            worst = max(worst, float(np.max(np.abs(got - exact) / s)))
    assert worst <= filter_eps(), worst * 2 ** 24


def test_bound_holds_for_every_order():
    """12 roundings of one unit in the last place of a sum of at most 1.01 S, and what the pieces leave."""
    assert 12 * 2.0 ** -23 * 1.01 + 2.0 ** -24 <= filter_eps()
