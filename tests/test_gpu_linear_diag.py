"""The anti-diagonal linear fill at the edges of its forms: lengths around its
8-symbol loads and 16-step blocks, bands around the lane counts of one, four
and sixteen wavefronts, pairs it hands on, both tie orders, costs that do not
fit a key, tail costs below the deletion costs; bit-exact against the oracle."""
import copy

import numpy as np
import pytest

import oracle
from poy5_amd import cost_matrix
from poy5_amd.batch import run_pairs
from poy5_amd.sequence import Context

pytestmark = pytest.mark.gpu

PLAIN = np.array([1, 2, 4, 8], np.uint8)
CODES = np.array([1, 2, 4, 8, 1, 2, 4, 8, 5, 15, 17, 24], np.uint8)


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def seq(rng, n, codes=PLAIN):
    return np.concatenate([[16], rng.choice(codes, n - 1)]).astype(np.uint8)


def related(rng, n, d):
    """A pair of about n symbols with substitutions and indels at rate d."""
    root = rng.choice(PLAIN, n)
    out = []
    for _ in range(2):
        s = root.copy()
        m = rng.random(n) < d
        s[m] = rng.choice(PLAIN, int(m.sum()))
        s = s[rng.random(n) >= d / 4]
        at = int(rng.integers(0, len(s) + 1))
        ins = rng.choice(PLAIN, int(rng.integers(0, 1 + int(n * d / 3))))
        out.append(np.concatenate([[16], s[:at], ins, s[at:]]).astype(np.uint8))
    return tuple(out)


def small_pairs():
    rng = np.random.default_rng(11)
    pairs = []
    for a, b in ((1, 1), (1, 5), (2, 2), (2, 9), (3, 40), (7, 8), (8, 7), (8, 8), (9, 30), (15, 17),
                 (16, 16), (63, 64), (64, 63), (65, 130), (120, 124), (126, 125), (128, 200)):
        pairs.append((seq(rng, a), seq(rng, b)))
        pairs.append((seq(rng, a, CODES), seq(rng, b, CODES)))
    for n in (60, 130, 250, 251, 300):
        for d in (0.0, 0.02, 0.1, 0.3):
            pairs.append(related(rng, n, d))
    return pairs


def wide_pairs():
    """Bands past one, four and sixteen wavefronts' narrow forms."""
    rng = np.random.default_rng(12)
    pairs = [related(rng, n, d) for n in (500, 900) for d in (0.05, 0.3)]
    pairs += [(seq(rng, 700), seq(rng, 760)), (seq(rng, 1150), seq(rng, 1100)),
              (seq(rng, 600), seq(rng, 1500))]
    return pairs


def tables(name):
    if name == "big":   # a value and a count do not share 32 bits
        return cost_matrix.of_transformations_and_gaps(3000, 5000), oracle.cm_dna(3000, 5000)
    m, o = cost_matrix.of_transformations_and_gaps(2, 3), oracle.cm_dna(2, 3)
    if name == "tails":  # ending in a gap is cheaper than inside
        m = copy.deepcopy(m)
        for k in range(1, 32):
            t = max(int(m.tail[k]) - 1, 0)
            m.tail[k] = t
            o.tail[k] = t
    return m, o


@pytest.mark.parametrize("table,copies", [("plain", 1), ("plain", 8), ("plain", 32), ("big", 1),
                                          ("tails", 1)])
def test_forms_match_oracle(ctx, table, copies):
    print(f"test_forms_match_oracle {table} x{copies}", flush=True)
    m, ocm = tables(table)
    ctx.set_cm(m)
    base = small_pairs() + wide_pairs()
    pairs = base * copies
    costs, outs = run_pairs(ctx, "align_2d", pairs)
    only, _ = run_pairs(ctx, "cost_2d", pairs)
    assert np.array_equal(only, costs)
    for k, (a, b) in enumerate(base):
        p1, p2, c, _ = oracle.align_2(a, b, ocm)
        an = oracle.ancestor_2(p1, p2, ocm)
        mw = oracle.median_2_with_gaps(p1, p2, ocm)
        for q in (k, k + (copies - 1) * len(base)):
            assert int(costs[q]) == c, (k, len(a), len(b))
            for got, want in zip(outs[q], (p1, p2, an, mw)):
                assert np.array_equal(got, want), (k, len(a), len(b))


@pytest.mark.parametrize("copies", [1, 32])
def test_deltaw_and_small_budget(ctx, copies):
    """DOS.distance's band hint, and the two-phase plan of a small budget."""
    print(f"test_deltaw_and_small_budget x{copies}", flush=True)
    m, ocm = tables("plain")
    ctx.set_cm(m)
    base = small_pairs() + wide_pairs()
    pairs = base * copies
    dw = [max(abs(len(a) - len(b)), 8) for a, b in pairs]
    costs, _ = run_pairs(ctx, "cost_2d", pairs, deltaw=dw)
    budget = 1 << 21
    two, outs = run_pairs(ctx, "align_2d", pairs, dm_budget=budget)
    for k, (a, b) in enumerate(base):
        assert int(costs[k]) == oracle.cost_2(a, b, ocm, dw[k])[0], k
        p1, p2, c, _ = oracle.align_2(a, b, ocm)
        assert int(two[k]) == c, k
        assert np.array_equal(outs[k][0], p1) and np.array_equal(outs[k][1], p2), k
