"""The anti-diagonal affine fill of gap-free pairs at the edges of its forms:
lengths around its loads and blocks, bands around the lane counts of one, four
and sixteen wavefronts, pairs it hands on; outputs against the oracle, and
rounds, band and cells against the stripe fills."""
import numpy as np
import pytest
import torch

import oracle
from poy5_amd import autotune, cost_matrix
from poy5_amd.batch import Batch, pack_pairs
from poy5_amd.sequence import Context

from test_gpu_linear_diag import PLAIN, related, seq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def base_pairs():
    rng = np.random.default_rng(21)
    iupac = np.array([1, 2, 4, 8, 1, 2, 4, 8, 3, 15], np.uint8)
    pairs = []
    for a, b in ((1, 1), (1, 5), (2, 2), (2, 9), (3, 40), (7, 8), (8, 7), (9, 30), (16, 16),
                 (63, 64), (64, 63), (65, 130), (126, 125), (128, 200)):
        pairs.append((seq(rng, a), seq(rng, b)))
        pairs.append((seq(rng, a, iupac), seq(rng, b, iupac)))
    for n in (60, 130, 250, 300, 600):
        for d in (0.0, 0.05, 0.3):
            pairs.append(related(rng, n, d))
    for n in (1200, 2600):
        for d in (0.1, 0.4):
            pairs.append(related(rng, n, d))
    # bands past one and four wavefronts
    pairs += [(seq(rng, 700), seq(rng, 1500)), (seq(rng, 1500), seq(rng, 1400)),
              (seq(rng, 400), seq(rng, 2400))]
    return pairs


def run(ctx, pairs):
    blob, o1, o2, l1, l2 = pack_pairs(pairs)
    b = Batch(ctx, "align_affine", l1, l2)
    cost, out, outlen = b.alloc_outputs()
    args = [torch.from_numpy(x).cuda() for x in (blob, o1, o2)]
    torch.cuda.synchronize()
    b.run(*args, cost, out, outlen)
    cells, _, rounds, newk = b.stats()
    oh, lh = out.cpu().numpy(), outlen.cpu().numpy()
    outs = [b.unpack(oh, lh, k) for k in range(len(pairs))]
    b.close()
    return cost.cpu().numpy(), outs, cells, rounds, newk


@pytest.mark.parametrize("model,copies", [((1, 1, 3), 1), ((1, 1, 3), 7), ((2, 1, 0), 7),
                                          ((1, 1, 3), 36), ((900, 1000, 3000), 1)])
def test_forms_match_oracle_and_stripes(ctx, model, copies):
    print(f"test_forms_match_oracle_and_stripes {model} x{copies}", flush=True)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(*model))
    ocm = oracle.cm_dna(*model)
    base = base_pairs()
    if model[0] > 100:
        # costs whose sums do not fit a key, below POY's HIGH_NUM (10^6)
        base = [p for p in base if len(p[0]) + len(p[1]) < 700]
    pairs = base * copies
    costs, outs, cells, rounds, newk = run(ctx, pairs)
    autotune.set_knobs(ctx, {"affine_rotating": 0})
    try:
        c0, o0, cells0, rounds0, newk0 = run(ctx, base)
    finally:
        autotune.set_knobs(ctx, {"affine_rotating": 1})
    for k, (a, b) in enumerate(base):
        sw = len(a) > len(b)
        si, sj = (b, a) if sw else (a, b)
        ref = oracle.align_affine_3(si, sj, ocm, int(sw))
        ra, rb = (ref["resj"], ref["resi"]) if sw else (ref["resi"], ref["resj"])
        for q in (k, k + (copies - 1) * len(base)):
            what = (k, q, len(a), len(b))
            assert int(costs[q]) == ref["cost"] == int(c0[k]), what
            for got, want in zip(outs[q], (ra, rb, ref["median"], ref["medianwg"])):
                assert np.array_equal(got, want), what
            assert (rounds[q], newk[q], cells[q]) == (rounds0[k], newk0[k], cells0[k]), what


def test_band_edges_in_every_halo_lane(ctx):
    """Four wavefronts per pair, length differences that put the band's last
    lane everywhere around a wavefront's end."""
    print("test_band_edges_in_every_halo_lane", flush=True)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 1, 3))
    rng = np.random.default_rng(22)
    pairs = []
    for k in range(300):
        root = rng.choice(PLAIN, 420 + k)
        a = np.concatenate([[16], root])
        at = int(rng.integers(1, len(a)))
        b = np.concatenate([a[:at], rng.choice(PLAIN, 90 + k), a[at:]])
        b[1:][rng.random(len(b) - 1) < 0.15] = 2
        pairs.append((a.astype(np.uint8), b.astype(np.uint8)))
    costs, outs, cells, rounds, newk = run(ctx, pairs)
    autotune.set_knobs(ctx, {"affine_rotating": 0})
    try:
        c0, o0, cells0, rounds0, newk0 = run(ctx, pairs)
    finally:
        autotune.set_knobs(ctx, {"affine_rotating": 1})
    assert np.array_equal(costs, c0) and np.array_equal(cells, cells0)
    assert np.array_equal(rounds, rounds0) and np.array_equal(newk, newk0)
    for x, y in zip(outs, o0):
        assert all(np.array_equal(p, q) for p, q in zip(x, y))


def test_second_round_keeps_the_optimum(ctx):
    """A pair whose doubling runs two computed rounds (half-widths 18 and 42):
    the rotating stripe fill's second round returns 87, below the full
    matrix's optimum of 88."""
    print("test_second_round_keeps_the_optimum", flush=True)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 1, 3))
    ocm = oracle.cm_dna(1, 1, 3)
    digits = "0123456789ABCDEFG"
    a, b = (np.array([digits.index(c) for c in s], np.uint8) for s in (
        "G822248488A222122811224B212242422221226221811481421841814428282221182444881D81482284812444414218212144481184822128821841",
        "G8111282222282244922144418218D14114218418144148322114424844482814811822448124448412822121184B18818248188218413284844432A88828441821"))
    ref = oracle.align_affine_3(a, b, ocm, 0)
    assert ref["cost"] == oracle.cost_affine_3(a, b, ocm) == 88
    for copies in (1, 300, 1600):
        costs, outs, _, _, _ = run(ctx, [(a, b)] * copies)
        assert np.all(costs == 88), copies
        assert np.array_equal(outs[-1][0], ref["resi"]) and np.array_equal(outs[-1][1], ref["resj"])
