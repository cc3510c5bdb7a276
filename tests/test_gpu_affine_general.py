"""The affine fill of pairs with gap-bit symbols at the edges of its stripes
and blocks, on one, two and four wavefronts a pair; outputs against the
oracle."""
import numpy as np
import pytest
import torch

import oracle
from poy5_amd import cost_matrix
from poy5_amd.batch import Batch, pack_pairs
from poy5_amd.sequence import Context

from test_gpu_linear_diag import seq

pytestmark = pytest.mark.gpu

CODES = np.array([1, 2, 4, 8, 1, 2, 4, 8, 15, 16, 17, 24, 31], np.uint8)


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def pairs_at_edges():
    rng = np.random.default_rng(29)
    pairs = []
    for a, b in ((1, 1), (1, 4), (2, 2), (2, 9), (3, 60), (16, 17), (63, 65), (64, 64), (65, 66),
                 (65, 200), (128, 130), (129, 129), (130, 400), (257, 300), (300, 330), (600, 640)):
        pairs.append((seq(rng, a, CODES), seq(rng, b, CODES)))
    for n, d in ((200, 0.02), (330, 0.1), (700, 0.05), (900, 0.2)):
        x = seq(rng, n, CODES)
        y = x[rng.random(len(x)) > d / 2]
        y = np.concatenate([x[:1], np.where(rng.random(len(y) - 1) < d, rng.choice(CODES, len(y) - 1),
                                            y[-(len(y) - 1):])]).astype(np.uint8)
        pairs.append((x, y) if len(x) <= len(y) else (y, x))
    return pairs


@pytest.mark.parametrize("go", [0, 3])
@pytest.mark.parametrize("per_cu", [0, 5, 9])
def test_general_fill_matches_the_oracle(ctx, per_cu, go):
    print(f"test_general_fill_matches_the_oracle per_cu={per_cu} go={go}", flush=True)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 2, go))
    ocm = oracle.cm_dna(1, 2, go)
    pairs = pairs_at_edges()
    want = [oracle.align_affine_3(x, y, ocm, 0) for x, y in pairs]
    # short pairs fill the launch up to `per_cu` pairs a CU
    rng = np.random.default_rng(30)
    short = [(seq(rng, 9, CODES), seq(rng, 12, CODES)) for _ in range(8)]
    n = per_cu * torch.cuda.get_device_properties(0).multi_processor_count
    every = pairs + [short[k % 8] for k in range(max(0, n - len(pairs)) + (1 if n else 0))]
    blob, o1, o2, l1, l2 = pack_pairs(every)
    b = Batch(ctx, "align_affine", l1, l2)
    cost, out, outlen = b.alloc_outputs()
    args = [torch.from_numpy(x).cuda() for x in (blob, o1, o2)]
    torch.cuda.synchronize()
    for _ in range(2):
        b.run(*args, cost, out, outlen)
        got, oh, lh = cost.cpu().numpy(), out.cpu().numpy(), outlen.cpu().numpy()
        for k, w in enumerate(want):
            where = (len(pairs[k][0]), len(pairs[k][1]))
            assert int(got[k]) == w["cost"], where
            for x, name in zip(b.unpack(oh, lh, k), ("resi", "resj", "median", "medianwg")):
                assert np.array_equal(x, w[name]), (where, name)
    b.close()
