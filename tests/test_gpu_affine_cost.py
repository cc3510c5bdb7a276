"""The full-plane affine cost at the edges of its stripes, blocks and
wavefronts, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from poy5_amd import cost_matrix
from poy5_amd.batch import Batch, pack_pairs
from poy5_amd.sequence import Context

from test_gpu_linear_diag import PLAIN, seq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()



@pytest.mark.parametrize("go", [0, 3])
def test_full_cost_at_block_and_stripe_edges(ctx, go):
    """The full-plane cost: lengths around the 64-row stripes, 16-step blocks
    and the pipeline of four wavefronts, gap-bit symbols, one-column pairs."""
    print(f"test_full_cost_at_block_and_stripe_edges go={go}", flush=True)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 2, go))
    ocm = oracle.cm_dna(1, 2, go)
    rng = np.random.default_rng(23)
    codes = np.array([1, 2, 4, 8, 3, 15, 16, 17, 24, 31], np.uint8)
    pairs = []
    for a, b in ((1, 1), (1, 2), (2, 2), (2, 3), (3, 70), (15, 16), (17, 17), (33, 48), (64, 65),
                 (65, 65), (66, 80), (129, 130), (257, 258), (258, 400), (300, 1100)):
        for c in (PLAIN, codes):
            pairs.append((seq(rng, a, c), seq(rng, b, c)))
            pairs.append((seq(rng, b, c), seq(rng, a, c)))
    blob, o1, o2, l1, l2 = pack_pairs(pairs)
    b = Batch(ctx, "cost_affine", l1, l2)
    cost, out, outlen = b.alloc_outputs()
    args = [torch.from_numpy(x).cuda() for x in (blob, o1, o2)]
    torch.cuda.synchronize()
    for _ in range(2):
        b.run(*args, cost, out, outlen)
        for (x, y), got in zip(pairs, cost.cpu().numpy()):
            assert int(got) == oracle.cost_affine_3(x, y, ocm), (len(x), len(y))
    b.close()
