"""Union merges whose columns a wavefront takes in chunks: counted runs around
the chunk's 64 entries, children that run out first, counts of another shape;
every array against the oracle."""
import numpy as np
import pytest

import oracle
from poy5_amd import unions
from poy5_amd.sequence import Context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def child(rng, moves, run, every, room, spoil):
    """A union of `moves` entries without a count, every `every`-th behind a
    run of `run` counted items; `room` unused entries in front."""
    off = []
    for m in range(moves):
        if run and m % every == 0:
            off += list(range(run, 0, -1))
        off.append(0)
    off = np.array(off[::-1], np.int32)
    if spoil and len(off):
        at = rng.integers(0, len(off), max(1, len(off) // 40))
        off[at] = rng.integers(0, 4, len(at))
    n = len(off)
    sym = rng.choice(np.array([1, 2, 4, 8, 17, 31], np.uint8), n)
    z = np.zeros(room + n, np.int32)
    return oracle.Union(np.concatenate([np.zeros(room, np.uint8), sym]), n,
                        np.concatenate([np.zeros(room, np.int32), off]), z, z)


@pytest.mark.parametrize("spoil", [False, True])
@pytest.mark.parametrize("run,every", [(0, 1), (1, 3), (5, 7), (62, 40), (63, 40), (64, 40),
                                       (65, 40), (200, 90)])
def test_chunks_match_the_oracle(ctx, run, every, spoil):
    print(f"test_chunks_match_the_oracle run={run} every={every} spoil={spoil}", flush=True)
    rng = np.random.default_rng(run * 2 + spoil)
    merges, want = [], []
    for n in (1, 2, 63, 64, 65, 127, 129, 300):
        for gaps in (0.0, 0.3, 0.9):
            for short in (0, 0, 1, 3):
                for close in (False, True):
                    u = rng.random(n)
                    a = np.where(u < gaps / 2, 16, rng.choice([1, 2, 4, 8], n)).astype(np.uint8)
                    b = np.where(u > 1 - gaps / 2, 16, rng.choice([1, 2, 4, 8], n)).astype(np.uint8)
                    med = np.where(rng.random(n) < gaps / 2, 16, a | b).astype(np.uint8)
                    med[0] = 16 if close else med[0] & 15 or 1
                    # as many entries as the columns move, some fewer or more
                    ma = int(np.sum(a != 16)) - (short if close else -short)
                    mb = int(np.sum((a == 16) | (b != 16)))
                    ua = child(rng, max(0, ma), run, every, n + 1, spoil)
                    ub = child(rng, max(0, mb), run // 2, every + 1, n + 1, spoil)
                    try:
                        want.append(oracle.union_merge(a, b, med, ua, ub))
                    except RuntimeError:
                        want.append(None)
                    merges.append((a, b, med, unions.Union(ua.seq, ua.length, ua.offset, ua.c1, ua.c2),
                                   unions.Union(ub.seq, ub.length, ub.offset, ub.c1, ub.c2)))
    assert any(w is not None for w in want)
    got = unions.union_level(ctx, merges)
    for g, w, m in zip(got, want, merges):
        assert (g is None) == (w is None), len(m[0])
        if w is None:
            continue
        assert g.length == w.length
        for f in ("seq", "offset", "c1", "c2"):
            assert np.array_equal(getattr(g, f), getattr(w, f)), (len(m[0]), f)
