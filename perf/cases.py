"""What this library's speed is judged by: the calls a tree search makes of it,
from one pair through the per-pair entry points to the levels, batches and
serving traffic of large searches.

A case names a *kind* of call and the ranges its inputs are drawn from.
``prepare`` makes the inputs on the device (or the host, for the entry points
that take host sequences) and the plan or handle a program keeps between
calls; ``run`` makes one call and returns everything it computes.

Kinds
    pair      one alignment through ``Align`` (host sequences in and out)
    batch     many pairs on device-resident sequences (``Batch``)
    triples   many triples through the 3D cube (``Batch3``)
    readjust  one level of ``Sequence.readjust`` (host sequences in and out)
    union     one level of union merges (``unions.Level``)
    rejoin    an SPR round's rejoin costs through the server (``Server``)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from poy5_amd import cost_matrix, readjust, spr, unions
from poy5_amd.batch import Batch, Batch3
from poy5_amd.sequence import Align, Context
from poy5_amd.serve import Server

GAP = 16
BASES = np.array([1, 2, 4, 8], np.uint8)
IUPAC = np.array([3, 5, 9, 6, 10, 12, 7, 11, 13, 14, 15], np.uint8)

# int32 operations a DP cell cannot do without: full affine cost, affine with
# the backtrace's flags, linear, 3D
OPS = {"cost_affine": 22, "align_affine": 35, "newkk_align": 35, "newkk_cost": 22,
       "align_2d": 6, "cost_2d": 6, "align_3d": 14}
AFFINE = ("align_affine", "cost_affine", "newkk_align", "newkk_cost")


def _batch(name, op, pairs, lo, hi, dlo, dhi, *, log=False, iupac=0.05, gaps=0.0, trans=1,
           indel=1, opening=3, budget_gb=0):
    return {"name": name, "kind": "batch", "op": op, "pairs": pairs, "lo": lo, "hi": hi,
            "log": log, "dlo": dlo, "dhi": dhi, "iupac": iupac, "gaps": gaps, "trans": trans,
            "indel": indel, "opening": opening if op in AFFINE else 0, "budget_gb": budget_gb}


def listed():
    return [
        # the smallest call: a short marker's alignment, one pair at a time
        {"name": "pair_affine_short", "kind": "pair", "op": "align_affine", "lo": 80, "hi": 150,
         "dlo": 0.02, "dhi": 0.25, "iupac": 0.05, "gaps": 0.0, "trans": 1, "indel": 1,
         "opening": 3},
        # an ordinary gene, cost then backtrace through align_2
        {"name": "pair_linear_gene", "kind": "pair", "op": "align_2d", "lo": 1400, "hi": 1600,
         "dlo": 0.02, "dhi": 0.15, "iupac": 0.05, "gaps": 0.0, "trans": 1, "indel": 2,
         "opening": 0},
        # the medians of one level of a mid-sized search, linear costs
        _batch("linear_1k", "align_2d", 1024, 300, 700, 0.13, 0.13, trans=1, indel=2),
        # long sequences with band doubling, planned in two phases within a
        # direction-store budget
        _batch("linear_long", "align_2d", 128, 16000, 100000, 0.01, 0.08, iupac=0.10,
               budget_gb=16),
        # uneven affine pairs over two orders of magnitude of length
        _batch("affine_uneven", "align_affine", 16384, 50, 5000, 0.02, 0.25, log=True),
        # inner nodes of an affine search: medians that carry gap bits
        _batch("affine_medians", "align_affine", 2048, 200, 2000, 0.02, 0.15, gaps=0.03),
        # DOS.distance under affine costs: the full DP's cost only
        _batch("affine_cost", "cost_affine", 2048, 300, 1800, 0.02, 0.15, gaps=0.01),
        # DOS.median's use_ukk branch: the diagonal-store aligner
        _batch("ukk_uneven", "newkk_align", 8192, 50, 5000, 0.02, 0.25, log=True),
        # three-way alignments of a node's neighbours
        {"name": "triples", "kind": "triples", "triples": 256, "lo": 200, "hi": 1000,
         "dlo": 0.03, "dhi": 0.15, "trans": 1, "indel": 1},
        # one level of node readjustment
        {"name": "readjust_level", "kind": "readjust", "nodes": 1024, "lo": 200, "hi": 1000,
         "dlo": 0.03, "dhi": 0.15, "trans": 1, "indel": 1, "opening": 0},
        # one level of unions over tip pairs
        {"name": "union_level", "kind": "union", "merges": 4096, "lo": 50, "hi": 5000,
         "dlo": 0.02, "dhi": 0.25},
        # pricing the rejoin edges of SPR clips on pool-resident medians
        {"name": "rejoin", "kind": "rejoin", "taxa": 48, "root": 1500, "requests": 4000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "batch", "batch", "batch", "batch", "long", "triples",
                       "readjust", "union", "rejoin"])
    dlo = rng.uniform(0.01, 0.12)
    dhi = rng.uniform(dlo, 0.25)
    if kind == "pair":
        op = rng.choice(["align_affine", "align_2d", "cost_2d", "cost_affine"])
        lo = _log(rng, 30, 4000)
        return {"kind": "pair", "op": op, "lo": lo, "hi": int(lo * rng.uniform(1.0, 1.25)),
                "dlo": dlo, "dhi": dhi, "iupac": 0.05, "gaps": rng.choice([0.0, 0.02]),
                "trans": 1, "indel": rng.choice([1, 2]),
                "opening": rng.choice([2, 3]) if op in AFFINE else 0}
    if kind == "batch":
        op = rng.choice(["align_2d", "cost_2d", "align_affine", "align_affine", "cost_affine",
                         "newkk_align"])
        lo = _log(rng, 50, 1200)
        hi = min(5000, _log(rng, lo, 10 * lo))
        # no more cells than the largest listed batch of the kind
        most = 4e9 if op == "cost_affine" else 2e10
        pairs = _log(rng, 64, max(64, min(16384, int(most / (hi * hi) * 2))))
        c = _batch("", op, pairs, lo, hi, dlo, dhi, log=rng.random() < 0.5,
                   gaps=rng.choice([0.0, 0.0, 0.02]), indel=rng.choice([1, 2]),
                   opening=rng.choice([2, 3]))
        del c["name"]
        return c
    if kind == "long":
        lo = _log(rng, 8000, 50000)
        c = _batch("", "align_2d", _log(rng, 16, 200), lo, min(100000, 2 * lo),
                   min(dlo, 0.04), min(dhi, 0.08), iupac=0.10, budget_gb=16)
        del c["name"]
        return c
    if kind == "triples":
        lo = _log(rng, 60, 600)
        return {"kind": "triples", "triples": _log(rng, 16, 200), "lo": lo,
                "hi": int(lo * rng.uniform(1.0, 1.5)), "dlo": min(dlo, 0.1),
                "dhi": min(max(dhi, 0.03), 0.15), "trans": 1, "indel": rng.choice([1, 2])}
    if kind == "readjust":
        lo = _log(rng, 60, 700)
        return {"kind": "readjust", "nodes": _log(rng, 64, 1024), "lo": lo,
                "hi": int(lo * rng.uniform(1.0, 2.0)), "dlo": min(dlo, 0.1),
                "dhi": min(max(dhi, 0.03), 0.15), "trans": 1, "indel": rng.choice([1, 2]),
                "opening": rng.choice([0, 0, 3])}
    if kind == "union":
        lo = _log(rng, 50, 1000)
        return {"kind": "union", "merges": _log(rng, 64, 4096), "lo": lo,
                "hi": min(5000, _log(rng, lo, 10 * lo)), "dlo": dlo, "dhi": dhi}
    return {"kind": "rejoin", "taxa": rng.randrange(16, 48), "root": _log(rng, 300, 1800),
            "requests": _log(rng, 500, 4000)}


# ---- inputs ------------------------------------------------------------------


def _root_lengths(case, n, rng):
    if case.get("log") or case["kind"] == "union":
        x = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"] + 1), n))
        return np.minimum(x.astype(np.int64), case["hi"])
    return rng.integers(case["lo"], case["hi"] + 1, n)


def _mutate(root, owner, n, div, iupac, gaps, rng):
    """One descendant of every root: substitutions and indel events in the
    ratio 10:3, indels of geometric length (mean 3), half of them deletions;
    then multi-base and gap-carrying codes.  Returns (symbols with a leading
    gap per sequence, lengths)."""
    m = len(root)
    d = div[owner]
    sub = rng.random(m, np.float32) < d * (10.0 / 13.0)
    base = np.where(sub, (root + rng.integers(1, 4, m, np.uint8)) & 3, root)
    event = np.flatnonzero(rng.random(m, np.float32) < d * (3.0 / 13.0))
    run = rng.geometric(1.0 / 3.0, len(event))
    insert = rng.random(len(event)) < 0.5
    copies = np.ones(m, np.int64)
    # a deletion covers `run` root symbols, within its own sequence
    ends = np.cumsum(np.bincount(owner, minlength=n))[owner]
    at, ln = event[~insert], run[~insert]
    cover = np.zeros(m + 1, np.int64)
    np.add.at(cover, at, 1)
    np.add.at(cover, np.minimum(at + ln, ends[at]), -1)
    copies[np.cumsum(cover[:-1]) > 0] = 0
    np.add.at(copies, event[insert], run[insert])
    # every sequence keeps a symbol after its leading gap
    first = np.concatenate([[True], owner[1:] != owner[:-1]])
    copies[first] = np.maximum(copies[first], 1)
    src = np.repeat(np.arange(m), copies)
    own = owner[src]
    last = np.concatenate([src[1:] != src[:-1], [True]])
    code = np.where(last, base[src], rng.integers(0, 4, len(src), np.uint8))
    code = BASES[code]
    if iupac > 0:
        k = np.flatnonzero(rng.random(len(src), np.float32) < iupac)
        code[k] = IUPAC[rng.integers(0, len(IUPAC), len(k))]
    if gaps > 0:
        k = np.flatnonzero(rng.random(len(src), np.float32) < gaps)
        code[k] |= GAP
    length = np.bincount(own, minlength=n) + 1
    out = np.empty(len(src) + n, np.uint8)
    start = np.cumsum(length) - length
    out[start] = GAP
    out[np.arange(len(src)) + own + 1] = code
    return out, length


def _family(case, n, members, seed):
    """`members` descendants of each of n random roots: (blob, offsets[members],
    lengths[members])."""
    rng = np.random.default_rng(seed)
    rl = _root_lengths(case, n, rng)
    owner = np.repeat(np.arange(n), rl)
    root = rng.integers(0, 4, int(rl.sum()), np.uint8)
    div = rng.uniform(case["dlo"], case["dhi"], n).astype(np.float32)
    blobs, offs, lens, at = [], [], [], 0
    for _ in range(members):
        b, ln = _mutate(root, owner, n, div, case.get("iupac", 0.0), case.get("gaps", 0.0), rng)
        offs.append(np.cumsum(ln) - ln + at)
        at += len(b)
        blobs.append(b)
        lens.append(ln.astype(np.int32))
    return np.concatenate(blobs), offs, lens


def _host(blob, offs, lens, k):
    return tuple(blob[o[k]:o[k] + ln[k]].copy() for o, ln in zip(offs, lens))


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _room(case, n, members):
    """Symbols that hold n families of `members` descendants of the case's
    roots, the same for every seed (so results of one case have one size):
    the expected total, a quarter more, and some of the longest."""
    lo, hi = case["lo"], case["hi"]
    log = (case.get("log") or case["kind"] == "union") and hi > lo
    mean = (hi - lo) / math.log(hi / lo) if log else (lo + hi) / 2
    return int(members * (n * (1.25 * mean + 8) + 8 * hi))


def _padded(x, size):
    out = np.zeros(max(size, len(x)), x.dtype)
    out[:len(x)] = x
    return out


def _zeros(need, size):
    return torch.zeros(max(need, size), dtype=torch.uint8, device="cuda")


def _context(case):
    ctx = Context(0)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(
        case["trans"], case["indel"], case["opening"] if case.get("opening") else None))
    return ctx


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pair":
        blob, offs, lens = _family(case, 1, 2, seed)
        a, b = _host(blob, offs, lens, 0)
        return {"case": case, "align": Align(_context(case)), "a": a, "b": b,
                "room": 2 * _room(case, 1, 1)}
    if kind == "batch":
        blob, offs, lens = _family(case, case["pairs"], 2, seed)
        ctx = _context(case)
        b = Batch(ctx, case["op"], lens[0], lens[1], dm_budget=case["budget_gb"] << 30)
        cost, out, outlen = b.alloc_outputs()
        if b.out_bytes:
            out = _zeros(b.out_bytes, 4 * (_room(case, b.n, 2) + 8 * b.n))
        s = {"case": case, "ctx": ctx, "batch": b,
             "args": (_dev(blob), *[_dev(o) for o in offs], cost, out, outlen)}
        torch.cuda.synchronize()
        return s
    if kind == "triples":
        blob, offs, lens = _family(case, case["triples"], 3, seed)
        ctx = _context(case)
        ctx.set_cm3(cost_matrix.three_d_of_two_dim_comb(ctx.cm))
        b = Batch3(ctx, "align_3d", *lens)
        cost, _, outlen = b.alloc_outputs()
        out = _zeros(b.out_bytes, 4 * (_room(case, b.n, 3) + 8 * b.n))
        s = {"case": case, "ctx": ctx, "batch": b,
             "args": (_dev(blob), *[_dev(o) for o in offs], cost, out, outlen)}
        torch.cuda.synchronize()
        return s
    if kind == "readjust":
        blob, offs, lens = _family(case, case["nodes"], 3, seed)
        return {"case": case, "ctx": _context(case), "room": 2 * _room(case, case["nodes"], 1),
                "nodes": [_host(blob, offs, lens, k) for k in range(case["nodes"])]}
    if kind == "union":
        n = case["merges"]
        blob, offs, lens = _family({**case, "iupac": 0.05}, n, 2, seed)
        ctx = Context(0)
        ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 1, 3))
        b = Batch(ctx, "align_affine", lens[0], lens[1])
        cost, out, outlen = b.alloc_outputs()
        b.run(_dev(blob), _dev(offs[0]), _dev(offs[1]), cost, out, outlen, sync=True)
        oh, lh = out.cpu().numpy(), outlen.cpu().numpy()
        merges = []
        for k in range(n):
            ri, rj, _, mwg = b.unpack(oh, lh, k)
            x, y = _host(blob, offs, lens, k)
            merges.append((ri, rj, mwg, unions.leaf(x), unions.leaf(y)))
        b.close()
        lv = unions.Level(ctx, merges)
        room = _room(case, n, 1)
        # the level's blobs, in buffers of one size for every seed
        for name, size in (("d_seq", 9 * room), ("d_int", 9 * room)):
            t = getattr(lv, name)
            setattr(lv, name, torch.nn.functional.pad(t, (0, max(0, size - t.numel()))))
        torch.cuda.synchronize()
        return {"case": case, "ctx": ctx, "level": lv}
    # rejoin: node and edge medians of a simulated tree, kept in the pool
    rng = np.random.default_rng(seed)
    ctx = Context(0)
    ctx.set_cm(cost_matrix.of_transformations_and_gaps(1, 2))
    sv = Server(ctx, n_slots=3, max_batch_pairs=2048, max_len=8192, slot_dm_bytes=1 << 30,
                pool_bytes=64 << 20)
    parent, children, leaves = spr.simulate(case["taxa"], case["root"], seed)
    mid = spr.downpass(sv, parent, children, leaves)
    emid = spr.edge_medians(sv, parent, mid)
    n = case["requests"]
    a, b, _, _ = spr.rejoin_requests(parent, children, mid, emid, n, rng)
    dw, _ = spr.rejoin_deltaw(sv, a, b)
    return {"case": case, "ctx": ctx, "server": sv, "a": a, "b": b, "dw": dw,
            "arrive": np.zeros(n), "ops": ["cost_2d"] * n}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pair":
        al, a, b, op = state["align"], state["a"], state["b"], case["op"]
        if op == "align_affine":
            m, ra, rb, cost, mwg = al.align_affine_3(a, b)
            return (cost, *[_padded(x, state["room"]) for x in (m, ra, rb, mwg)])
        if op == "align_2d":
            ra, rb, cost = al.align_2(a, b)
            return cost, _padded(ra, state["room"]), _padded(rb, state["room"])
        return al.cost_2(a, b)
    if kind in ("batch", "triples"):
        state["batch"].run(*state["args"], sync=True)
        if case.get("op") in ("cost_affine", "cost_2d"):
            return state["args"][-3]
        return state["args"][-3:]
    if kind == "readjust":
        res = readjust.readjust_level(state["ctx"], state["nodes"])
        return (np.array([r[0] for r in res]), np.array([r[1] for r in res]),
                _padded(np.concatenate([r[2] for r in res]), state["room"]),
                _padded(np.concatenate([r[3] for r in res]), state["room"]))
    if kind == "union":
        lv = state["level"]
        lv.run(sync=True)
        return lv.d_seq, lv.d_int, lv.d_len, lv.d_st
    return state["server"].replay(state["arrive"], state["ops"], state["a"], state["b"],
                                  deltaw=state["dw"])[0]


def work(case):
    """Bytes of the inputs and results, and the operations of the cells that
    no plan can skip: every cell of a full DP; of a banded one, the cells of
    a band that just holds the expected indels."""
    rng = np.random.default_rng(0)
    kind = case["kind"]
    if kind == "rejoin":
        n, ln = case["requests"], float(case["root"])
        # every clade and edge median read once, a band of 10% of the length
        return {"bytes": 4 * case["taxa"] * ln + 4 * n, "flops": n * 6 * ln * 0.1 * ln}
    n = case.get("pairs") or case.get("triples") or case.get("nodes") or case.get("merges") or 1
    ln = _root_lengths(case, n, rng).astype(np.float64) + 1
    if kind == "union":
        # aligned triple, two unions in, one out; a few operations a column
        return {"bytes": float(ln.sum()) * (3 + 2 * 5 + 2 * 13), "flops": float(ln.sum()) * 8}
    div = (case["dlo"] + case["dhi"]) / 2
    band = np.minimum(ln, 1 + 2 * 3 * div * (3.0 / 13.0) * ln)
    if kind == "triples":
        return {"bytes": float(ln.sum()) * 15, "flops": OPS["align_3d"] * float((ln ** 3).sum())}
    if kind == "readjust":
        ops = OPS["align_affine" if case["opening"] else "align_2d"]
        return {"bytes": float(ln.sum()) * 5, "flops": 10 * ops * float((ln * band).sum())}
    op = case["op"]
    cells = float((ln * ln).sum()) if op == "cost_affine" else float((ln * band).sum())
    out = 2 if op.startswith("cost") else 6
    return {"bytes": float(ln.sum()) * out + 4 * n, "flops": OPS[op] * cells}
