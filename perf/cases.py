"""Performance cases of the semi-local LCS engine.

Each case is one call, or one burst of calls, that a program built on
``lcs_amd`` makes through its public entry points: single pairs from host
strings and from device strings, batches, a merge of two permutations, score
queries, the LCS length alone and a burst of served requests.  Sizes are
those of the repository's own workloads (uniform4096, the mutated 2^20 pair,
the planted Zipf pair, 10,000 pairs in [256, 16384], requests in
[1024, 262144], the reference's run script) or ragged sizes in between.

Every output is whole numbers, so every case is compared exactly.
"""
import functools
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "platform-independent-lcs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import lcs_amd  # noqa: E402

DEV = "cuda:0"

# Largest extents that draw() takes (a drawn case costs less than the largest
# listed one, the 2^40 cells of the mutated pair).
MAX_HOST, MAX_DEVICE = 262144, 700000


def listed():
    return [
        # one short pair per call from host strings, as a script of small
        # comparisons makes them: launches, copies and waits are what counts
        {"name": "comb_short", "kind": "comb", "m": 300, "n": 500, "alphabet": 4},
        # uniform4096: the reference's own CPU-sized pair, its whole timed
        # call (host strings in, both permutation rows out)
        {"name": "permutation_4096", "kind": "permutation", "m": 4096, "n": 4096, "alphabet": 4, "rate": 1.0},
        # a served-size pair of protein-like strings, ragged, one call
        {"name": "comb_protein", "kind": "comb", "m": 50021, "n": 70207, "alphabet": 20},
        # word tokens (symbols above 255, the 32-bit symbol path), ragged
        {"name": "comb_tokens", "kind": "comb", "m": 9771, "n": 11302, "alphabet": 40000},
        # the largest size of the reference's sweep, binary strings, resident
        {"name": "device_200000", "kind": "device", "m": 200000, "n": 200000, "alphabet": 2, "rate": 1.0},
        # the headline pair
        {"name": "device_2^20", "kind": "device", "m": 1 << 20, "n": 1 << 20, "alphabet": 4},
        # a short query in a long text with planted copies, skewed alphabet
        {"name": "device_zipf", "kind": "zipf", "m": 1 << 14, "n": 1 << 22, "alphabet": 26, "copies": 64},
        # the batched workload: 10,000 uneven pairs, resident
        {"name": "batch_10000", "kind": "batch", "pairs": 10000, "lo": 256, "hi": 16384, "alphabet": 4, "sizes": 7},
        # merging the permutations of two halves of a text (host permutations)
        {"name": "braid_65000", "kind": "braid", "m": 65000, "n1": 40000, "n2": 50001, "alphabet": 4, "rows": False},
        # substring scores of the 2^19-strand permutation: index and 2^20 queries
        {"name": "queries_2^19", "kind": "queries", "m": 1 << 18, "n": 1 << 18, "alphabet": 4, "queries": 1 << 20},
        # the LCS length alone of the headline pair
        {"name": "length_2^20", "kind": "length", "m": 1 << 20, "n": 1 << 20, "alphabet": 4},
        # a burst of served requests, lengths log-uniform in [1024, 262144],
        # alphabets 4 and 20
        {"name": "served_24", "kind": "served", "requests": 24, "lo": 1024, "hi": 262144, "sizes": 11},
    ]


def _log_int(rng, lo, hi):
    return min(max(int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))), lo), hi)


def draw(rng):
    kind = rng.choice(["comb", "comb", "permutation", "device", "device", "zipf", "batch", "braid", "queries",
                       "length", "served"])
    alphabet = rng.choice([2, 4, 4, 20, 26, 40000])
    rate = rng.choice([1.0, round(rng.uniform(0.05, 0.3), 3)])
    if kind in ("comb", "permutation"):
        return {"kind": kind, "m": _log_int(rng, 64, MAX_HOST), "n": _log_int(rng, 64, MAX_HOST),
                "alphabet": alphabet, "rate": rate}
    if kind == "device":
        m = _log_int(rng, 1024, MAX_DEVICE)
        return {"kind": kind, "m": m, "n": min(MAX_DEVICE, max(64, int(m * math.exp(rng.uniform(-0.7, 0.7))))),
                "alphabet": alphabet, "rate": rate}
    if kind == "zipf":
        return {"kind": kind, "m": _log_int(rng, 512, 1 << 15), "n": _log_int(rng, 1 << 18, 1 << 22),
                "alphabet": rng.choice([4, 20, 26]), "copies": rng.randint(1, 64)}
    if kind == "batch":
        lo = _log_int(rng, 16, 1024)
        return {"kind": kind, "pairs": _log_int(rng, 16, 8000), "lo": lo, "hi": lo * rng.choice([2, 8, 16]),
                "alphabet": rng.choice([2, 4, 20, 26]), "sizes": rng.randrange(1 << 20)}
    if kind == "braid":
        return {"kind": kind, "m": _log_int(rng, 100, 1 << 18), "n1": _log_int(rng, 100, 1 << 17),
                "n2": _log_int(rng, 100, 1 << 17), "alphabet": rng.choice([2, 4, 20]), "rows": rng.random() < 0.5}
    if kind == "queries":
        return {"kind": kind, "m": _log_int(rng, 500, 1 << 18), "n": _log_int(rng, 500, 1 << 18),
                "alphabet": rng.choice([4, 20]), "queries": _log_int(rng, 64, 1 << 20)}
    if kind == "length":
        m = _log_int(rng, 300, 1 << 19)
        return {"kind": kind, "m": m, "n": min(1 << 19, max(64, int(m * math.exp(rng.uniform(-1.5, 1.5))))),
                "alphabet": rng.choice([2, 4, 20, 26, 100])}
    lo = _log_int(rng, 256, 4096)
    return {"kind": "served", "requests": rng.randint(4, 24), "lo": lo, "hi": lo * rng.choice([4, 16, 64]),
            "sizes": rng.randrange(1 << 20)}


@functools.lru_cache(maxsize=None)
def _context():
    return lcs_amd.Context(0)


@functools.lru_cache(maxsize=None)
def _server():
    return lcs_amd.Server(_context(), hbm_budget=16 << 30, max_inflight=4)


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(g, length, alphabet):
    return torch.randint(0, alphabet, (length,), generator=g, device=DEV, dtype=torch.int32)


def _zipf(g, length, alphabet, s=1.1):
    weights = torch.arange(1, alphabet + 1, device=DEV, dtype=torch.float64) ** -s
    edges = torch.cumsum(weights / weights.sum(), 0)[:-1].contiguous()
    u = torch.rand(length, generator=g, device=DEV, dtype=torch.float64)
    return torch.searchsorted(edges, u, right=True).to(torch.int32)


def _mutated(g, a, starts, lengths, out_starts, out_lengths, alphabet, sub, indel):
    """Concatenated strings derived from the concatenated sources: every
    output symbol copies the next source symbol (cyclically), skips one
    (deletion), or is a random insertion, and is substituted at rate `sub`."""
    total = int(out_lengths.sum())
    pair = torch.repeat_interleave(torch.arange(len(out_lengths), device=DEV), out_lengths)
    u = torch.rand(total, generator=g, device=DEV)
    step = 1 + (u < indel[pair] / 2).to(torch.int64) - (u > 1 - indel[pair] / 2).to(torch.int64)
    walk = torch.cumsum(step, 0) - step
    walk = walk - walk[out_starts][pair]
    b = a[starts[pair] + walk % lengths[pair]]
    other = torch.randint(1, max(alphabet, 2), (total,), generator=g, device=DEV, dtype=torch.int32)
    changed = (torch.rand(total, generator=g, device=DEV) < sub[pair]) | (step == 0)
    return torch.where(changed, (b + other) % alphabet, b).to(torch.int32)


def _pair(g, m, n, alphabet, rate):
    """a uniform, b = a with substitutions and indels (rate 1: independent)."""
    a = _uniform(g, m, alphabet)
    if rate >= 1.0:
        return a, _uniform(g, n, alphabet)
    one = lambda x, dtype=torch.int64: torch.tensor([x], device=DEV, dtype=dtype)  # noqa: E731
    b = _mutated(g, a, one(0), one(m), one(0), one(n), alphabet, one(rate * 5 / 6, torch.float32),
                 one(rate / 6, torch.float32))
    return a, b


def _lengths(case, count):
    r = random.Random(case["sizes"])
    return [(_log_int(r, case["lo"], case["hi"]), _log_int(r, case["lo"], case["hi"])) for _ in range(count)]


def _empty(n):
    return torch.empty(n, device=DEV, dtype=torch.int32)


def _starts(lengths):
    return torch.cumsum(lengths, 0) - lengths


def prepare(case, seed):
    kind, g, ctx = case["kind"], _generator(seed), _context()
    state = dict(case)
    if kind in ("comb", "permutation"):
        a, b = _pair(g, case["m"], case["n"], case["alphabet"], case.get("rate", 0.12))
        state.update(a=a.cpu().numpy(), b=b.cpu().numpy())
    elif kind == "device":
        a, b = _pair(g, case["m"], case["n"], case["alphabet"], case.get("rate", 0.12))
        state.update(a=a, b=b, h=_empty(case["m"]), v=_empty(case["n"]))
    elif kind == "zipf":
        m, n = case["m"], case["n"]
        a, b = _zipf(g, m, case["alphabet"]), _zipf(g, n, case["alphabet"])
        at = torch.randint(0, max(n - m, 1), (case["copies"],), generator=g, device=DEV).tolist()
        for o in at:
            part = b[o:o + m]
            keep = torch.rand(len(part), generator=g, device=DEV) >= 0.05
            b[o:o + m] = torch.where(keep, a[:len(part)], part)
        state.update(a=a, b=b, h=_empty(m), v=_empty(n))
    elif kind == "batch":
        m, n = (np.array(x, np.int32) for x in zip(*_lengths(case, case["pairs"])))
        dm, dn = (torch.from_numpy(x).to(DEV).to(torch.int64) for x in (m, n))
        a = _uniform(g, int(m.sum()), case["alphabet"])
        rate = 0.05 + 0.15 * torch.rand(len(m), generator=g, device=DEV)
        b = _mutated(g, a, _starts(dm), dm, _starts(dn), dn, case["alphabet"], 0.8 * rate, 0.2 * rate)
        split = lambda x, sizes: np.split(x.cpu().numpy(), np.cumsum(sizes)[:-1])  # noqa: E731
        state.update(layout=lcs_amd.BatchLayout(split(a, m), split(b, n)), a=a, b=b, h=_empty(len(a)),
                     v=_empty(len(b)))
    elif kind == "braid":
        m, n1, n2 = case["m"], case["n1"], case["n2"]
        a, b = (x.cpu().numpy() for x in _pair(g, m, n1 + n2, case["alphabet"], 0.12))
        if case["rows"]:   # the two parts are cut from the rows: glued on the n columns
            parts = [ctx.comb_permutation(x, a)[0] for x in (b[:n1], b[n1:])]
        else:
            parts = [ctx.comb_permutation(a, x)[0] for x in (b[:n1], b[n1:])]
        state.update(p=parts[0], q=parts[1])
    elif kind == "queries":
        m, n = case["m"], case["n"]
        a, b = (x.cpu().numpy() for x in _pair(g, m, n, case["alphabet"], 0.12))
        perm = torch.from_numpy(ctx.comb_permutation(a, b)[0]).to(DEV)
        ends = torch.randint(0, n + 1, (2, case["queries"]), generator=g, device=DEV, dtype=torch.int32)
        q = torch.sort(ends, 0)[0]
        state.update(perm=perm, q0=q[0].contiguous(), q1=q[1].contiguous(), out=_empty(case["queries"]))
    elif kind == "length":
        a, b = _pair(g, case["m"], case["n"], case["alphabet"], 0.12)
        state.update(a=a, b=b, out=_empty(1))
    else:
        _server()
        r = random.Random(case["sizes"] + 1)
        pairs = []
        for m, n in _lengths(case, case["requests"]):
            alphabet = r.choice([4, 20])
            pairs.append([x.cpu().numpy() for x in _pair(g, m, n, alphabet, r.uniform(0.05, 0.2))])
        state.update(pairs=pairs)
    torch.cuda.synchronize()   # the engine runs on streams of its own
    return state


def run(state):
    kind, ctx = state["kind"], _context()
    if kind == "comb":
        return ctx.comb(state["a"], state["b"])
    if kind == "permutation":
        return ctx.comb_permutation(state["a"], state["b"])
    if kind in ("device", "zipf"):
        a, b, h, v = state["a"], state["b"], state["h"], state["v"]
        rc = lcs_amd.lib().lcs_comb_device(ctx.handle, a.data_ptr(), a.numel(), b.data_ptr(), b.numel(), None,
                                           h.data_ptr(), v.data_ptr(), None)
        if rc:
            raise lcs_amd.LcsError("lcs_comb_device", rc)
        return h, v
    if kind == "batch":
        lcs_amd.batch_comb_device(ctx, state["layout"], *(state[x].data_ptr() for x in "abhv"))
        return state["h"], state["v"]
    if kind == "braid":
        k = state["m"]
        return ctx.braid_multiply(state["p"], state["q"], k, state["rows"])
    if kind == "queries":
        index = lcs_amd.DominanceIndex(ctx, size=state["perm"].numel(), device_ptr=state["perm"].data_ptr())
        index.query_device(state["m"], state["n"], lcs_amd.SEMI_STRING_SUBSTRING, state["q0"].data_ptr(),
                           state["q1"].data_ptr(), state["q0"].numel(), state["out"].data_ptr())
        index.close()
        return state["out"]
    if kind == "length":
        ctx.llcs_device(state["a"].data_ptr(), state["m"], state["b"].data_ptr(), state["n"], state["alphabet"],
                        state["out"].data_ptr())
        return state["out"]
    server = _server()
    ids = [server.submit(a, b) for a, b in state["pairs"]]
    out = [server.wait(i) for i in ids]
    for i in ids:
        server.release(i)
    return out


def work(case):
    """Symbols in and strands out once, and four 32-bit operations a cell
    (the length alone: four per 32 cells)."""
    kind = case["kind"]
    if kind == "batch":
        pairs = _lengths(case, case["pairs"])
    elif kind == "served":
        pairs = _lengths(case, case["requests"])
    elif kind == "braid":
        size = case["m"] * 3 + 2 * (case["n1"] + case["n2"])   # p, q and their product
        return {"bytes": 4 * size, "flops": case["m"] * math.log2(max(case["m"], 2))}
    elif kind == "queries":
        size = case["m"] + case["n"]
        return {"bytes": 4 * size + 12 * case["queries"], "flops": (size + 2 * case["queries"]) * math.log2(size)}
    else:
        pairs = [(case["m"], case["n"])]
    cells, symbols = sum(m * n for m, n in pairs), sum(m + n for m, n in pairs)
    if kind == "length":
        return {"bytes": 4 * symbols, "flops": cells / 8}
    return {"bytes": (12 if kind == "permutation" else 8) * symbols, "flops": 4 * cells}


def tolerance(case):
    return "exact"


def _comb_exact(a, b):
    """The strands of a against b by anti-diagonals (64-bit integers)."""
    m, n = len(a), len(b)
    rows = a[::-1].astype(np.int64)   # row i holds a[m-1-i]; v strands run from high i to low i
    h, v = np.arange(m, dtype=np.int64), np.arange(m, m + n, dtype=np.int64)
    cols = b.astype(np.int64)
    for d in range(m + n - 1):        # cells (m-1-r, j) with r + j = d
        j0, j1 = max(0, d - m + 1), min(n, d + 1)
        i0 = m - 1 - d + j0
        hs, vs = h[i0:i0 + j1 - j0].copy(), v[j0:j1].copy()
        swap = (rows[i0:i0 + j1 - j0] == cols[j0:j1]) | (hs > vs)
        h[i0:i0 + j1 - j0] = np.where(swap, vs, hs)
        v[j0:j1] = np.where(swap, hs, vs)
    return h, v


def exact(case, seed):
    """Small pairs by a plain restatement of the comb, lengths by the
    word-parallel recurrence on Python integers; None where that is slow."""
    kind = case["kind"]
    if kind in ("comb", "permutation", "device") and case["m"] * case["n"] <= 1 << 28:
        s = prepare(case, seed)
        a, b = (np.asarray(x.cpu() if torch.is_tensor(x) else x) for x in (s["a"], s["b"]))
        h, v = _comb_exact(a, b)
        score = int((v < len(a)).sum())
        if kind == "device":
            return h, v
        if kind == "comb":
            return h, v, score
        c2r = np.concatenate([v, h])
        r2c = np.empty_like(c2r)
        r2c[c2r] = np.arange(len(c2r))
        return r2c, c2r, score
    if kind == "length" and case["m"] * case["n"] <= 1 << 32:
        s = prepare(case, seed)
        a, b = s["a"].cpu().tolist(), s["b"].cpu().tolist()
        masks, full = {}, (1 << len(a)) - 1
        for c in set(a):
            bits = (np.array(a) == c).astype(np.uint8)
            masks[c] = int.from_bytes(np.packbits(bits, bitorder="little").tobytes(), "little")
        row = full
        for c in b:
            u = row & masks.get(c, 0)
            row = ((row + u) | (row - u)) & full
        return np.array([len(a) - bin(row).count("1")])
    return None
