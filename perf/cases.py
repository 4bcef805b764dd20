"""The work this framework is used for, as cases that a timing program can prepare and run.

    listed()            the cases, dicts of plain values
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and handles as a calling program holds them
    run(state)          one pass through the public entry points, and its outputs
    work(case)          bytes and operations of a pass that the path cannot do without
    exact(case, seed)   None throughout: every output is a whole number (level counts, gate indices, distances,
                        rotations, letters), decided exactly by the search, so there is nothing to round

Kinds of case:
    proof    a gate-count search of a Toffoli-like target at a budget below its optimum: an exhaustive proof that no
             circuit of that many gates exists, on a context kept between searches
    oneshot  the same search as the command line runs it (context opened and closed inside the pass), with its
             options: the distance table of the last K gates, the meet-in-the-middle join, no symmetry classes
    search   seeded random Clifford+T circuits re-synthesised at budget = their length, one context each
    batch    several such searches of one gate set advancing in the same launches
    tcount   a T-count table built and one target searched with it (the command line's whole call)
    tcbatch  a batch of T-count targets searched together with a table that is kept
    cliffopt the Clifford table built and one circuit's Clifford segments and T placements optimised
    query    distances of many Clifford words already on the device, with a table that is kept
    serve    a burst of mixed requests answered by the request server
"""
import ctypes
import re

import numpy as np
import torch

import cheese_amd
from cheese_amd import clifford, serve, tcount
from cheese_amd import workloads as W

# the textbook Toffoli circuit on controls a, b and target c (15 gates, 7 T): budgets of 14 and below are proofs
_TOFFOLI = (("h", "c"), ("cx", "bc"), ("tdg", "c"), ("cx", "ac"), ("t", "c"), ("cx", "bc"), ("t", "b"), ("tdg", "c"),
            ("cx", "ac"), ("cx", "ab"), ("t", "a"), ("tdg", "b"), ("cx", "ab"), ("t", "c"), ("h", "c"))
# gates a seed may leave on a control beside the Toffoli: they commute with it and lower its gate count nowhere
_PHASES = ((), ("sdg",), ("s",), ("z",))


def listed():
    return [
        # re-synthesis of 2-qubit circuits, as a peephole pass calls it: short searches, launches and set-up count
        {"name": "search2-l12", "kind": "search", "n": 2, "length": 12, "count": 8},
        # re-synthesis of 3-qubit circuits of a compiler's block size, one process-like call each
        {"name": "search3-l12", "kind": "search", "n": 3, "length": 12, "count": 8},
        # the smallest proof that is quoted: latency of a handful of levels
        {"name": "proof-d9", "kind": "proof", "depth": 9},
        # the headline proof: budget 12
        {"name": "proof-d12", "kind": "proof", "depth": 12},
        # the largest proof: every circuit of up to 14 gates excluded, which makes 15 the optimum
        {"name": "proof-d14", "kind": "proof", "depth": 14},
        # the proof with a distance table of the last 6 gates, table built in the call
        {"name": "table6-d13", "kind": "oneshot", "depth": 13, "table": 6, "mitm": False, "sym": True},
        # a mapper's worth of 3-qubit blocks in one batch
        {"name": "batch3-c24", "kind": "batch", "n": 3, "count": 24, "lmin": 4, "lmax": 10},
        # a T-count question asked once: 3-qubit table of depth 4 and one search
        {"name": "tcount3-k4", "kind": "tcount", "n": 3, "K": 4},
        # T-counts of a whole circuit library against one table
        {"name": "tcbatch3-c96", "kind": "tcbatch", "n": 3, "K": 4, "count": 96},
        # the Clifford part of a 3-qubit circuit: whole group tabulated, then the beam search over T placements
        {"name": "cliffopt3-t6", "kind": "cliffopt", "n": 3, "t": 6, "beam": 16},
        # a pass over many Clifford words
        {"name": "query-1e5", "kind": "query", "n": 3, "count": 100000},
        # a burst at the server: half gate counts, a third T-counts, the rest Clifford words
        {"name": "serve-c48", "kind": "serve", "count": 48, "lmax": 10},
    ]


def draw(rng):
    def between(lo, hi):    # log-uniform whole number
        return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))
    kind = rng.choice(("proof", "oneshot", "search", "batch", "tcount", "tcbatch", "cliffopt", "query", "serve"))
    if kind == "proof":
        return {"kind": kind, "depth": rng.randint(6, 13)}
    if kind == "oneshot":
        how = rng.choice(("table", "mitm", "nosym"))
        if how == "table":
            return {"kind": kind, "depth": rng.randint(8, 13), "table": rng.randint(2, 7), "mitm": False, "sym": True}
        return {"kind": kind, "depth": rng.randint(6, 11 if how == "mitm" else 10), "table": 0, "mitm": how == "mitm",
                "sym": False}
    if kind == "search":
        return {"kind": kind, "n": rng.randint(2, 3), "length": rng.randint(3, 12), "count": rng.randint(1, 8)}
    if kind == "batch":
        return {"kind": kind, "n": rng.randint(2, 3), "count": between(2, 32), "lmin": rng.randint(2, 5),
                "lmax": rng.randint(6, 10)}
    if kind == "tcount":
        n = rng.randint(2, 3)
        return {"kind": kind, "n": n, "K": rng.randint(2, 4 if n == 3 else 6)}
    if kind == "tcbatch":
        n = rng.randint(2, 3)
        return {"kind": kind, "n": n, "K": rng.randint(3, 4), "count": between(1, 128)}
    if kind == "cliffopt":
        return {"kind": kind, "n": rng.randint(2, 3), "t": rng.randint(1, 10), "beam": between(1, 64)}
    if kind == "query":
        return {"kind": kind, "n": rng.randint(2, 3), "count": between(1, 1 << 20)}
    return {"kind": kind, "count": between(4, 64), "lmax": rng.randint(6, 10)}


# ---- inputs ----

def _seeds(seed, tag):
    return W.SplitMix64((seed * 0x9E3779B97F4A7C15 + tag * 0xD1B54A32D192ED03 + 1) & W.MASK64)


def _toffoli_like(seed):
    """a Toffoli on a seeded placement of its controls and target, with a seeded phase gate on each control"""
    r = _seeds(seed, 1)
    free = [0, 1, 2]
    at = {x: free.pop(r.below(len(free))) for x in "abc"}
    circ = [(g, tuple(at[x] for x in qs)) for g, qs in _TOFFOLI]
    for x in "ab":
        circ += [(g, (at[x],)) for g in _PHASES[r.below(4)]]
    return circ


def _gate_spec(n, circ, depth):
    return W.spec_from_skeleton(W.skeleton(n), W.unitary(n, circ), depth)


def _random_specs(seed, n, count, lmin, lmax):
    r = _seeds(seed, 2)
    return [W.random_spec(r.next() >> 1, n, lmin, lmax)[1] for _ in range(count)]


def _tcount_targets(seed, n, count, kmin=3, kmax=7):
    r = _seeds(seed, 3)
    out = []
    for _ in range(count):
        _, circ = tcount.random_target(r.next() >> 1, n, kmin, kmax, lambda q: tcount.random_clifford_word(q, n))
        out.append(tcount.tspec_text(n, W.unitary(n, circ)))
    return out


def _requests(seed, count, lmax):
    """the mixed stream of the server: gate counts of 2 and 3 qubits, T-counts, Clifford words"""
    r = _seeds(seed, 4)
    out = []
    for _ in range(count):
        x = r.below(100)
        if x < 50:
            n = 2 + r.below(2)
            out.append({"kind": serve.GATES, "text": W.random_spec(r.next() >> 1, n, 4, lmax)[1], "budget": -1})
        elif x < 85:
            out.append({"kind": serve.TCOUNT, "text": _tcount_targets(r.next() >> 1, 3, 1, 2, 7)[0], "budget": 16})
        else:
            out.append({"kind": serve.CLIFFORD, "word": [r.below(21) for _ in range(5 + r.below(36))]})
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "proof":
        return {"kind": kind, "searcher": cheese_amd.Searcher(_gate_spec(3, _toffoli_like(seed), case["depth"]))}
    if kind == "oneshot":
        return {"kind": kind, "spec": _gate_spec(3, _toffoli_like(seed), case["depth"]),
                "options": {"table": case["table"], "mitm": case["mitm"], "sym": case["sym"]}}
    if kind == "search":
        return {"kind": kind, "specs": _random_specs(seed, case["n"], case["count"], case["length"], case["length"])}
    if kind == "batch":
        return {"kind": kind, "specs": _random_specs(seed, case["n"], case["count"], case["lmin"], case["lmax"])}
    if kind == "tcount":
        return {"kind": kind, "K": case["K"], "target": _tcount_targets(seed, case["n"], 1)[0]}
    if kind == "tcbatch":
        targets = _tcount_targets(seed, case["n"], case["count"])
        return {"kind": kind, "targets": targets, "table": tcount.CosetTable(targets[0], K=case["K"])}
    if kind == "cliffopt":
        job, _ = clifford.random_job(_seeds(seed, 5).next(), case["n"], case["t"])
        return {"kind": kind, "n": case["n"], "job": job, "beam": case["beam"]}
    if kind == "query":
        table = clifford.CliffordTable(case["n"])
        g = np.random.default_rng(seed)
        lens = g.integers(5, 41, case["count"])
        offs = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
        letters = g.integers(0, table.ng, int(offs[-1])).astype(np.uint8)
        state = {"kind": kind, "table": table, "count": case["count"], "letters": torch.from_numpy(letters).cuda(),
                 "offs": torch.from_numpy(offs).cuda(),
                 "dist": torch.empty(case["count"], dtype=torch.int32, device="cuda")}
        torch.cuda.synchronize()    # the table's own stream reads these
        return state
    requests = _requests(seed, case["count"], case["lmax"])
    server = serve.Server(_gate_spec(2, [], 1), _gate_spec(3, [], 1), _tcount_targets(seed, 3, 1)[0])
    return {"kind": kind, "server": server, "requests": requests}


# ---- passes ----
# A search's outputs have the lengths that its answer happens to have; they are laid out here in arrays as long as the
# longest answer (the framework's own limits), with -1 behind the end.

_LEVEL = ("dir", "t", "parents", "prefixes", "cut_w3", "cut_lb", "survivors", "distinct", "proved_unsat")
_TC_LEVEL = ("t", "parents", "children", "cosets", "new")
_MAX_LEVELS, _MAX_OPT = 2 * cheese_amd.DMAX + 1, 1024


def _padded(values, n):
    a = np.full(n, -1, dtype=np.int64)
    v = np.array(list(values), dtype=np.int64)
    a[:len(v)] = v
    return a


def _rows(levels, fields, n=_MAX_LEVELS):
    a = np.full((n, len(fields)), -1, dtype=np.int64)
    for i, lv in enumerate(levels):
        a[i] = [lv[f] for f in fields]
    return a


def _stacked(outs):
    return {k: np.stack([o[k] for o in outs]) for k in outs[0]}


def _search_out(o):
    circuit = o.get("circuit_idx")
    split = o.get("split")
    return {"result": _padded([o["rc"], o.get("found", 0), len(o["levels"])], 3), "levels": _rows(o["levels"], _LEVEL),
            "circuit": _padded(circuit if circuit is not None else (), cheese_amd.DMAX),
            "split": _padded(split[1] if split else (), 2)}


def _tc_out(r):
    return {"result": _padded([r["rc"], r["tcount"]] + r["split"], 4),
            "rotations": _padded((x for pair in r["rotations"] for x in pair), 2 * tcount.TMAX),
            "levels": _rows(r["levels"], _TC_LEVEL, tcount.TMAX + 1)}


_OPT_GATES = ("h", "s", "sdg", "x", "z", "y", "cx", "t", "tdg")


def _opt_out(text):
    """the optimiser's counts and gate list as numbers (its summary line without the seconds)"""
    head, *gates = text.strip().splitlines()
    counts = [int(re.search(f'"{k}": ([0-9]+)', head).group(1))
              for k in ("clifford_gates", "clifford_gates_before", "t_gates")]
    flat = []
    for ln in gates:
        g, *qs = ln.split()
        flat += [_OPT_GATES.index(g)] + [int(q) for q in qs]
    return {"counts": _padded(counts, 3), "circuit": _padded(flat, _MAX_OPT)}


def run(state):
    kind = state["kind"]
    if kind == "proof":
        return _search_out(state["searcher"].run())
    if kind == "oneshot":
        return _search_out(cheese_amd.search(state["spec"], **state["options"]))
    if kind == "search":
        return _stacked([_search_out(cheese_amd.search(s)) for s in state["specs"]])
    if kind == "batch":
        return _stacked([_search_out(o) for o in cheese_amd.search_many(state["specs"])])
    if kind == "tcount":
        table = tcount.CosetTable(state["target"], K=state["K"])
        try:
            return {"table": _rows(table.levels, _TC_LEVEL, tcount.TMAX + 1), "size": table.size,
                    "result": _tc_out(table.search([state["target"]])[0])}
        finally:
            table.close()
    if kind == "tcbatch":
        return _stacked([_tc_out(r) for r in state["table"].search(state["targets"])])
    if kind == "cliffopt":
        table = clifford.CliffordTable(state["n"])
        try:
            return {"levels": _padded(table.levels(), 128), "result": _opt_out(table.optimize(state["job"], state["beam"]))}
        finally:
            table.close()
    if kind == "query":
        p = ctypes.c_void_p
        rc = cheese_amd.lib().chz_cliff_query_words_noalloc(
            state["table"].h, p(state["letters"].data_ptr()), p(state["offs"].data_ptr()),
            ctypes.c_longlong(state["count"]), p(state["dist"].data_ptr()), None)
        if rc:
            raise RuntimeError(f"chz_cliff_query_words_noalloc exit {rc}")
        return state["dist"]
    answers, _ = serve.replay(state["server"], state["requests"], [0.0] * len(state["requests"]))
    return _stacked([{"result": _padded([a["rc"], a["len"], a["found"]] + a["split"], 5),
                      "out": _padded(a["out"], 2 * serve.DMAX)} for _, a in sorted(answers.items())])


# ---- what a pass cannot do without ----

def _search_work(n, depth, classes=1.0):
    """a proof's or search's children and kept nodes by budget.  The bounds leave about 4.6 times as many prefixes per
    gate of budget at 3 qubits (Toffoli: 36 thousand at 9, 7.0 million at 12, 150 million at 14) and 2.5 at 2; one in
    ten is kept.  A child costs its residual's coefficients (an addition or move each); a kept node is written and
    read once."""
    coeffs = 4 << (2 * n)
    children = (0.075 * 4.6 ** depth if n == 3 else 40.0 * 1.8 ** depth) * classes
    return {"bytes": int(children * (2 * 0.1 * coeffs * 4)) + 20000, "flops": int(children * coeffs)}


def _scaled(w, by):
    return {k: int(v * by) for k, v in w.items()}


def _tcount_work(n, depth, targets=1):
    """cosets reached by `depth` rotations: each one's channel representation (4^n x 4^n residues) formed once with a
    rotation (a quarter of its entries change) and its key and place stored"""
    p2 = 1 << (4 * n)
    rots = (1 << (2 * n)) - 1
    cosets = 1.0
    for t in range(1, depth + 1):
        cosets *= rots * (1.0 if t == 1 else 0.75)
    return {"bytes": int(targets * cosets * 16) + 20000, "flops": int(targets * cosets * p2 / 2)}


_CLIFFORD = {1: 24, 2: 11520, 3: 92897280}


def _clifford_work(n):
    """every element reached from every other by every gate: a tableau update and one look-up each"""
    gates = 5 * n + n * (n - 1)
    return {"bytes": _CLIFFORD[n] * 16, "flops": _CLIFFORD[n] * gates * 8}


def work(case):
    kind = case["kind"]
    if kind == "proof":
        return _search_work(3, case["depth"])
    if kind == "oneshot":
        depth = case["depth"] - (case["table"] or (case["depth"] // 2 if case["mitm"] else 0))
        w = _search_work(3, max(depth, (case["depth"] + 1) // 2), 1.0 if case["sym"] else 4.0)
        if case["table"]:   # 1.7 * 7.6^K classes (K = 4: 5.4 thousand, K = 7: 2.7 million), 27 children and a key each
            classes = 1.7 * 7.6 ** case["table"]
            w = {"bytes": w["bytes"] + int(classes * 2 * 1024), "flops": w["flops"] + int(classes * 27 * 256)}
        return w
    if kind == "search":
        return _scaled(_search_work(case["n"], case["length"] - 2), case["count"])
    if kind == "batch":
        return _scaled(_search_work(case["n"], (case["lmin"] + case["lmax"]) / 2), case["count"])
    if kind == "tcount":
        return _tcount_work(case["n"], case["K"])
    if kind == "tcbatch":
        return _tcount_work(case["n"], 2, case["count"])
    if kind == "cliffopt":
        return _clifford_work(case["n"])
    if kind == "query":
        return {"bytes": int(case["count"] * (22.5 + 8 + 8 + 4)), "flops": int(case["count"] * 22.5 * 8)}
    per = _search_work(3, case["lmax"] - 2)
    return _scaled(per, case["count"] / 4)


def exact(case, seed):
    return None
