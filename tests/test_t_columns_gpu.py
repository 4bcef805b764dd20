"""T columns (formed for 3-qubit frontiers of 32,768 nodes and more while a search has six gates left) carried through a
batch: searches that wait for memory, levels of captured steps after large ones, and roots that join beside them leave every
search the levels and the circuit it gets alone."""
import re

import pytest

import cheese_amd
from cheese_amd import workloads as W

from conftest import read_spec

pytestmark = pytest.mark.gpu


def _strip(o):
    return (o["rc"], o.get("circuit_idx"), [{f: v for f, v in lv.items() if f != "seconds"} for lv in o["levels"]])


def _toffoli(depth):
    return re.sub(r"^depth \d+", f"depth {depth}", read_spec("toffoli-d9"), count=1, flags=re.M)


@pytest.fixture(scope="module")
def searches():
    """(spec, depth, its result alone): proofs and random circuits, large frontiers among them"""
    specs = [_toffoli(d) for d in (12, 13, 4)] + [W.random_spec(seed, 3, 4, 13)[1] for seed in range(700, 712)]
    out = [(s, int(re.search(r"^depth (\d+)", s, re.M).group(1)), cheese_amd.search(s)) for s in specs]
    assert sum(any(lv["distinct"] >= 32768 and d - lv["t"] >= 6 for lv in o["levels"]) for _, d, o in out) >= 2
    return out


@pytest.mark.parametrize("budget", [0, 1e8, 6e8])
def test_columns_of_searches_that_wait(searches, budget):
    st = {}
    outs = cheese_amd.search_many([s for s, _, _ in searches], budget=budget, stats=st)
    assert (st["waits"] > 0) == (budget > 0)
    assert st["kernel_stats"]["level_graph"]["launches"] > 0
    for (_, _, alone), o in zip(searches, outs):
        assert _strip(alone) == _strip(o)


def test_columns_beside_joining_roots(searches):
    b = cheese_amd.Batch(searches[0][0])
    outs = [{"levels": []} for _ in searches]
    try:
        assert b.add(searches[0][0], 0) == 0 and b.add(searches[1][0], 1) == 0
        nxt, beside = 2, 0
        while True:
            for tag, kind, d in b.events():
                if kind == "level":
                    outs[tag]["levels"].append(d)
                else:
                    outs[tag].update(d)
            if nxt < len(searches) and b.nodes >= 32768:
                assert b.add(searches[nxt][0], nxt) == 0
                nxt, beside = nxt + 1, beside + 1
            elif not b.live:
                if nxt == len(searches):
                    break
                assert b.add(searches[nxt][0], nxt) == 0
                nxt += 1
            assert b.step() == 0
    finally:
        b.close()
    assert beside >= 3
    for (_, _, alone), o in zip(searches, outs):
        assert _strip(alone) == _strip(o)
