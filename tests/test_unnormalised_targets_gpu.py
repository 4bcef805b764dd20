"""Targets written with a common factor of sqrt2 over a higher exponent: parse_spec keeps them as they stand, and every
search of one has the level lines and the circuit of the normalised target.  Bounds taken from a parent alone hold only
for a normalised parent, and they are used where a parent's candidates are split little: gate sets of up to four
candidates, and frontiers of some thousand roots."""
import pytest

import cheese_amd
from cheese_amd import specgen
from cheese_amd import workloads as W

pytestmark = pytest.mark.gpu

SQRT2 = (0, 1, 0, -1)


def _scaled(U, j):
    """U = (k, rows) as sqrt2^j times its entries over sqrt2^(k + j)"""
    k, rows = U
    for _ in range(j):
        rows = [[W._zmul(SQRT2, z) for z in row] for row in rows]
    return k + j, rows


def _strip(o):
    return (o["rc"], o.get("circuit_idx"), o.get("found"),
            [{f: v for f, v in lv.items() if f != "seconds"} for lv in o["levels"]])


@pytest.mark.parametrize("n,gates,circ", [
    (1, ("h", "t"), [("t", (0,))]),
    (1, ("h", "t"), [("h", (0,)), ("t", (0,)), ("h", (0,))]),
    (2, ("h", "cx"), [("cx", (0, 1))]),
    (2, ("h", "cx"), [("h", (1,)), ("cx", (1, 0)), ("h", (0,))]),
    (3, ("t",), [("t", (1,))]),
    (3, ("h",), [("h", (2,)), ("h", (0,))]),
], ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else str(v) if isinstance(v, int) else str(len(v)))
@pytest.mark.parametrize("j", [1, 2, 3, 6])
def test_few_candidates(n, gates, circ, j):
    U = W.unitary(n, circ)
    spec = specgen.spec_text(n, circ, len(circ), gates=gates)
    plain = cheese_amd.search(spec)
    assert plain["rc"] == 0 and plain["verified"] and len(plain["circuit"]) == len(circ)
    assert _strip(cheese_amd.search(W.spec_from_skeleton(spec, _scaled(U, j), len(circ)))) == _strip(plain)
    # one gate fewer: no circuit, by the same levels
    low = len(circ) - 1
    if low:
        short = [W.spec_from_skeleton(spec, V, low) for V in (U, _scaled(U, j))]
        a, b = (cheese_amd.search(s) for s in short)
        assert a["rc"] == 1 and _strip(a) == _strip(b)


@pytest.mark.parametrize("n,count", [(3, 2304), (2, 4352)])
def test_a_frontier_of_thousands_of_roots(n, count):
    """one batch of `count` targets, each scaled by sqrt2^(0..3), against the same batch of normalised ones"""
    skel = W.skeleton(n)
    plain, scaled = [], []
    for i in range(count):
        circ = W.random_circuit(1000 + i % 96, n, 1, 3)
        U = W.unitary(n, circ)
        plain.append(W.spec_from_skeleton(skel, U, len(circ)))
        scaled.append(W.spec_from_skeleton(skel, _scaled(U, i % 4), len(circ)))
    print(f"{count} roots of {n} qubits", flush=True)
    want, got = cheese_amd.search_many(plain), cheese_amd.search_many(scaled)
    bad = [i for i in range(count) if want[i]["circuit_idx"] and _strip(want[i]) != _strip(got[i])]
    assert all(o["rc"] == 0 and o["verified"] for o in want)
    assert not bad, (len(bad), _strip(want[bad[0]]), _strip(got[bad[0]]))
