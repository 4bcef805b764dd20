"""The specialised expansion (one table of one-qubit cuts, its kernel's own T columns at 3 qubits) against the general one:
naming a cut twice leaves every bound as it is, but only the general kernel takes such a spec, so the level lines and the
circuit of both are equal.  The largest searches here have frontiers past the size from which T columns are formed."""
import re

import pytest

import cheese_amd
from cheese_amd import workloads as W

from conftest import read_spec


def _cut_named_twice(spec):
    """the spec with its first cut repeated behind the others: entry idx of the cx table, whatever the new need is"""
    m = re.search(r"^cuts (\d+)\n((?:.*\n)*?)cxtable (\d+)\n(.*)\n", spec, re.M)
    n, lines, size, table = int(m.group(1)), m.group(2), int(m.group(3)), m.group(4)
    first = lines.splitlines()[0]
    return (spec[:m.start()] + f"cuts {n + 1}\n{lines}{first}\ncxtable {3 * size}\n" + " ".join([table.strip()] * 3) + "\n" +
            spec[m.end():])


def _strip(o):
    return (o["rc"], o.get("circuit_idx"), [{k: v for k, v in lv.items() if k != "seconds"} for lv in o["levels"]])


def _spec(case):
    if case[0] == "toffoli":
        return re.sub(r"^depth \d+", f"depth {case[1]}", read_spec("toffoli-d9"), count=1, flags=re.M)
    return W.random_spec(case[2], case[1], case[3], case[3])[1]


@pytest.mark.gpu
@pytest.mark.parametrize("case", [("toffoli", 1), ("toffoli", 9), ("toffoli", 11), ("random", 2, 3, 1), ("random", 2, 5, 11),
                                  ("random", 3, 4, 2), ("random", 3, 11, 10)], ids=lambda c: "-".join(map(str, c)))
def test_specialised_and_general_expansion_agree(case):
    spec = _spec(case)
    special, general = (cheese_amd.search(s, sym=False) for s in (spec, _cut_named_twice(spec)))
    assert _strip(special) == _strip(general)
