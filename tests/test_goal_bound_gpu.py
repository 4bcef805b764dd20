"""A cx table whose entry for no need at all is not 0 gives the goal itself a bound above 0.  The goal is looked for before
the bounds, so a circuit whose last gate leaves no budget for such a bound is found all the same: level lines and circuit
are the oracle's."""
import re

import pytest

import cheese_amd
from cheese_amd import specgen

from conftest import oracle_run, strip_seconds


def _raised(spec, by):
    """the spec with the first entry of its cx table raised"""
    return re.sub(r"^(cxtable \d+)\n0", rf"\1\n{by}", spec, count=1, flags=re.M)


@pytest.mark.gpu
@pytest.mark.parametrize("by", [1, 2])
@pytest.mark.parametrize("n,gates,circ", [
    (1, ("h", "t"), [("h", (0,)), ("t", (0,))]),
    (2, ("h", "cx"), [("h", (0,)), ("cx", (1, 0))]),
    (2, ("h", "cx"), [("cx", (0, 1)), ("h", (0,)), ("cx", (1, 0))]),
    (2, ("t", "cx"), [("cx", (0, 1)), ("t", (1,)), ("cx", (0, 1)), ("t", (0,))]),
], ids=["ht", "h-cx", "cx-h-cx", "cx-t-cx-t"])
def test_the_goal_is_found_past_its_own_bound(oracle_lib, n, gates, circ, by):
    spec = _raised(specgen.spec_text(n, circ, len(circ), gates=gates), by)
    assert f"\n{by}" in spec
    rc, log = oracle_run(oracle_lib, spec)
    lines = strip_seconds(log)
    out = cheese_amd.search(spec)
    assert out["rc"] == rc
    assert strip_seconds("\n".join(cheese_amd.level_line(lv) for lv in out["levels"])) == [l for l in lines if "prefixes" in l]
    if rc == 0:
        assert out["verified"] and out["circuit"] == [l["circuit"] for l in lines if "circuit" in l][0]
