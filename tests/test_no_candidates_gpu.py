"""A gate set without candidates: the search ends with a proof after its first, empty level, and leaves nothing behind that the
thread's next search would report."""
import pytest

import cheese_amd
from cheese_amd import specgen

from conftest import read_log, read_spec, strip_seconds

pytestmark = pytest.mark.gpu


def _toffoli_as_logged():
    out = cheese_amd.search(read_spec("toffoli-d8"))
    assert out["rc"] == 1, out.get("error")
    got = strip_seconds("\n".join(cheese_amd.level_line(lv) for lv in out["levels"]))
    assert got == [l for l in strip_seconds(read_log("toffoli-d8")) if "prefixes" in l]


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("dedupe", [True, False])
def test_a_search_without_candidates(n, dedupe):
    spec = specgen.spec_text(n, [("t", (0,))], 2, gates=())
    assert "gates 0\n" in spec
    out = cheese_amd.search(spec, dedupe=dedupe)
    assert out["rc"] == 1, out.get("error")
    assert [(lv["t"], lv["parents"], lv["prefixes"], lv["distinct"]) for lv in out["levels"]] == [(1, 1, 0, 0)]
    _toffoli_as_logged()


def test_a_search_of_no_survivors():
    """one candidate that the budget rules out: a level of one child and none kept"""
    spec = specgen.spec_text(3, [("h", (0,)), ("t", (0,)), ("h", (0,))], 1, gates=("h",))
    assert cheese_amd.search(spec)["rc"] == 1
    _toffoli_as_logged()
