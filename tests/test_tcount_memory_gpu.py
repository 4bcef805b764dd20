"""A closed T-count table gives back all of its device memory: opening and closing tables again and again leaves the card's
free memory where the second table left it (the first one fills the block cache)."""
import ctypes

import pytest

from cheese_amd import tcount as T

from conftest import read_tspec


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.gpu
def test_closed_tables_give_their_memory_back():
    spec = read_tspec("toffoli")
    free = []
    for _ in range(10):
        table = T.CosetTable(spec, K=4)
        size = table.size
        table.close()
        assert size == 5605741
        free.append(_free_bytes())
    # one table's 8.13 million children hold 32 MB in a 4-byte array: below that no buffer of the last level is lost
    assert free[1] - free[-1] < 16 << 20, [free[1] - f for f in free]
