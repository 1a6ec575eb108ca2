"""The teams of blocks that solve a small mesh in one launch: however many devices share
an XCD (eight XCDs of four shader engines with eight CUs each, a block a CU), all their
teams fit on it at once, counted by engines, and a batch whose XCDs would hold more
than 36 k nodes each is solved kernel by kernel."""
import ctypes as C

import pytest

from helpers import emcgpu


@pytest.fixture(scope="module")
def blocks():
    f = C.CDLL(emcgpu.LIB_PATH).emc_xcd_blocks
    f.restype, f.argtypes = C.c_int, [C.c_size_t, C.c_int, C.c_int]
    return lambda n, k: f(n, k, 256)


@pytest.mark.parametrize("nodes", [27, 512, 513, 4096, 9072, 11193, 13524, 18432, 18433, 32508, 32768])
def test_teams_fit(blocks, nodes):
    for k in range(1, 129):
        per, b = -(-k // 8), blocks(nodes, k)
        if b == 0:
            assert nodes * per > 36864 or per > 8, (k, b)
            continue
        assert nodes * per <= 36864
        assert b <= -(-nodes // 512)  # no block without a node
        # every team's blocks go to the engines in turn: the fullest has their ceilings
        assert per * -(-b // 4) <= 8, (k, b)


def test_one_device_has_a_thread_per_node(blocks):
    assert [blocks(n, 1) for n in (27, 512, 513, 9072, 16384, 32768)] == [1, 1, 2, 18, 32, 32]
