"""Everything a device's steps work in is allocated with its population, the deposit's
blocks too: the memory in use does not grow from the initial population to the first
step, nor with more of them, so a server's measured footprint is the request's whole."""
import pytest
import torch

from helpers import deck, emcgpu

pytestmark = pytest.mark.gpu


def used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


# 76 800 cells: 600 tiles; 600 k slots: 800 further blocks
@pytest.mark.parametrize("refine,electrons", [(2, 2000), (2, 300000), (1, 300000)])
def test_steps_allocate_nothing(refine, electrons):
    warm = []
    try:
        # the runtime's own buffers (a queue's scratch) come with each queue's first use
        for q in range(8):
            e = emcgpu.Engine(deck("warm", refine=1, electrons=100, holes=10), device=0)
            warm.append(e)
            e.particles_init()
            e.step(2)
        e = emcgpu.Engine(deck("mem", refine=refine, electrons=electrons, holes=electrons // 10), device=0)
        warm.append(e)
        e.particles_init()
        before = used()
        e.step(1)
        first = used()
        e.step(3)
        e.deposit()
        # below one block of the allocator; the deposit's blocks here are 5 to 28 MB
        assert first - before < 2 << 20 and used() - first < 2 << 20, (before, first, used())
    finally:
        for e in warm:
            e.close()
