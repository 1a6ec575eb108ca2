"""The effective potential's blocks of targets against the oracle's term-by-term sum,
bit for bit: meshes of odd sizes, a last block of few targets, windows cut by every
mesh face and rows of mixed shapes, and a window too large for a block, which takes
the kernel without staging."""
import os

import numpy as np
import pytest

from helpers import emcgpu
from test_gpu_qc import oracle_qc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refine,lg,wfin,ratio,region", [
    (1, 10, 4, 4, None),                   # windows of a few nodes
    (1, 13, 7, 60, None),                  # every window is the whole mesh
    (2, 11, 4, 4, None),                   # several blocks a plane
    (2, 15, 5, 4, (0, 10, -20, -18.5, 0, 5)),
    (2, 15, 5, 80, (0, 1, -20, -18, 0, 5)),  # one plane of the window exceeds a block's LDS
])
def test_blocks_equal_the_oracle(tmp_path, refine, lg, wfin, ratio, region):
    emcgpu.write_deck(str(tmp_path), refine=refine, electrons=100, holes=10, qc=1, lg=lg, wfin=wfin)
    ldg = os.path.join(str(tmp_path), "ldg.txt")
    text = open(ldg).read().replace("ep_parm 4 0.5 4 0.5 4 0.5 3.1", f"ep_parm {ratio} 0.5 {ratio} 0.5 {ratio} 0.5 3.1")
    if region:
        text = "\n".join("surface_scatter_range " + " ".join(map(str, region)) if l.startswith("surface_scatter_range")
                         else l for l in text.split("\n"))
    open(ldg, "w").write(text)
    e = emcgpu.Engine(str(tmp_path / "input.txt"), device=0)
    try:
        rng = np.random.default_rng(3)
        pot = rng.normal(size=e.mesh.nnode) * 10.0
        want = oracle_qc(e, pot)
        assert np.any(want != pot)
        np.testing.assert_array_equal(e.qc_potential(pot), want)
    finally:
        e.close()
