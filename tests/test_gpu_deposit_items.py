"""Deposit of tiles whose particles are shared among several workgroups: populations
crowded into one tile, at and around whole shares, next to sparse ones, against the
oracle, every tally bit for bit."""
import numpy as np
import pytest

import oracle_lib
from helpers import cfg1_deck, emcgpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = emcgpu.Engine(cfg1_deck(electrons=6000, holes=600), device=0)
    e.particles_init()
    yield e, e.download()
    e.close()


# a share holds 768 particles
@pytest.mark.parametrize("crowd", [0, 1, 767, 768, 769, 1536, 1537, 5000])
def test_crowded_tile(eng, crowd):
    e, p0 = eng
    p = p0.subset(np.arange(min(p0.n, 7000)))
    m = e.mesh_arrays()
    rng = np.random.default_rng(crowd)
    # the first `crowd` particles into the 4 x 8 x 4 cells of one tile, of which a
    # quarter into a single cell
    c = np.arange(crowd)
    one = c % 4 == 0
    for f, lo, n, l, x in (("i", 8, 4, "lx", "x"), ("j", 16, 8, "ly", "y"), ("k", 4, 4, "lz", "z")):
        q = np.where(one, lo, lo + rng.integers(0, n, crowd)).astype(np.int32)
        getattr(p, f)[:crowd] = q
        u = rng.uniform(0, 1, crowd)
        getattr(p, x)[:crowd] = m[l][q] * u + m[l][q + 1] * (1 - u)
    e.upload(p)
    want = oracle_lib.deposit(e, p, p.n)
    for rep in range(2):  # the second sorts from the segments of the first
        got = e.deposit()
        for g, w, name in zip(got, want, ("node_q", "node_stat", "cell_q", "cell_n")):
            np.testing.assert_array_equal(g, np.asarray(w).reshape(-1), err_msg=f"{name} {rep}")
