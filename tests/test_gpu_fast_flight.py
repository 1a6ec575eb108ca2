"""The fast pass of the flight against the oracle, bit for bit, where its bounds and
reciprocals have to hand a particle over: particles on cell faces and corners and a
rounding error beside them, steps with hardly an event and with dozens, reflecting,
periodic and surface-scattering faces, fields of zero and strong ones."""
import numpy as np
import pytest

import oracle_lib
from helpers import bulk_deck, deck, emcgpu, field_like, uniform_fields
from test_gpu_parity import assert_same_population, assert_same_tallies

pytestmark = pytest.mark.gpu

DECKS = {
    "fin": lambda dt: deck("fast", electrons=6000, holes=1500, dt=dt),
    "fin_plain": lambda dt: deck("fast", electrons=6000, holes=1500, dt=dt, surface=0),
    "bulk": lambda dt: bulk_deck(electrons=4000, holes=4000, dt=dt),
    "bulk_doped": lambda dt: bulk_deck(electrons=4000, holes=4000, dt=dt, donor=1e25),
}


@pytest.mark.parametrize("kind", sorted(DECKS))
@pytest.mark.parametrize("dt", [1e-19, 1e-16, 4e-15])
@pytest.mark.parametrize("field", ["zero", "strong", "device"])
def test_edges(kind, dt, field):
    e = emcgpu.Engine(DECKS[kind](dt), device=0)
    try:
        e.particles_init()
        p = e.download()
        m = e.mesh_arrays()
        live = np.nonzero(p.i[:p.n] >= 0)[0]
        q = np.arange(len(live))
        # a third as sampled; of the rest each coordinate on the cell's lower or upper
        # face, or the next number inside it, or as sampled
        how = np.random.default_rng(5).integers(0, 5, (3, len(live)))
        for a, (x, i, l) in enumerate((("x", "i", "lx"), ("y", "j", "ly"), ("z", "k", "lz"))):
            v, c = getattr(p, x), getattr(p, i)[live]
            lo, hi = m[l][c], m[l][c + 1]
            new = np.choose(how[a], [lo, hi, np.nextafter(lo, hi), np.nextafter(hi, lo), v[live]])
            v[live] = np.where(q % 3 == 0, v[live], new)
        e.upload(p)
        if field == "device":
            _, f = field_like(e, seed=2, scale=15.0)
        else:
            f = uniform_fields(e, *((0.0, 0.0, 0.0) if field == "zero" else (25.0, -30.0, 8.0)))
        e.fields_set(f)
        e.tallies_reset()
        po = e.download()
        for step in range(2):
            tg = e.fly_step(700 + step)
            pg = e.download()
            po, to, _ = oracle_lib.fly_step(e, po, po.n, f, 700 + step)
            assert_same_tallies(tg, to, f"step {step}")
            assert_same_population(pg, po, f"step {step}")
            po = pg
    finally:
        e.close()
