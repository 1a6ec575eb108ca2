"""A step whose Poisson solve fails (a potential that is not finite) returns the
solver's error before the fields, the corrected potential and the flight: fields,
population and counts stay as they were, and stepping goes on from there once the
potential is good again."""
import numpy as np
import pytest

from helpers import cfg1_deck, emcgpu, sort_by_key

pytestmark = pytest.mark.gpu

F = emcgpu.abi.CELL_FIELDS
P = emcgpu.abi.PARTICLE_F64 + emcgpu.abi.PARTICLE_I32 + ("key",)


def state(e):
    p = sort_by_key(e.download())
    f = e.fields_get()
    return {"n": p.n, **{k: getattr(p, k)[:p.n].copy() for k in P}, **{"f_" + k: getattr(f, k).copy() for k in F}}


def same(got, want, what):
    assert got["n"] == want["n"], what
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=f"{what} {k}")


def spoil(e):
    """The potential not a number, the fields as they were; what restore() needs."""
    pot, rho = e.potential(), e.fields_get().rho.copy()
    with pytest.raises(emcgpu.EmcError) as err:
        e.poisson_solve(np.zeros(e.mesh.nnode), x0=np.full(e.mesh.nnode, np.nan))
    assert err.value.code == emcgpu.abi.EMC_ERR_SOLVER
    return pot, rho


def failing(step):
    with pytest.raises(emcgpu.EmcError) as err:
        step()
    assert err.value.code == emcgpu.abi.EMC_ERR_SOLVER


# below and above the one-launch solve's largest mesh, without and with the quantum
# correction
@pytest.mark.parametrize("refine,qc", [(1, 0), (1, 1), (2, 0)])
def test_step_leaves_the_state(refine, qc):
    e = emcgpu.Engine(cfg1_deck(refine=refine, electrons=5000, holes=500, qc=qc), device=0)
    try:
        e.particles_init()
        e.step(2)
        before = state(e)
        pot, rho = spoil(e)
        e.tallies_reset()
        failing(lambda: e.step(1))
        same(state(e), before, "after the failed step")
        assert np.isnan(e.potential()).any()
        e.compute_field(pot, rho)
        e.step(2)
        assert np.isfinite(e.potential()).all()
        w = e.stat_window()
        assert w["steps"] == 2
        if qc:  # the corrected potential of the last good step, three times entered
            assert np.isfinite(w["stat_qc_pot"]).all()
    finally:
        e.close()
