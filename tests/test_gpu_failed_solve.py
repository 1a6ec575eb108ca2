"""A step whose Poisson solve fails (a potential that is not finite) returns the
solver's error before the fields, the corrected potential and the flight: fields,
population and counts stay as they were, for the device and for every other device
of its batch, and stepping goes on from there once the potential is good again."""
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


@pytest.mark.parametrize("refine,bad", [(1, 0), (1, 1), (1, 2), (2, 1)])
def test_batch_leaves_every_device(refine, bad):
    def engines():
        out = []
        for q in range(3):
            e = emcgpu.Engine(cfg1_deck(refine=refine, electrons=4000 + 500 * q, holes=400, vd=0.2 + 0.1 * q), device=0,
                              seed=5 + q)
            e.particles_init()
            out.append(e)
        return out
    together, alone = engines(), engines()
    b = emcgpu.Batch(together)
    try:
        b.step(2)
        before = [state(e) for e in together]
        start = [(e.potential(), e.fields_get().rho.copy()) for e in together]
        spoil(together[bad])
        failing(lambda: b.step(1))
        for q, e in enumerate(together):
            same(state(e), before[q], f"device {q} after the failed step")
        # the others' solves may have moved their start: put it back for all
        for e, (pot, rho) in zip(together, start):
            e.compute_field(pot, rho)
        acc = b.step(2)
        for q, e in enumerate(alone):
            # a device alone whose own step failed in between
            e.step(2)
            pot, rho = spoil(e)
            failing(lambda: e.step(1))
            e.compute_field(pot, rho)
            t = e.step(2)
            same(state(together[q]), state(e), f"device {q}")
            np.testing.assert_array_equal(together[q].potential(), e.potential())
            for k, v in emcgpu.tallies_dict(t).items():
                np.testing.assert_array_equal(emcgpu.tallies_dict(acc[q])[k], v, err_msg=f"device {q} {k}")
    finally:
        b.close()
        for e in together + alone:
            e.close()


def test_step_that_missed_the_tolerance_is_taken_up():
    """One iteration allowed: the step reports the solver's error, but it has flown,
    and its clones, tallies and window are the device's, alone and in a batch."""
    def engines():
        out = []
        for q in range(3):
            e = emcgpu.Engine(cfg1_deck(electrons=6000 + 500 * q, holes=600, vd=0.2 + 0.1 * q), device=0, seed=5 + q,
                              poisson_maxit=1)
            e.particles_init()
            out.append(e)
        return out
    together, alone = engines(), engines()
    b = emcgpu.Batch(together)
    try:
        for step in range(6):
            failing(lambda: b.step(1))
            for e in alone:
                failing(lambda: e.step(1))
        made = 0
        for q, (e, f) in enumerate(zip(together, alone)):
            same(state(e), state(f), f"device {q}")
            w, v = e.stat_window(), f.stat_window()
            assert w["steps"] == v["steps"] == 6
            t = emcgpu.tallies_dict(w["tallies"])
            for k, x in emcgpu.tallies_dict(v["tallies"]).items():
                np.testing.assert_array_equal(t[k], x, err_msg=f"device {q} {k}")
            made += t["n_gen"]
        assert made > 0  # the contacts put carriers in
    finally:
        b.close()
        for e in together + alone:
            e.close()


@pytest.mark.parametrize("refine", [1, 2])
def test_failed_batch_step_after_losses(refine):
    """The failed step's sort has dropped the slots of carriers that left in the step
    before: the count is that of the carriers that are left, none of them twice."""
    es = [emcgpu.Engine(cfg1_deck(refine=refine, electrons=20000, holes=2000, vd=0.6 + 0.1 * q), device=0, seed=2 + q)
          for q in range(2)]
    b = None
    try:
        for e in es:
            e.particles_init()
        b = emcgpu.Batch(es)
        for _ in range(200):
            acc = b.step(1)
            if all(t.n_catch > t.n_gen + 1 for t in acc):
                break
        else:
            pytest.fail("no step in which both devices lose carriers")
        before = [state(e) for e in es]
        spoil(es[1])
        failing(lambda: b.step(1))
        for q, e in enumerate(es):
            assert e.count() == before[q]["n"]
            same(state(e), before[q], f"device {q}")
    finally:
        if b:
            b.close()
        for e in es:
            e.close()
