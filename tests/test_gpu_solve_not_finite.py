"""A Poisson solve whose residual is not a number is an error in every form of the
call, on meshes solved in one launch and on larger ones, in a step and in a batch;
it is not taken for a residual of zero."""
import numpy as np
import pytest

from helpers import cfg1_deck, emcgpu

pytestmark = pytest.mark.gpu

SOLVER = emcgpu.abi.EMC_ERR_SOLVER


def refused(call):
    with pytest.raises(emcgpu.EmcError) as err:
        call()
    assert err.value.code == SOLVER


@pytest.mark.parametrize("refine", [1, 2])
@pytest.mark.parametrize("fp32", [2, 0])
@pytest.mark.parametrize("where", ["start", "rhs"])
@pytest.mark.parametrize("what", [np.nan, np.inf])
def test_solve(refine, fp32, where, what):
    e = emcgpu.Engine(cfg1_deck(refine=refine, electrons=3000, holes=300), device=0, poisson_fp32=fp32)
    try:
        e.particles_init()
        rhs, x0 = e.rhs_from_charge(e.deposit()[0]), np.zeros(e.mesh.nnode)
        free = np.flatnonzero(np.asarray(e.mesh_arrays()["node_kind"]) == 0)
        (x0 if where == "start" else rhs)[free[len(free) // 2]] = what
        refused(lambda: e.poisson_solve(rhs, x0=x0))
        refused(lambda: e.poisson_solve_noalloc(rhs, x0=x0))
        refused(lambda: e.poisson_solve_mixed(rhs, x0))
    finally:
        e.close()


@pytest.mark.parametrize("refine", [1, 2])
def test_step_and_batch(refine):
    es = [emcgpu.Engine(cfg1_deck(refine=refine, electrons=3000 + 100 * q, holes=300), device=0) for q in range(3)]
    b = None
    try:
        for e in es:
            e.particles_init()
        b = emcgpu.Batch(es)
        b.step(2)
        nan = np.full(es[1].mesh.nnode, np.nan)
        refused(lambda: es[1].poisson_solve(np.zeros(es[1].mesh.nnode), x0=nan))
        refused(lambda: b.step(1))
        refused(lambda: es[1].step(1))
    finally:
        if b:
            b.close()
        for e in es:
            e.close()
