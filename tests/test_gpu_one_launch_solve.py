"""The solve in one launch (small meshes): every device of a batch gets the potential
of its step alone bit for bit, however many blocks a device has and however many
devices share an XCD, and the potential meets the tolerance on the operator as
assembled, whatever was solved before it."""
import numpy as np
import pytest

from helpers import deck, emcgpu

pytestmark = pytest.mark.gpu


# meshes of 9 k to 18 k nodes: one node per thread in 18 blocks, a last block of few
# nodes, and a mesh whose partial sums fill more than one pass of the blocks
@pytest.mark.parametrize("lg,wfin,points,fp32", [(10, 4, 1, 2), (15, 5, 9, 2), (30, 8, 2, 2), (13, 4, 17, 0)])
def test_batch_equals_alone(lg, wfin, points, fp32):
    def engines():
        out = []
        for q in range(points):
            d = deck("one_launch", refine=1, electrons=2000 + 100 * q, holes=200, vd=0.1 + 0.02 * q, vg=0.5, lg=lg,
                     wfin=wfin, phims=0.3)
            e = emcgpu.Engine(d, device=0, seed=3 + q, poisson_fp32=fp32)
            e.particles_init()
            out.append(e)
        return out
    alone, together = engines(), engines()
    b = emcgpu.Batch(together)
    try:
        b.step(3)
        for e, f in zip(alone, together):
            e.step(3)
            np.testing.assert_array_equal(e.potential(), f.potential())
    finally:
        b.close()
        for e in alone + together:
            e.close()


@pytest.mark.parametrize("lg,wfin", [(10, 4), (15, 5), (30, 8)])
def test_solve_meets_the_tolerance(lg, wfin):
    """The residual of the returned potential on the assembled operator is within
    the tolerance (1e-10) and the result of a run on another right-hand side in
    between does not enter it."""
    e = emcgpu.Engine(deck("one_launch_res", refine=1, electrons=2000, holes=200, lg=lg, wfin=wfin), device=0)
    try:
        e.particles_init()
        rhs = e.rhs_from_charge(e.deposit()[0])
        x, it, rel = e.poisson_solve(rhs)
        assert 0 < it < 20 and rel <= 1e-10
        e.poisson_solve(2.0 * rhs)
        y, _, _ = e.poisson_solve(rhs)
        np.testing.assert_array_equal(x, y)
        z, _, _ = e.poisson_solve_noalloc(rhs)
        np.testing.assert_array_equal(x, z)
        m, ma = e.mesh, e.mesh_arrays()
        shp = (m.pny, m.pnx, m.pnz)
        u = x.reshape(shp)
        r = rhs.reshape(shp) - np.asarray(ma["diag"]).reshape(shp) * u
        for c, ax in (("cy", 0), ("cx", 1), ("cz", 2)):
            w = np.take(np.asarray(ma[c]).reshape(shp), range(shp[ax] - 1), axis=ax)
            lo = [slice(None)] * 3
            hi = [slice(None)] * 3
            lo[ax], hi[ax] = slice(0, -1), slice(1, None)
            r[tuple(lo)] -= w * u[tuple(hi)]
            r[tuple(hi)] -= w * u[tuple(lo)]
        free = np.asarray(ma["node_kind"]).reshape(shp) == 0
        # the recomputed residual rounds at a few ulp of |A||x|, far below 1e-10 |b|
        assert np.linalg.norm(r[free]) <= 1.01e-10 * np.linalg.norm(rhs)
        assert e.poisson_solve(rhs, x0=x)[1] == 0  # a start within the tolerance takes no iteration
    finally:
        e.close()
