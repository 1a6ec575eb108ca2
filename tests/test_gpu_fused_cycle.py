"""The multigrid cycle's fused coarse levels on meshes where tiles end unevenly (odd and
even node counts on every axis, three and more levels, both cycle precisions): the CG
it preconditions takes the iterations of the cycle the hierarchy describes, and the
potential meets the tolerance on the operator as assembled.  A value missing at a
tile's edge makes the preconditioner unsymmetric there and shows in the count."""
import numpy as np
import pytest

from helpers import deck, emcgpu

pytestmark = pytest.mark.gpu


# 69 k to 298 k nodes
@pytest.mark.parametrize("refine,lg,wfin,fp32", [(2, 11, 4, 2), (2, 12, 5, 0), (2, 19, 8, 2), (3, 15, 5, 2), (3, 14, 6, 0)])
def test_fused_cycle(refine, lg, wfin, fp32):
    e = emcgpu.Engine(deck("fused", refine=refine, electrons=2000, holes=200, lg=lg, wfin=wfin), device=0,
                      poisson_fp32=fp32)
    try:
        m, ma = e.mesh, e.mesh_arrays()
        shp = (m.pny, m.pnx, m.pnz)
        free = np.asarray(ma["node_kind"]).reshape(shp) == 0
        e.particles_init()
        rhs = e.rhs_from_charge(e.deposit()[0])
        rng = np.random.default_rng(lg)
        noise = np.where(free.reshape(-1), rng.normal(size=m.nnode) * np.abs(rhs[free.reshape(-1)]).mean(), rhs)
        for b, most in ((rhs, 12), (noise, 14)):
            x, it, rel = e.poisson_solve(b)
            assert rel <= 1e-10 and 0 < it <= most, it
            u = x.reshape(shp)
            r = b.reshape(shp) - np.asarray(ma["diag"]).reshape(shp) * u
            for c, ax in (("cy", 0), ("cx", 1), ("cz", 2)):
                w = np.take(np.asarray(ma[c]).reshape(shp), range(shp[ax] - 1), axis=ax)
                lo, hi = [slice(None)] * 3, [slice(None)] * 3
                lo[ax], hi[ax] = slice(0, -1), slice(1, None)
                r[tuple(lo)] -= w * u[tuple(hi)]
                r[tuple(hi)] -= w * u[tuple(lo)]
            # the CG's residual and the one formed here differ by rounding, a few
            # hundred ulp of |A||x| at most
            scale = np.linalg.norm(np.asarray(ma["diag"]) * x)
            assert np.linalg.norm(r[free]) <= 1e-10 * np.linalg.norm(b) + 1e-13 * scale
    finally:
        e.close()
