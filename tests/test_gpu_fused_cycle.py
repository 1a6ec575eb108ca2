"""The multigrid cycle's fused coarse levels on meshes where tiles end unevenly (odd and
even node counts on every axis, three and more levels, both cycle precisions): the CG
it preconditions takes the iterations of the cycle the hierarchy describes, and the
potential meets the tolerance on the operator as assembled, and its first iterates are
those of the same CG and cycle on the CPU, node by node.  (On the meshes that are also
solved in one launch, whose cycle is not fused, test_gpu_solver_forms.py compares the
two bit for bit.)"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import deck, emcgpu
from test_multigrid import a27_to_csr, fine_operator, pcg, prolong_1d, vcycle

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


# the first iterates against the same CG on the CPU, its cycle from the hierarchy's own
# operators level by level in FP64
@pytest.mark.parametrize("refine,lg,wfin,fp32", [(2, 11, 4, 2), (2, 12, 5, 0), (3, 14, 6, 2)])
def test_iterates_are_the_hierarchy_s(refine, lg, wfin, fp32):
    e = emcgpu.Engine(deck("fused", refine=refine, electrons=2000, holes=200, lg=lg, wfin=wfin), device=0,
                      poisson_fp32=fp32)
    try:
        A, fixed, _ = fine_operator(e)
        lv = e.mg_levels()
        ops, fx, Ps = [A], [fixed], []
        for level in range(1, len(lv)):
            fd = lv[level - 1][0]
            P = sp.kron(sp.kron(prolong_1d(fd[1]), prolong_1d(fd[0])), prolong_1d(fd[2])).tocsr()
            Ps.append(sp.diags((~fx[-1]).astype(float)) @ P)
            ops.append(a27_to_csr(lv[level][1], lv[level][0]))
            fx.append(np.asarray(abs(ops[-1]).sum(axis=1)).ravel() == ops[-1].diagonal())
        cinv = np.linalg.inv(ops[-1].toarray())
        rng = np.random.default_rng(lg)
        b = np.where(fixed, 0.0, rng.normal(size=A.shape[0]) * A.diagonal())
        for n in (1, 2, 4):
            want, _ = pcg(A, b, fixed, lambda r: vcycle(lv, ops, fx, Ps, cinv, 0, r), rtol=0.0, maxit=n)
            got, it, rel = np.zeros_like(b), C.c_int(0), C.c_double(0)
            d = lambda x: x.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
            st = e.lib.emc_poisson_solve(e.ctx, d(b), d(got), 1e-10, n, C.byref(it), C.byref(rel))
            assert st == emcgpu.abi.EMC_ERR_SOLVER and it.value == n  # stopped before the tolerance
            # The coarse operators are held in FP32 (6e-8 of a coefficient), the FP32
            # cycle's vectors too; a handful of sweeps and levels and the CG's own
            # amplification (condition below 10) leave well under these bounds, a value
            # missing or wrong at a tile's edge is of the order of the iterate itself.
            bound = (2e-4 if fp32 else 2e-5) * np.abs(want).max()
            assert np.abs(got - want).max() <= bound, (n, np.abs(got - want).max() / np.abs(want).max())
    finally:
        e.close()
