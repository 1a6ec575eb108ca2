"""The forms of the solve against each other: one launch on one XCD, kernel by kernel,
and the redo of a one-launch solve whose blocks gave up finding together or waiting for
one another.  Potential, iterations and residual are the same bit for bit on the same
right-hand side, from a single-level mesh to both sides of the largest mesh that is
solved in one launch; so are the steps of a device and of a batch."""
import numpy as np
import pytest

from helpers import bulk_deck, cfg1_deck, deck, emcgpu, sort_by_key

pytestmark = pytest.mark.gpu

A = emcgpu.abi
FORMS = (A.SOLVE_AUTO, A.SOLVE_KERNELS, A.SOLVE_NO_MEET, A.SOLVE_NO_WAIT)
LARGEST = 32768

MESHES = {
    "single_level": (lambda: bulk_deck(cells=7, electrons=500, holes=500), 512),
    "small": (lambda: deck("forms", refine=1, electrons=2000, holes=200, lg=10, wfin=4), 9072),
    "odd": (lambda: deck("forms", refine=1, electrons=2000, holes=200, lg=30, wfin=8), 18816),
    "largest": (lambda: deck("forms", refine=1, electrons=2000, holes=200, lg=60, wfin=10), 32508),
    "beyond": (lambda: deck("forms", refine=1, electrons=2000, holes=200, lg=61, wfin=10), 32886),
}


@pytest.mark.parametrize("fp32", [2, 0])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_forms_agree(mesh, fp32):
    inp, nodes = MESHES[mesh]
    e = emcgpu.Engine(inp(), device=0, poisson_fp32=fp32)
    try:
        assert e.mesh.nnode == nodes
        rng = np.random.default_rng(nodes)
        scale = np.abs(np.asarray(e.mesh_arrays()["diag"]))
        rhs, x0 = rng.normal(size=nodes) * scale, rng.normal(size=nodes)
        got, redone = {}, 0
        for form in FORMS:
            assert e.poisson_form(form) == redone
            got[form] = [e.poisson_solve(rhs), e.poisson_solve(rhs, x0=x0), e.poisson_solve_noalloc(rhs, x0=x0)]
            m = e.poisson_solve_mixed(rhs, x0)
            got[form].append((m[0], m[1:3], m[3]))
            now = e.poisson_form()
            if form in (A.SOLVE_AUTO, A.SOLVE_KERNELS) or nodes > LARGEST:
                assert now == redone
            elif form == A.SOLVE_NO_MEET or nodes > 512:  # one block waits for no one
                assert now == redone + 3 + m[1]  # the mixed solve's refinements are one each
            else:
                assert now == redone
            redone = now
        want = got[A.SOLVE_KERNELS]
        assert want[0][1] > 0 and want[0][2] <= 1e-10
        for form in FORMS:
            for q, (x, it, rel) in enumerate(got[form]):
                np.testing.assert_array_equal(x, want[q][0], err_msg=f"form {form} solve {q}")
                assert it == want[q][1] and rel == want[q][2], (form, q)
    finally:
        e.close()


def result(e, t):
    p = sort_by_key(e.download())
    out = {f: getattr(p, f)[:p.n] for f in A.PARTICLE_F64 + A.PARTICLE_I32 + ("key",)}
    f = e.fields_get()
    out.update({k: getattr(f, k) for k in A.CELL_FIELDS})
    w = e.stat_window()
    out.update({k: np.asarray(w[k]) for k in ("stat_pot", "stat_qc_pot", "node_stat", "cell_count", "rcur", "lcur")})
    out.update({"t_" + k: v for k, v in emcgpu.tallies_dict(t).items()})
    out["pot"] = e.potential()
    return out


def same(got, want, what):
    assert sorted(got) == sorted(want)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=f"{what} {k}")


@pytest.mark.parametrize("qc,fp32", [(0, 2), (1, 0), (0, 1)])
def test_step_redone(qc, fp32):
    """A step whose solve is redone is the step of a solve that was not."""
    want = None
    for form in FORMS:
        e = emcgpu.Engine(cfg1_deck(electrons=5000, holes=500, qc=qc), device=0, poisson_fp32=fp32)
        try:
            e.particles_init()
            e.poisson_form(form)
            got = result(e, e.step(4))
            redone = e.poisson_form()
            if form in (A.SOLVE_AUTO, A.SOLVE_KERNELS):
                assert redone == 0
            else:
                assert redone >= 4 if fp32 == 1 else redone == 4
            if want is None:
                want = got
            same(got, want, f"form {form}")
        finally:
            e.close()


@pytest.mark.parametrize("fp32", [2, 0])
@pytest.mark.parametrize("form", FORMS[1:])
def test_batch_redone(form, fp32):
    """A batch in which one device's solve is redone: every device takes the step that
    it takes alone, kernel by kernel."""
    def engines():
        out = []
        for q in range(3):
            e = emcgpu.Engine(cfg1_deck(electrons=4000 + 500 * q, holes=400, vd=0.2 + 0.1 * q), device=0, seed=5 + q,
                              poisson_fp32=fp32)
            e.particles_init()
            out.append(e)
        return out
    together, alone = engines(), engines()
    together[1].poisson_form(form)
    b = emcgpu.Batch(together)
    try:
        acc = b.step(4)
        assert [e.poisson_form() for e in together] == [0, 0 if form == A.SOLVE_KERNELS else 4, 0]
        for q, e in enumerate(alone):
            e.poisson_form(A.SOLVE_KERNELS)
            same(result(together[q], acc[q]), result(e, e.step(4)), f"device {q}")
    finally:
        b.close()
        for e in together + alone:
            e.close()
