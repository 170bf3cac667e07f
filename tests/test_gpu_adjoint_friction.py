"""Gradients with the linear and the hybrid bottom friction laws, whose factors the adjoint stage forms at run time
(quadratic friction is fixed at compile time): the nonlinear equations in plane and spherical coordinates against
fourth-order central differences, and with a beach that floods and dries against the frozen-branch oracle."""
import numpy as np
import pytest

from dgswem_amd import adjoint, mesh
from oracle.oracle import Oracle
from test_gpu_adjoint import TOL, TOL_LIMITER, central_fd, directions, fd4, frozen_oracle_loss
from test_gpu_edge_cases import closed, wetdry_state

pytestmark = pytest.mark.gpu

LAWS = {"linear": 0, "hybrid": 2}


def set_law(case, law):
    p = case.params
    p.nolibf = LAWS[law]
    p.hbreak, p.ftheta, p.fgamma = 4.0, 3.0, 0.4


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("ics", [1, 2])
@pytest.mark.parametrize("law", LAWS)
def test_against_central_differences(p, ics, law):
    c = mesh.delaunay_basin(n_elem=900, seed=31, lx=6.0e4, ly=3.6e4, depth_range=(2.0, 10.0), shelf=False, wetdry=False,
                            slopeflag=0, p=p, nsteps=40, cf=1e-4, ics=ics, cfl=0.3 if p == 1 else 0.15)
    set_law(c, law)
    prob = adjoint.twin_problem(c, nsteps=40, ng=20, seed=5, perturb=0.5)
    J, gn, gdp = prob.gradient(c.manning, c.dp)
    assert J > 0.0 and np.abs(gn).max() > 0.0 and np.isfinite(gdp).all()
    z = np.zeros(c.np_)
    for i, (vn, vd) in enumerate(directions(c, 3, seed=12)):
        # the friction's own parameter alone once, and both together
        for a, b in ((vn, z), (vn, vd)) if i == 0 else ((vn, vd),):
            ad = float(gn @ a + gdp @ b)
            fd = central_fd(prob, c, a, b)
            print(f"adjoint {ad:.12e} fd {fd:.12e} rel {abs(fd - ad) / abs(ad):.2e}", flush=True)
            assert abs(fd - ad) <= TOL * abs(ad)
    prob.solver.close()


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("law", LAWS)
def test_with_wetting_and_drying_against_the_frozen_branch_oracle(p, law):
    """The basin, the step of the differences and the map are those of the quadratic law's test, where the kinks of the
    wave-speed bound at the shoreline leave up to 8e-7 at this step; they leave the differences here a tolerance of
    1e-5."""
    nst = 40
    c = closed(12, 6, p, nolifa=2, slopeflag=5)
    c.dp = 2.0 - 0.0004 * c.x
    c.manning = 0.02 + 0.01 * np.random.default_rng(4).random(c.np_)
    set_law(c, law)
    st = wetdry_state(c, 2.0)
    prob = adjoint.twin_problem(c, nsteps=nst, ng=20, seed=8, state0=st, perturb=0.5)
    J, gn, gdp = prob.gradient(c.manning, c.dp)
    o = Oracle(c, threads=8)
    o.set_state(*st)
    o.limiter_record(nst)
    o.step(nst)
    records = o.limiter_records()
    assert (np.bincount(records[2] & 3, minlength=4)[2:] > 0).all()
    loss = frozen_oracle_loss(c, prob, 20, 8, records)
    assert loss(c.manning, c.dp) == pytest.approx(J, rel=1e-9, abs=0.0)
    for vn, vd in directions(c, 3, seed=13):
        ad = float(gn @ vn + gdp @ vd)
        fd = fd4(lambda t: loss(c.manning + t * vn, c.dp + t * vd), 1e-6)
        print(f"adjoint {ad:.12e} frozen-branch oracle fd {fd:.12e} rel {abs(fd - ad) / abs(ad):.2e}", flush=True)
        assert abs(fd - ad) <= TOL_LIMITER * abs(ad)
    prob.solver.close()
