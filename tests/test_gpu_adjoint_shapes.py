"""The adjoint stage kernel at the edges of its tiles of 64 elements (one short, a full tile, one pair more, several
tiles), at both orders, with ocean, land and flow sides, the nonlinear and the linearised equations: gradients against
fourth-order central differences, with the tolerance of the gradient tests on larger meshes (the difference's
truncation is O(1e-16), its rounding about 1e-13/1e-4)."""
import numpy as np
import pytest

from dgswem_amd import adjoint, mesh
from test_gpu_adjoint import TOL, central_fd, directions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(31, 1), (8, 4), (11, 3), (13, 8)])
@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("nonlinear", [1, 0])
def test_tile_edges(nx, ny, p, nonlinear):
    c = mesh.structured_basin(nx=nx, ny=ny, dx=900.0, dy=1100.0, depth=6.0, amp=0.3, p=p, dt=6.0 if p == 1 else 3.0,
                              flow_side=True, flow_amp=0.5, cori=1.0e-4)
    c.params.nolica = c.params.nolicat = nonlinear
    c.params.cf = 1e-4
    rng = np.random.default_rng(nx * 10 + p)
    c.x = c.x + rng.uniform(-60.0, 60.0, c.np_)          # no two sides alike: no ties between wave speeds
    c.y = c.y + rng.uniform(-60.0, 60.0, c.np_)
    c.dp = c.dp * (1.0 + 0.2 * rng.uniform(-1.0, 1.0, c.np_))
    prob = adjoint.twin_problem(c, nsteps=20, ng=7, seed=3)
    J, gn, gdp = prob.gradient(c.manning, c.dp)
    assert J > 0.0 and np.isfinite(gn).all() and np.isfinite(gdp).all()
    for vn, vd in directions(c, 3, seed=8):
        ad = float(gn @ vn + gdp @ vd)
        fd = central_fd(prob, c, vn, vd)
        print(f"adjoint {ad:.12e} fd {fd:.12e} rel {abs(fd - ad) / abs(ad):.2e}", flush=True)
        assert abs(fd - ad) <= TOL * abs(ad)


# runs kept whole (no spacing given) against runs recomputed from checkpoints: over the ends of the forcing tables'
# 2048 steps, and with limiter, wetting and drying
@pytest.mark.parametrize("steps,interval", [(1, 1), (2047, 100), (2048, 100), (2049, 500), (4100, 999)])
def test_kept_stages_equal_recomputed_ones(steps, interval):
    c = mesh.structured_basin(nx=11, ny=3, dx=900.0, dy=1100.0, depth=6.0, amp=0.3, dt=6.0)
    prob = adjoint.twin_problem(c, nsteps=steps, ng=7, seed=3)
    ref = prob.solver.gradient(prob.data, prob.weight, interval)
    prob.reset()
    out = prob.solver.gradient(prob.data, prob.weight, 0)
    for a, b in zip(out, ref):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("p", [1, 2])
def test_kept_flags_equal_recomputed_ones(p):
    c = mesh.delaunay_basin(n_elem=700, seed=34, p=p, lx=6.0e4, ly=3.6e4, depth_range=(2.0, 10.0), shelf=True,
                            wetdry=True, slopeflag=5, nsteps=40, cf=1e-4)
    prob = adjoint.twin_problem(c, nsteps=40, ng=9, seed=5, state0="cold")
    outs = []
    for interval in (0, 7, 0, 40):
        prob.reset()
        outs.append(prob.solver.gradient(prob.data, prob.weight, interval))
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            np.testing.assert_array_equal(a, b)
