"""The stage kernel's forms against each other, bit for bit, in the variants that larger runs use: storm basins at both
orders with and without the limiter, as single runs and batched, the tidal potential, the schemes that keep their
right-hand sides, and the one-lane form's block sizes above the size to which four waves per 64 elements run (a block
of 128 is the one-lane form at every size).  And the range check of the short flux against the oracle."""
import numpy as np
import pytest

from conftest import load_case
from dgswem_amd import gpu, mesh
from oracle.oracle import Oracle
from test_gpu_edge_cases import closed
from test_gpu_stage_shapes import run, same

pytestmark = pytest.mark.gpu


def storm(n, seed, p, slopeflag=5):
    return mesh.storm_basin(n, seed=seed, p=p, slopeflag=slopeflag, depth_range=(2.0, 30.0), cfl=0.25 if p == 1 else 0.12)


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("slopeflag", [0, 5])
def test_storm_basin(p, slopeflag):
    c = storm(3000, 21, p, slopeflag)
    out = run(c, 40)
    assert (out[3] == 0).any() and (out[3] == 1).any()
    same(out, run(c, 40, block=128))


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("graph", [False, True])
def test_storm_ensemble(p, graph):
    outs = []
    for block in (None, 128):
        ms = [gpu.GpuSolver(storm(n, 30 + k, p)) for k, n in enumerate((1500, 2600, 900))]
        e = gpu.Ensemble(ms)
        e.use_graph(graph)
        if block:
            e.set_block(block)
        e.step(41)
        outs.append(e.state())
        for s in ms + [e]:
            s.close()
    same(*outs)


@pytest.mark.parametrize("p", [1, 2])
def test_tidal_potential(p):
    c = load_case("tipot2k")
    c.dg.pl = c.dg.ph = p
    c.params.dtdp = c.params.dtdp / p
    same(run(c, 30), run(c, 30, block=128))


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("stages,order", [(3, 2), (4, 2), (5, 2), (3, 3)])
def test_schemes_with_kept_rhs(p, stages, order):
    c = mesh.structured_basin(nx=20, ny=9, dx=500.0, dy=500.0, depth=6.0, amp=0.4, manning=None, p=p, dt=2.0, rk_stage=stages,
                              slopeflag=0, nolifa=2, nolibf=0, cori=1.0e-4, flow_side=True, flow_amp=1.0)
    c.dg.rk_order = order
    same(run(c, 30), run(c, 30, block=128))


@pytest.mark.parametrize("p,n", [(1, 100000), (2, 93000)])
def test_one_lane_block_sizes_on_larger_storm_basins(p, n):
    c = storm(n, 41, p)
    ref = run(c, 12, block=128)
    same(run(c, 12, block=64), ref)
    same(run(c, 12), ref)
    if p == 1:
        same(run(c, 12, block=256), ref)


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("depth", [2.0 ** -499, 2.0 ** -500, np.nextafter(2.0 ** -500, 0.0), 2.0 ** -501, 2.0 ** -510, 0.0, -0.5])
def test_depths_at_the_short_fluxs_limit(p, depth):
    """One forward Euler step with a few elements at rest of this depth among ones of half a metre and more.  For
    positive depths every value is finite and equals the oracle's.  A depth of zero or less makes NaN in the elements
    that touch it, where the oracle's wave-speed bound keeps one that the device's maximum drops: the others equal the
    oracle's, and the two forms agree everywhere."""
    c = closed(12, 10, p)
    c.dg.rk_stage = c.dg.rk_order = 1
    c.params.h0 = 0.0
    n, dof = c.ne, 3 if p == 1 else 6
    low = np.zeros(n, bool)
    low[[40, 41, 111, 180]] = True                       # two of them share a side
    at_low = np.isin(np.arange(1, c.np_ + 1), c.nm[low])
    c.dp = np.where(at_low, 0.0, 10.0)
    rng = np.random.default_rng(2)
    ze, qx, qy = np.zeros((n, dof)), np.zeros((n, dof)), np.zeros((n, dof))
    ze[:, 0] = 0.5 + rng.uniform(0.0, 0.5, n)
    qx[:, 0], qy[:, 0] = rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n)
    ze[low, 0], qx[low], qy[low] = depth, 0.0, 0.0
    wd = np.ones(n, np.int32)
    o = Oracle(c, threads=1)
    o.set_state(ze, qx, qy, wd)
    o.step(1)
    ref = o.state()
    out = run(c, 1, (ze, qx, qy, wd))
    same(out, run(c, 1, (ze, qx, qy, wd), block=128))
    touch = low if depth > 0.0 else np.isin(c.nm, np.flatnonzero(at_low) + 1).any(axis=1)
    ok = np.ones(n, bool) if depth > 0.0 else ~touch
    assert ok.sum() >= 0.8 * n
    for a, b in zip(out[:3], ref[:3]):
        assert np.isfinite(b[ok]).all()
        np.testing.assert_array_equal(a[ok], b[ok])
