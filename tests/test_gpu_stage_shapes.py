"""The two forms of the stage kernel (one lane per element; four waves per 64 elements, the rule for small
meshes) and the fluxes' range check, against each other and against the oracle, bit for bit.

Closed basins with uniform friction (no transcendental function on the path) equal the oracle exactly; with
tides, Manning friction or Holland forcing the two forms equal each other exactly.
"""
import numpy as np
import pytest

from conftest import load_case
from dgswem_amd import adjoint, gpu, mesh
from oracle.oracle import Oracle
from test_gpu_edge_cases import closed, wetdry_state

pytestmark = pytest.mark.gpu


def run(case, steps, state0=None, block=None):
    g = gpu.GpuSolver(case)
    if state0 is not None:
        g.set_state(*state0)
    if block:
        g.set_block(block)
    g.step(steps)
    out = g.state()
    g.close()
    return out


def same(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


# one element pair, one short of a tile, a full tile, one pair more, two tiles
@pytest.mark.parametrize("nx,ny", [(1, 1), (31, 1), (8, 4), (11, 3), (8, 8)])
@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("slopeflag", [0, 5])
def test_tile_edges(nx, ny, p, slopeflag):
    c = closed(nx, ny, p, nolifa=2, slopeflag=slopeflag)
    c.dp = 2.0 - 2.5 * c.x / max(c.x.max(), 1.0)            # dry in the east
    st = wetdry_state(c, 0.5)
    o = Oracle(c, threads=2)
    o.set_state(*st)
    o.step(25)
    ref = o.state()
    same(run(c, 25, st), ref)
    same(run(c, 25, st, block=64), ref)


@pytest.mark.parametrize("name,steps", [("c1var", 30), ("delaunay4k", 40), ("delaunay4k_nolim", 40), ("storm3k", 30),
                                        ("tipot2k", 20), ("c1fseries", 20)])
def test_split_equals_one_lane(name, steps):
    c = load_case(name)
    same(run(c, steps), run(c, steps, block=128))


@pytest.mark.parametrize("p", [1, 2])
def test_three_stage_scheme_with_kept_rhs(p):
    c = mesh.structured_basin(nx=20, ny=9, dx=500.0, dy=500.0, depth=6.0, amp=0.4, manning=None, p=p, dt=4.0, rk_stage=3,
                              slopeflag=0, nolifa=2, nolibf=0, cori=1.0e-4, flow_side=True, flow_amp=1.0)
    same(run(c, 40), run(c, 40, block=64))


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("depth", [2.0 ** -510, 0.0, -0.5])
def test_depths_outside_the_short_flux(p, depth):
    """Elements whose depth is below 2^-500, zero or negative at their vertices take the general flux.  The
    oracle's wave-speed bound keeps the NaN of a negative depth's square root where the device's maximum
    drops it, so the oracle's finite values are compared; the two forms agree everywhere."""
    c = closed(6, 5, p)
    ze, qx, qy, wd = adjoint.hump_state(c, amplitude=0.2, width=0.3)
    qx[:, 0] = 0.01
    low = np.arange(c.ne) % 7 == 3
    ze[low, 0] = -10.0
    c.dp = np.full(c.np_, 10.0)
    if depth == 2.0 ** -510:
        c.dp = np.where(np.isin(np.arange(1, c.np_ + 1), c.nm[low]), 0.0, c.dp)
        ze[low, 0] = depth
        c.params.h0 = 0.0
    else:
        ze[low, 0] = depth - 10.0
    o = Oracle(c, threads=1)
    o.set_state(ze, qx, qy, wd)
    o.step(1)
    ref = o.state()
    one = run(c, 1, (ze, qx, qy, wd), 64)
    same(run(c, 1, (ze, qx, qy, wd)), one)
    for x, y in zip(one, ref):
        ok = ~np.isnan(y)
        assert ok.any() or depth == 0.0
        np.testing.assert_array_equal(x[ok], y[ok])


def fan(k, p):
    """A closed disc of k sectors and three rings around one node: the centre node belongs to k elements (the
    limiter's node lists hold eight per entry)."""
    rings = 3
    r = np.concatenate([[0.0], np.repeat(np.arange(1, rings + 1) * 1000.0, k)])
    t = np.concatenate([[0.0], np.tile(np.arange(k) * 2.0 * np.pi / k, rings)])
    nid = lambda i, j: 2 + (i - 1) * k + j % k
    nm = [(1, nid(1, j), nid(1, j + 1)) for j in range(k)]
    for i in range(1, rings):
        for j in range(k):
            nm += [(nid(i, j), nid(i + 1, j), nid(i + 1, j + 1)), (nid(i, j), nid(i + 1, j + 1), nid(i, j + 1))]
    c = closed(1, 1, p, nolifa=2, slopeflag=5)
    c.x, c.y = r * np.cos(t), r * np.sin(t)
    c.nm = np.array(nm, dtype=np.int32)
    n = len(c.x)
    c.slam, c.sfea, c.sfac, c.corif = c.x / 6378206.4, c.y / 6378206.4, np.ones(n), np.zeros(n)
    c.dp = 3.0 - 0.0015 * c.x
    c.land_segs = [(0, np.array([nid(rings, j) for j in range(k + 1)], dtype=np.int32))]
    c.params.dtdp = 0.5
    return c


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("k", [5, 8, 9, 17])
def test_limiter_nodes_of_many_elements(k, p):
    c = fan(k, p)
    rng = np.random.default_rng(k)
    ze, qx, qy, wd = wetdry_state(c, 1.0)
    wet = wd == 1
    ze[wet, 1:3] += rng.uniform(-0.3, 0.3, (wet.sum(), 2))
    qx[wet, :3] += rng.uniform(-1.0, 1.0, (wet.sum(), 3))
    o = Oracle(c, threads=1)
    o.set_state(ze, qx, qy, wd)
    o.step(20)
    same(run(c, 20, (ze, qx, qy, wd)), o.state())
