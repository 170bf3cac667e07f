"""The slope limiter's form for large meshes (a wave per tile): against the oracle bit for bit, and batches that take it
against single runs that are small enough for the other form.  With wetting and drying it runs from 250,000 elements
(p=1) or 90,000 (p=2) on, without from 750,000 or 550,000.

The mesh of the first test is a closed basin with a dry coast whose elements are numbered at random, so that every tile
of 64 has hundreds of halo elements and nodes, with a disc beside it whose centre belongs to 17 elements (the node
lists hold eight per entry)."""
import copy

import numpy as np
import pytest

from dgswem_amd import adjoint, gpu, mesh
from oracle.oracle import Oracle
from test_gpu_edge_cases import closed, wetdry_state
from test_gpu_stage_shapes import fan, same

pytestmark = pytest.mark.gpu


def basin_with_disc(nx, ny, p, nolifa):
    c = closed(nx, ny, p, nolifa=nolifa, slopeflag=5)
    c.dp = 6.0 - 6.5 * c.x / c.x.max()                      # dry in the east
    if nolifa < 2:
        c.dp = 6.0 - 4.0 * c.x / c.x.max()                  # all wet without wetting and drying
    d = fan(17, p)
    n = c.np_
    ring = (0, d.land_segs[0][1] + n)
    nm = np.concatenate([c.nm, d.nm + n])
    rng = np.random.default_rng(3)
    nm = nm[rng.permutation(len(nm))]
    c = copy.deepcopy(c)
    c.x, c.y = np.concatenate([c.x, d.x - 20000.0]), np.concatenate([c.y, d.y])
    c.dp = np.concatenate([c.dp, np.full(d.np_, 4.0)])
    c.nm = np.ascontiguousarray(nm.astype(np.int32))
    m = c.np_
    c.slam, c.sfea, c.sfac, c.corif = c.x / 6378206.4, c.y / 6378206.4, np.ones(m), np.zeros(m)
    c.land_segs = [c.land_segs[0], (ring[0], ring[1].astype(np.int32))]
    c.params.dtdp = 0.5
    return c


@pytest.mark.parametrize("p,nolifa,nx,ny", [(1, 2, 500, 250), (2, 2, 300, 151), (1, 1, 1000, 375), (2, 1, 1000, 275)])
def test_against_the_oracle(p, nolifa, nx, ny):
    c = basin_with_disc(nx, ny, p, nolifa)
    assert c.ne % 64 != 0
    ze, qx, qy, wd = wetdry_state(c, 0.5)
    rng = np.random.default_rng(p)
    deep = c.dp[c.nm - 1].min(axis=1) > 1.5
    ze[deep, 1:3] += rng.uniform(-0.2, 0.2, (deep.sum(), 2))
    qx[deep, :3] += rng.uniform(-0.5, 0.5, (deep.sum(), 3))
    o = Oracle(c, threads=8)
    o.set_state(ze, qx, qy, wd)
    o.step(4)
    ref = o.state()
    assert all(np.isfinite(a).all() for a in ref[:3])
    if nolifa == 2:
        assert 0 < (ref[3] == 0).sum() < c.ne
    g = gpu.GpuSolver(c)
    g.set_state(ze, qx, qy, wd)
    g.step(4)
    same(g.state(), ref)
    g.close()


@pytest.mark.parametrize("p", [1, 2])
def test_batch_equals_its_single_runs(p):
    """Three storm basins with a dry coast, together past the limit and each under it: states and gradients."""
    cs = [mesh.storm_basin(n, seed=60 + k, p=p, depth_range=(2.0, 30.0), cfl=0.25 if p == 1 else 0.12)
          for k, n in enumerate((95000, 85000, 99000) if p == 1 else (50000, 65000, 80000))]
    steps, ng = 4, 5
    singles = [gpu.GpuSolver(c) for c in cs]
    ens = gpu.Ensemble(singles)
    limit = 250_000 if p == 1 else 90_000
    assert ens.ne >= limit > max(c.ne for c in cs)
    gauges = [adjoint.seeded_gauges(c, ng, k) for k, c in enumerate(cs)]
    ens.set_gauges(*(np.concatenate([a[j] + (ens.eoff[k] if j == 0 else 0) for k, a in enumerate(gauges)])
                     for j in range(3)))
    for s in [ens] + singles:
        s.step(20)
    for k, (a, s) in enumerate(zip(ens.split(ens.state()), singles)):
        print(f"member {k}: {cs[k].ne} elements", flush=True)
        same(a, s.state())
    data = np.full((steps, ng * len(cs)), 0.1)
    J, gn, gdp = ens.gradient(data)
    parts = ens.split([gn, gdp], nodes=True)
    for k, s in enumerate(singles):
        s.set_gauges(*gauges[k])
        _, sn, sd = s.gradient(data[:, k * ng:(k + 1) * ng])
        assert np.abs(sd).max() > 0.0
        np.testing.assert_array_equal(parts[k][0], sn)
        np.testing.assert_array_equal(parts[k][1], sd)
        s.close()
    ens.close()
