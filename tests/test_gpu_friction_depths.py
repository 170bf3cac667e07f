"""The device's DEPTH**(1/3): one forward Euler step of elements of uniform depth, drawn over every exponent class
of the reduction in dg_crmath.hpp, with Manning friction, against the oracle's C library bit for bit.  Elements whose
depth the C library itself does not round correctly (a fraction of a percent) are left out."""
import math

import numpy as np
import pytest

from dgswem_amd import gpu
from oracle.oracle import Oracle
from test_crmath_cpu import exact_pow3
from test_gpu_edge_cases import closed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("block", [None, 64, 128])
def test_depths_of_every_class(p, block):
    c = closed(25, 20, p)
    c.dg.rk_stage = c.dg.rk_order = 1
    c.dp = np.full(c.np_, 1.0)                   # the bathymetry's mean is 1 and its slope 0 exactly
    c.manning = np.full(c.np_, 0.03)
    c.params.cf = 1.0e-6                         # under the Manning friction of every depth
    c.params.dtdp = 0.01
    rng = np.random.default_rng(5 + p)
    n, dof = c.ne, 3 if p == 1 else 6
    ze, qx, qy = np.zeros((n, dof)), np.zeros((n, dof)), np.zeros((n, dof))
    ze[:, 0] = 2.0 ** rng.uniform(-6.0, 13.0, n) - 1.0
    depth = ze[:, 0] + 1.0
    qx[:, 0], qy[:, 0] = depth * rng.uniform(-0.5, 0.5, n), depth * rng.uniform(-0.5, 0.5, n)
    wd = np.ones(n, np.int32)
    o = Oracle(c, threads=2)
    o.set_state(ze, qx, qy, wd)
    o.step(1)
    g = gpu.GpuSolver(c)
    if block:
        g.set_block(block)
    g.set_state(ze, qx, qy, wd)
    g.step(1)
    ok = np.array([math.pow(d, 1.0 / 3.0) == exact_pow3(d) for d in depth])
    assert ok.mean() > 0.98
    for a, b in zip(g.state()[:3], o.state()[:3]):
        np.testing.assert_array_equal(a[ok], b[ok])
    g.close()
