"""modal2nodal's rows of incident elements around the size of one group of loads (six at p=1, four at p=2) and of two,
with dry elements in them, and mesh sizes around a block of 64 nodes; against the oracle, bit for bit."""
import numpy as np
import pytest

from dgswem_amd import gpu
from oracle.oracle import Oracle
from test_gpu_edge_cases import closed, wetdry_state
from test_gpu_stage_shapes import fan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4, 5, 6, 7, 8, 9, 12, 13, "21x2", "20x2"])
@pytest.mark.parametrize("p", [1, 2])
def test_rows_of_incident_elements(k, p):
    if isinstance(k, str):                       # 22*3 and 21*3 nodes: over and under 64
        nx, ny = map(int, k.split("x"))
        c = closed(nx, ny, p, nolifa=2)
        c.dp = 2.0 - 2.5 * c.x / c.x.max()
    else:
        c = fan(k, p)
    st = wetdry_state(c, 1.0)
    assert (st[3] == 0).any() and (st[3] == 1).any()
    g, o = gpu.GpuSolver(c), Oracle(c, threads=1)
    em = np.full(c.np_, -99999.0)
    g.set_etamax(em)
    o.set_etamax(em)
    g.set_state(*st)
    o.set_state(*st)
    g.nodal_update()
    ref = o.nodal()
    out = g.get_nodal()
    for a, b in zip(out[:3], ref):
        np.testing.assert_array_equal(a, b)
    # the oracle sets NODECODE in its steps only: nodes with a wet element
    wet = np.zeros(c.np_, np.int32)
    wet[(c.nm[st[3] == 1] - 1).ravel()] = 1
    np.testing.assert_array_equal(out[3], wet)
    np.testing.assert_array_equal(out[4], o.etamax())
    g.close()
