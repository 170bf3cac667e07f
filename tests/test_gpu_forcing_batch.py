"""The forcing arrays are formed for a batch of steps: many steps in one call (several batches, the last one cut
short), one step per call and replayed graphs (with a remainder) give the same bits."""
import numpy as np
import pytest

from conftest import load_case
from dgswem_amd import gpu, mesh

pytestmark = pytest.mark.gpu


def river():
    return mesh.structured_basin(nx=20, ny=9, dx=500.0, dy=500.0, depth=6.0, amp=0.4, manning=None, p=2, dt=4.0,
                                 rk_stage=3, slopeflag=0, nolifa=2, nolibf=0, flow_side=True, flow_amp=1.0)


# tide, storm, tidal potential, time series of the boundary values, normal flow (three stages)
@pytest.mark.parametrize("name", ["c1var", "storm3k", "tipot2k", "c1fseries", "river"])
@pytest.mark.parametrize("steps", [1, 2, 4, 64, 65, 131])
def test_batches(name, steps):
    c = river() if name == "river" else load_case(name)

    def run(how):
        g = gpu.GpuSolver(c)
        g.use_graph(how == "graph")
        if how == "single":
            for _ in range(steps):
                g.step(1, sync=False)
        else:
            g.step(steps)
        out = g.state()
        g.close()
        return out

    ref = run("single")
    assert np.isfinite(ref[0]).all()
    for how in ("call", "graph"):
        for a, b in zip(run(how), ref):
            np.testing.assert_array_equal(a, b)


# table rows of a call in launch arguments (one launch, several) and over a copy, with several scenarios
@pytest.mark.parametrize("steps", [1, 9, 16, 17, 40])
def test_table_rows_of_an_ensemble(steps):
    cases = [mesh.storm_basin(n, seed=3 + n, p=1, nsteps=200) for n in (400, 700, 500)]
    single = []
    for c in cases:
        g = gpu.GpuSolver(c)
        for _ in range(steps):
            g.step(1, sync=False)
        single.append(g.state())
        g.close()
    for graph in (False, True):
        members = [gpu.GpuSolver(c) for c in cases]
        ens = gpu.Ensemble(members)
        for m in members:
            m.close()
        ens.use_graph(graph)
        ens.step(steps)
        out = ens.state()
        ens.close()
        for k in range(4):
            np.testing.assert_array_equal(out[k], np.concatenate([s[k] for s in single]))
