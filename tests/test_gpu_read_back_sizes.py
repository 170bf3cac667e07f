"""Results read back through page-locked chunks around the size from which there are more of them (16 MiB), and a handle
whose results fall on both sides of it in turn."""
import numpy as np
import pytest

from dgswem_amd import gpu
from test_gpu_edge_cases import closed

pytestmark = pytest.mark.gpu


def random_state(n, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((n, 3)) for _ in range(3)] + [rng.integers(0, 2, n).astype(np.int32)]


@pytest.mark.parametrize("nx", [11037, 11038])       # 76 bytes an element: just under and over
def test_around_the_larger_size(nx):
    c = closed(nx, 10, 1, nolifa=2)
    g = gpu.GpuSolver(c)
    for seed in (1, 2):
        st = random_state(c.ne, seed)
        g.set_state(*st)
        for a, b in zip(g.state(), st):
            np.testing.assert_array_equal(a, b)
    g.close()


def test_smaller_and_larger_results_in_turn():
    c = closed(500, 500, 1, nolifa=2)                # nodal values 7 MB, state 38 MB
    g, h = gpu.GpuSolver(c), gpu.GpuSolver(c)
    st = random_state(c.ne, 3)
    st[0][:, 0] += 20.0
    for s in (g, h):
        s.set_state(*st)
    ref = g.nodal()
    for a, b in zip(h.state(), st):                  # the other handle starts with the larger one
        np.testing.assert_array_equal(a, b)
    for s in (g, h, g):
        for a, b in zip(s.state(), st):
            np.testing.assert_array_equal(a, b)
        for a, b in zip(s.nodal(), ref):
            np.testing.assert_array_equal(a, b)
    g.close()
    h.close()
