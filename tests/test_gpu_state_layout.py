"""Setting and reading back the state: every value's bits and every flag, around the sizes of a thread block."""
import numpy as np
import pytest

from dgswem_amd import gpu
from test_gpu_edge_cases import closed

pytestmark = pytest.mark.gpu


# 2 elements; under, at and over 256 values a field (p=1: 86 elements, p=2: 43) and 256 flags
@pytest.mark.parametrize("nx,ny", [(1, 1), (7, 3), (11, 2), (43, 1), (16, 8), (43, 3)])
@pytest.mark.parametrize("p", [1, 2])
def test_round_trip(nx, ny, p):
    c = closed(nx, ny, p, nolifa=2)
    g = gpu.GpuSolver(c)
    n, dof = 2 * nx * ny, 3 if p == 1 else 6
    rng = np.random.default_rng(nx * 100 + ny)
    st = [rng.standard_normal((n, dof)) for _ in range(3)]
    st[0][0, 0], st[1][-1, -1], st[2][n // 2, 1] = -0.0, np.nan, np.inf
    wd = rng.integers(0, 2, n).astype(np.int32)
    g.set_state(*st, wd)
    g.step(0)
    out = g.state()
    for a, b in zip(out[:3], st):
        np.testing.assert_array_equal(np.asarray(a).reshape(n, dof).view(np.int64), b.view(np.int64))
    np.testing.assert_array_equal(out[3], wd)
    g.set_state(*st[::-1])                                   # without flags: they stay
    out = g.state()
    for a, b in zip(out[:3], st[::-1]):
        np.testing.assert_array_equal(np.asarray(a).reshape(n, dof).view(np.int64), b.view(np.int64))
    np.testing.assert_array_equal(out[3], wd)
    g.close()


# just under and over the size from which the state is read back in chunks (6 MiB), and more chunks than there are
# slots for them; the elements of one size also by two threads at once, each with its own solver
@pytest.mark.parametrize("nx,p", [(4139, 1), (4140, 1), (2125, 2), (2126, 2), (5000, 2)])
def test_large_round_trip(nx, p):
    from concurrent.futures import ThreadPoolExecutor
    c = closed(nx, 10, p, nolifa=2)
    n, dof = 20 * nx, 3 if p == 1 else 6

    def trip(seed):
        g = gpu.GpuSolver(c)
        rng = np.random.default_rng(seed)
        for _ in range(2):
            st = [rng.standard_normal((n, dof)) for _ in range(3)]
            wd = rng.integers(0, 2, n).astype(np.int32)
            g.set_state(*st, wd)
            for a, b in zip(g.state(), st + [wd]):
                np.testing.assert_array_equal(np.asarray(a).reshape(b.shape), b)
        g.close()

    trip(1)
    if nx == 5000:
        with ThreadPoolExecutor(2) as ex:
            list(ex.map(trip, (2, 3)))
