"""Small states travel in one copy, larger ones in a copy per array, the smallest set without flags without a kernel:
bits and flags around the sizes where the way changes (1 MiB, 256 KiB), and subsets of the arrays."""
import ctypes as C

import numpy as np
import pytest

from dgswem_amd import gpu
from test_gpu_edge_cases import closed

pytestmark = pytest.mark.gpu


def random_state(n, dof, seed):
    rng = np.random.default_rng(seed)
    st = [rng.standard_normal((n, dof)) for _ in range(3)]
    st[0][0, 0], st[1][-1, -1], st[2][n // 2, 1] = -0.0, np.nan, np.inf
    return st, rng.integers(0, 2, n).astype(np.int32)


def bits(a, b):
    np.testing.assert_array_equal(np.asarray(a).reshape(b.shape).view(np.int64), b.view(np.int64))


# bytes an element: p=1 72 and 76, p=2 144 and 148 without and with the flags
@pytest.mark.parametrize("p,n", [(1, 3640), (1, 3642), (1, 13796), (1, 13798), (2, 1820), (2, 1822), (2, 7084), (2, 7086)])
def test_round_trips(p, n):
    c = closed(n // 2, 1, p, nolifa=2)
    assert c.ne == n
    dof = 3 if p == 1 else 6
    g = gpu.GpuSolver(c)
    a, wa = random_state(n, dof, 1)
    b, wb = random_state(n, dof, 2)
    g.set_state(*a, wa)
    out = g.state()
    for x, y in zip(out[:3], a):
        bits(x, y)
    np.testing.assert_array_equal(out[3], wa)
    g.set_state(*b)                                          # the flags stay
    out = g.state()
    for x, y in zip(out[:3], b):
        bits(x, y)
    np.testing.assert_array_equal(out[3], wa)
    g.set_state(*a, wb)
    np.testing.assert_array_equal(g.state()[3], wb)
    g.close()


@pytest.mark.parametrize("n", [58, 20000])
def test_subsets_of_the_arrays(n):
    """dg_gpu_get_state writes the arrays that are given and no others."""
    c = closed(n // 2, 1, 1, nolifa=2)
    g = gpu.GpuSolver(c)
    st, wd = random_state(n, 3, 5)
    g.set_state(*st, wd)
    L = gpu.load_library()
    get = C.CFUNCTYPE(C.c_int, C.c_int, *[C.c_void_p] * 4)(("dg_gpu_get_state", L))
    for mask in range(16):
        arrays = [np.full((n, 3), 7.0) for _ in range(3)] + [np.full(n, 7, np.int32)]
        assert get(g.h, *[a.ctypes.data if mask >> i & 1 else None for i, a in enumerate(arrays)]) == 0
        for i, (a, ref) in enumerate(zip(arrays, st + [wd])):
            if mask >> i & 1:
                np.testing.assert_array_equal(a, ref)
            else:
                assert (a == 7).all()
    g.close()


def test_a_small_read_takes_one_copy():
    """Reading 1,600 elements with their flags against the mass, which is one copy of a few KB: half as long again; with a copy per
    array it took three times as long."""
    import time
    c = closed(40, 20, 1, nolifa=2)
    g = gpu.GpuSolver(c)
    g.step(1)

    def median(f):
        ts = []
        for _ in range(300):
            t = time.perf_counter()
            f()
            ts.append(time.perf_counter() - t)
        return 1e6 * np.median(ts)

    state, mass = median(g.state), median(g.mass)
    print(f"state {state:.1f} us, mass {mass:.1f} us", flush=True)
    assert state < 2.3 * mass
    g.close()
