"""Times of the storm forcing from the kernel profiler: its launches cover several steps, and each timed step counts
as one, as the other kernels' launches of these steps do."""
import pytest

from conftest import load_case
from dgswem_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [1, 4, 7])
@pytest.mark.parametrize("calls", [(30,), (10, 9, 11), (1,) * 30])
def test_met_counts_the_timed_steps(every, calls):
    g = gpu.GpuSolver(load_case("storm3k"))
    g.step(3)
    g.profile(True, every=every)
    for n in calls:
        g.step(n)
    _, ms, met = g.kernel_stats(gpu.K_MET)
    _, _, stage = g.kernel_stats(gpu.K_STAGE)
    timed = len(range(0, 30, every))
    print(f"every {every}, calls {calls}: {met} steps, {ms:.4f} ms", flush=True)
    assert met == timed and stage == 2 * timed and ms > 0.0
    g.autotune()                                   # launches of its own, which belong to no step
    assert g.kernel_stats(gpu.K_MET)[1:] == (ms, met)
    g.close()
