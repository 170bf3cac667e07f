"""The stage kernel's launch shapes: the block size that the autotuner reports runs the shape that it found."""
import pytest

from dgswem_amd import gpu, mesh

pytestmark = pytest.mark.gpu


def stage_time(g):
    """Microseconds per launch of the stage kernel."""
    g.step(20)
    g.profile(True)
    g.step(100)
    _, ms, n = g.kernel_stats(gpu.K_STAGE)
    g.profile(False)
    return 1.0e3 * ms / n


@pytest.mark.parametrize("p", [1, 2])
def test_reported_block_runs_the_tuned_shape(p):
    """On a small storm basin the shapes differ by a factor of two: a second run that sets the reported block must
    take the tuned run's time, and one to which nothing is said no more."""
    c = mesh.storm_basin(5000, seed=3, p=p)
    g = gpu.GpuSolver(c)
    block = g.autotune()
    tuned = stage_time(g)
    g.close()
    h = gpu.GpuSolver(c)
    h.set_block(block)
    again = stage_time(h)
    h.close()
    d = gpu.GpuSolver(c)
    default = stage_time(d)
    d.close()
    print(f"block {block}: tuned {tuned:.1f} us, set again {again:.1f} us, default {default:.1f} us", flush=True)
    assert again < 1.4 * tuned
    assert default < 1.4 * tuned
