"""Device memory in which gradients keep the stages of their runs: all handles of a process together hold no more than
a sixteenth of the device's, a run that would exceed it is recomputed from checkpoints to the same bits, and a closed
handle gives its share back."""
import numpy as np
import pytest
import torch

from dgswem_amd import adjoint, gpu, mesh

pytestmark = pytest.mark.gpu


def test_handles_share_the_bound():
    c = mesh.structured_basin(nx=400, ny=250, dx=900.0, dy=1100.0, depth=6.0, amp=0.3, dt=6.0)
    total = torch.cuda.mem_get_info()[1]
    step = 2 * 9 * 8 * c.ne                                  # bytes of a step's two stages
    steps = int(0.55 * (total / 16) / step)                  # two runs together exceed the bound, one does not
    free = lambda: torch.cuda.mem_get_info()[0]
    data = np.full((steps, 4), 0.1)

    def solver():
        g = gpu.GpuSolver(c)
        g.set_gauges(*adjoint.seeded_gauges(c, 4, 1))
        g.step(1)
        return g

    a, b = solver(), solver()
    f0 = free()
    ref = a.gradient(data)
    f1 = free()
    out = b.gradient(data)
    f2 = free()
    print(f"{steps} steps of {c.ne} elements: {(f0 - f1) / 2**30:.2f} GiB, then {(f1 - f2) / 2**30:.2f} GiB more", flush=True)
    assert f0 - f1 >= steps * step
    assert f1 - f2 < steps * step / 4
    a.close()
    again = b.gradient(data)                                 # the first handle's share is free again
    f3 = free()
    assert f2 - f3 < steps * step / 4
    for o in (out, again):
        for x, y in zip(o, ref):
            np.testing.assert_array_equal(x, y)
    d = solver()
    for x, y in zip(d.gradient(data), ref):                  # b holds it now
        np.testing.assert_array_equal(x, y)
    assert f3 - free() < steps * step / 4
    b.close()
    d.close()
    assert free() >= f0 - steps * step / 100
