"""Reads of fields and samples around the size up to which they pass through pinned
memory (256 KiB): what was written comes back, and p0 of the last step is what the
receivers sampled, bit for bit."""
import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, ny", [(40, 41), (255, 256), (256, 256), (257, 256), (300, 219)])
def test_reads_around_the_pinned_size(nx, ny):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, 3)
    conf.Domains = [W.domain(0, 0, nx, ny, 1.0)]
    conf.Speakers = [(W._world_pos(nx / 3), W._world_pos(ny / 2), 0.0)]
    rng = np.random.RandomState(nx)
    cells = [(0, 0), (nx - 1, ny - 1), (nx - 1, 0)] + [(rng.randint(nx), rng.randint(ny)) for _ in range(8)]
    conf.Receivers = [(W._world_pos(x + 0.25), W._world_pos(y + 0.25), 0.0) for x, y in cells]
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    dev = k.prepare()
    wrote = {}
    for name in ("px0", "py0", "vx0", "vy0", "p0"):
        wrote[name] = rng.uniform(-1, 1, dev.field(0, name).shape).astype(np.float32)
        dev.set_field(0, name, wrote[name])
    for name, values in wrote.items():
        assert np.array_equal(dev.field(0, name), values), name
    for steps in (1, 2, 21):
        samples = dev.advance(steps)
        p0 = dev.field(0, "p0")
        assert np.array_equal(samples[-1], [p0[y, x] for x, y in cells])
        assert np.array_equal(p0, dev.field(0, "p0"))
