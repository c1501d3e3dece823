"""Reads of fields around the size up to which they pass through pinned memory (1 MiB),
in the FFT form with p0 formed where it is read and in the matrix form, where a pass
forms it: every field as written, and after steps as a second read and the receivers
have it."""
import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W

pytestmark = pytest.mark.gpu
FIELDS = ("p0", "px0", "py0", "vx0", "vy0")


@pytest.mark.parametrize("form", ["fft", "gemm_f16"])
@pytest.mark.parametrize("nx, ny", [(257, 256), (511, 513), (512, 512), (513, 511), (1300, 201), (201, 1310), (600, 601)])
def test_reads_around_the_pinned_size(nx, ny, form):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, 9)
    conf.Domains = [W.domain(0, 0, nx, ny, 1.0)]
    rng = np.random.RandomState(nx)
    cells = [(0, 0), (nx - 1, ny - 1), (nx - 1, 0), (0, ny - 1)] + [(rng.randint(nx), rng.randint(ny)) for _ in range(12)]
    conf.Receivers = [(W._world_pos(x + 0.25), W._world_pos(y + 0.25), 0.0) for x, y in cells]
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    k.set_form(form)
    dev = k.prepare()
    wrote = {f: rng.uniform(-1, 1, dev.field(0, f).shape).astype(np.float32) for f in FIELDS}
    for f, v in wrote.items():
        dev.set_field(0, f, v)
    for f, v in wrote.items():
        assert np.array_equal(dev.field(0, f), v), f
    samples = dev.advance(2)
    p0 = dev.field(0, "p0")
    assert np.array_equal(samples[-1], [p0[y, x] for x, y in cells])
    # the interior is not attenuated: p0 is the sum of the parts that a read returns
    assert np.array_equal(p0, dev.field(0, "px0") + dev.field(0, "py0"))
    vx, vy = dev.field(0, "vx0"), dev.field(0, "vy0")
    dev.set_field(0, "vx0", vx[::-1].copy())
    dev.set_field(0, "vy0", vy[:, ::-1].copy())
    assert np.array_equal(dev.field(0, "vx0"), vx[::-1])
    assert np.array_equal(dev.field(0, "vy0"), vy[:, ::-1])
