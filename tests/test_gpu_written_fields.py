"""vy and py written by the host are turned into the device's layout together, before
the next step or read: what was written comes back, and a step sees it, in whatever
order writes, reads and steps follow each other."""
import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W

pytestmark = pytest.mark.gpu
FIELDS = ("p0", "px0", "py0", "vx0", "vy0")


def solver(sizes, form):
    """One scene per size, as one batch: nine domains each (a room and its absorbing layers)."""
    confs = []
    for nx, ny in sizes:
        c = P.PSTDConfiguration()
        W.base_settings(c, 50)
        c.Domains = [W.domain(0, 0, nx, ny, 1.0)]
        c.Receivers = [(W._world_pos(nx / 2 + 0.25), W._world_pos(ny / 3 + 0.25), 0.0)]
        confs.append(c)
    return P.BatchSolver(confs, form=form)


def domains(b):
    return [(s, d) for s, k in enumerate(b.kernels) for d in range(k.domain_count())]


# 1 to 9 scenes: fewer than 64 fields, and more than two launches' worth; sides
# around the 64 x 64 pieces; a field above 256 KiB
@pytest.mark.parametrize("sizes, form", [
    ([(63, 65)], "fft"), ([(65, 128), (129, 66)], "fft"), ([(41 + 3 * i, 81 - 4 * i) for i in range(9)], "fft"),
    ([(300, 257), (70, 900)], "fft"), ([(256, 256), (256, 127)], "gemm_f16")])
def test_written_fields_reach_reads_and_steps(sizes, form):
    a, b = solver(sizes, form), solver(sizes, form)
    rng = np.random.RandomState(len(sizes))

    def write(names, turned_one_by_one):
        wrote = {}
        for s, d in domains(a):
            for f in names:
                for _ in range(2):  # the second write counts
                    v = rng.uniform(-1, 1, a.kernels[s]._shape(d, f)).astype(np.float32)
                    a.set_field(s, d, f, v)
                    b.set_field(s, d, f, v)
                    if turned_one_by_one:
                        assert np.array_equal(b.field(s, d, f), v), (s, d, f)
                wrote[s, d, f] = v
        return wrote

    def same():
        for s, d in domains(a):
            for f in FIELDS:
                assert np.array_equal(a.field(s, d, f), b.field(s, d, f)), (s, d, f)

    wrote = write(FIELDS, True)
    for (s, d, f), v in reversed(wrote.items()):
        assert np.array_equal(a.field(s, d, f), v), (s, d, f)
    for steps, names in ((1, ("vy0",)), (22, ("py0", "vy0")), (2, ("p0", "py0")), (1, ())):
        write(names, True)
        assert np.array_equal(a.advance(steps), b.advance(steps))
    same()
    write(("vy0", "vx0"), True)
    # (allocation-free advances of the matrix form share an array of the device: one
    # after the other)
    for one in (a, b):
        one.advance_static(1)
        one.synchronize()
    same()
