"""Line tiles of the FFT form at the edges of their length classes, and p0 formed
on the fly against p0 formed by the pass over the state.

Tolerance of the fields after two steps, rel-L2 against the FP64 oracle: 2e-6,
as in test_gpu_parity.py (FP32 roundings of one derivative are a few 1e-7 of its
largest value, the twelve stages of two steps add up at random).
"""
import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W
from oracle import binding as ob

from test_gpu_parity import THREADS, compare_fields, device

pytestmark = pytest.mark.gpu


def scene(nx, ny, patch, steps=2):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, steps)
    conf.Settings.SetPatchError(patch)
    conf.Domains = [W.domain(0, 0, nx, ny, {"T": 1.0, "L": 0.4, "B": 0.7, "R": 1.0})]
    conf.Speakers = [(W._world_pos(nx / 2 + 0.5), W._world_pos(ny / 2 + 0.5), 0.0),
                     (W._world_pos(nx - 3.5), W._world_pos(2.5), 0.0)]  # into the halos of two edges
    conf.Receivers = [(W._world_pos(nx / 2 + 2.25), W._world_pos(ny / 2 + 1.25), 0.0)]
    return conf


# the shortest and the longest line of every FFT length (a line of n cells has n
# and n + 1 values and two windows of w), the other side odd: a lone last line
@pytest.mark.parametrize("patch, n", [
    (70.0, 65), (70.0, 191), (70.0, 193), (70.0, 447), (70.0, 449), (70.0, 959), (70.0, 961), (70.0, 1983),
    (70.0, 1985), (70.0, 4031), (70.0, 4033), (50.0, 67), (50.0, 91), (50.0, 93), (60.0, 203), (60.0, 205)])
@pytest.mark.parametrize("across", [False, True])
def test_line_length_edges(patch, n, across):
    conf = scene(*((67, n) if across else (n, 67)), patch)
    k, dev = device(conf)
    dev.advance(2)
    o = ob.OracleScene(conf, 64, THREADS)
    o.step(2)
    compare_fields(k, dev, o, 2e-6)


@pytest.mark.parametrize("nx, ny, copies", [(301, 217, 2), (1250, 77, 12), (77, 1250, 12), (2100, 66, 8)])
def test_p0_on_the_fly_is_bitwise_the_pass(nx, ny, copies):
    """Small plans add px and py of the two layouts where a tile reads them, large
    ones form p0 in a pass after every stage (by the bytes the two move; a plan's
    share of lines above 1024 points decides how large): the same scene alone and
    in a batch, fields and series bitwise equal, also after a host write and with
    spectral receivers between the cells."""
    confs = [scene(nx, ny, 70.0, 60) for _ in range(copies)]
    batch = P.BatchSolver(confs)
    k, dev = device(confs[0])
    assert np.array_equal(batch.scene_samples(batch.advance(23), copies - 1), dev.advance(23))
    p = dev.field(0, "p0") * np.float32(0.5)
    for s in range(copies):
        batch.set_field(s, 0, "p0", p)
    dev.set_field(0, "p0", p)
    vy = dev.field(0, "vy0")[::-1].copy()
    for s in range(copies):
        batch.set_field(s, 0, "vy0", vy)
    dev.set_field(0, "vy0", vy)
    assert np.array_equal(dev.field(0, "vy0"), vy)
    assert np.array_equal(batch.scene_samples(batch.advance(22), copies - 1), dev.advance(22))
    for f in ("p0", "px0", "py0", "vx0", "vy0"):
        for d in range(k.domain_count()):
            assert np.array_equal(batch.field(copies - 1, d, f), dev.field(d, f)), (f, d)


@pytest.mark.parametrize("nx, ny, n", [(600, 700, 3), (1100, 300, 3), (90, 1300, 4), (447, 959, 4)])
def test_values_per_thread_are_bitwise_neutral(nx, ny, n):
    """1024- and 2048-point lines take 8 values per thread in a scene of few
    wavefronts and 16 in a batch of many: the same bits."""
    conf = P.PSTDConfiguration()
    W.base_settings(conf, 5)
    conf.Domains = [W.domain(0, 0, nx, ny, 0.9)]
    conf.Speakers = [(W._world_pos(nx / 3), W._world_pos(ny / 2), 0.0)]
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    one = k.prepare()
    batch = P.BatchSolver([conf] * n)
    one.advance(5)
    batch.advance(5)
    for d in range(k.domain_count()):
        for f in ("p0", "px0", "py0", "vx0", "vy0"):
            want = one.field(d, f)
            for i in range(n):
                assert np.array_equal(batch.field(i, d, f), want), (i, d, f)
