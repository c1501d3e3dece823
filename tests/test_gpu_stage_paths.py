"""Plans that take different paths through a stage give the same bits: p0 formed by a
pass after every stage or where it is read, 8 or 16 values per thread, a scene alone or
in a batch.  Each test asserts from the context which path its solvers take.  Lengths
that the other tests leave out are compared with the FP64 oracle; the tolerance of
fields after two steps is 2e-6 rel-L2, as in test_gpu_parity.py (FP32 roundings of one
derivative are a few 1e-7 of its largest value, twelve stages add up at random)."""
import ctypes as C

import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import abi_types as T
from openpstd_amd import workloads as W
from openpstd_amd._lib import lib
from oracle import binding as ob

from test_gpu_parity import THREADS, compare_fields, device
from test_gpu_plan_checks import Domain, Plan

pytestmark = pytest.mark.gpu
FIELDS = ("p0", "px0", "py0", "vx0", "vy0")


def scene(nx, ny, steps, spectral=False, patch=70.0):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, steps)
    conf.Settings.SetPatchError(patch)
    conf.Domains = [W.domain(0, 0, nx, ny, {"T": 1.0, "L": 0.4, "B": 0.7, "R": 1.0})]
    conf.Speakers = [(W._world_pos(nx / 2 + 0.5), W._world_pos(ny / 2 + 0.5), 0.0),
                     (W._world_pos(nx - 3.5), W._world_pos(2.5), 0.0)]  # into the halos of two edges
    conf.Receivers = [(W._world_pos(nx / 2 + 2.25), W._world_pos(ny / 2 + 1.25), 0.0),
                      (W._world_pos(nx - 2.625), W._world_pos(1.5), 0.0)]
    if spectral:
        conf.receiver_mode = T.PSTD_RECEIVER_SPECTRAL
    return conf


def assert_same_fields(k, dev, batch, s):
    for f in FIELDS:
        for d in range(k.domain_count()):
            assert np.array_equal(batch.field(s, d, f), dev.field(d, f)), (f, d)


# 2048- and 4096-point lines along and across, with 128- and 256-point lines beside them
# (a plan without lines above 1024 points never takes the pass)
@pytest.mark.parametrize("spectral", [False, True])
@pytest.mark.parametrize("nx, ny, copies", [(1250, 77, 30), (77, 1250, 30), (2100, 66, 4), (66, 2101, 4)])
def test_p0_pass_is_bitwise_p0_on_the_fly(nx, ny, copies, spectral):
    conf = scene(nx, ny, 30, spectral)
    k, dev = device(conf)
    batch = P.BatchSolver([conf] * copies)
    assert not dev.tuning()["p0_pass"] and batch.tuning()["p0_pass"]
    last = copies - 1
    got = dev.advance(7)
    assert np.abs(got).max() > 0
    assert np.array_equal(batch.scene_samples(batch.advance(7), last), got)
    # host writes between steps: an explicit p0 (half of what it was) and another vy
    p, vy = dev.field(0, "p0") * np.float32(0.5), dev.field(0, "vy0")[::-1].copy()
    for f, v in (("p0", p), ("vy0", vy)):
        dev.set_field(0, f, v)
        for s in range(copies):
            batch.set_field(s, 0, f, v)
    assert np.array_equal(batch.scene_samples(batch.advance(23), last), dev.advance(23))
    assert_same_fields(k, dev, batch, last)


# the shortest and the longest lines of 1024 and 2048 points along and across, the other
# side odd (a lone last line)
@pytest.mark.parametrize("across", [False, True])
@pytest.mark.parametrize("n", [449, 959, 961, 1983])
def test_eight_and_sixteen_values_are_bitwise_equal(n, across):
    conf = scene(*((67, n) if across else (n, 67)), 2)
    k, dev = device(conf)
    copies = 6
    batch = P.BatchSolver([conf] * copies)
    assert dev.tuning()["eight_value_points"] == 2048 and batch.tuning()["eight_value_points"] == 512
    assert np.array_equal(batch.scene_samples(batch.advance(2), copies - 1), dev.advance(2))
    assert_same_fields(k, dev, batch, copies - 1)


@pytest.mark.parametrize("patch, n", [(70.0, 33), (50.0, 33), (70.0, 8127)])
@pytest.mark.parametrize("across", [False, True])
def test_shortest_and_longest_lines(patch, n, across):
    """128-point lines barely longer than the window, the longest 8192-point ones."""
    conf = scene(*((67, n) if across else (n, 67)), 2, patch=patch)
    k, dev = device(conf)
    dev.advance(2)
    o = ob.OracleScene(conf, 64, THREADS)
    o.step(2)
    compare_fields(k, dev, o, 2e-6)


@pytest.mark.parametrize("across", [False, True])
def test_8192_point_lines_in_either_order_and_in_a_batch(across):
    conf = scene(*((41, 4100) if across else (4100, 41)), 3)
    k, a = device(conf)
    b = device(conf)[1]
    a.set_tile_order(False)
    b.set_tile_order(True)
    batch = P.BatchSolver([conf, scene(300, 77, 3), conf])
    want = a.advance(3)
    assert np.array_equal(b.advance(3), want)
    assert np.array_equal(batch.scene_samples(batch.advance(3), 2), want)
    for f in FIELDS:
        for d in range(k.domain_count()):
            assert np.array_equal(a.field(d, f), b.field(d, f)), (f, d)
    assert_same_fields(k, a, batch, 2)


def fft_wavefronts(k):
    """Wavefronts of the line tiles of one stage with 16 values per thread from 1024
    points on, counted from the plan's segments (all of them in the FFT form)."""
    total = 0
    for s in k.segments():
        d = k.domain_info(s["domain"])
        n = (d["nx"] if s["direction"] == 0 else d["ny"]) + (1 if s["field"] else 0) + 2 * s["wlen"]
        f = 1 << (n - 1).bit_length()
        if not s["interp_only"]:
            total += (s["line_end"] - s["line_begin"]) // 2 * (f // (8 if f <= 512 else 16)) // 64
    return total


# rigid walls above and below: spectral receivers read lines there that no stage runs,
# which took (1060, 600) and (1300, 530) past the limit
@pytest.mark.parametrize("nx, ny", [(1060, 600), (1300, 530), (1060, 650), (700, 500)])
def test_lines_of_receivers_only_choose_no_values_per_thread(nx, ny):
    points, series = [], []
    for spectral in (False, True):
        conf = scene(nx, ny, 2, spectral)
        conf.Domains = [W.domain(0, 0, nx, ny, {"T": 0.0, "B": 0.0, "L": 1.0, "R": 1.0})]
        k, dev = device(conf)
        assert any(s["interp_only"] for s in k.segments()) == spectral
        points.append(dev.tuning()["eight_value_points"])
        assert points[-1] == (2048 if fft_wavefronts(k) <= 2750 else 512)
        dev.advance(2)
        series.append([dev.field(d, f) for d in range(k.domain_count()) for f in FIELDS])
    assert points[0] == points[1]
    for a, b in zip(*series):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("form", ["gemm_f16", "gemm_bf16"])
def test_lines_of_the_matrix_form_choose_no_values_per_thread(form):
    """A 1024 x 1024 scene in the matrix form: the line tiles are its absorbing layers',
    few wavefronts; the same bits as in a batch, whose layers are many."""
    conf = scene(1024, 1024, 2)
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    k.set_form(form)
    dev = k.prepare()
    batch = P.BatchSolver([conf] * 4, form=form)
    assert dev.tuning()["eight_value_points"] == 2048 and batch.tuning()["eight_value_points"] == 512
    assert np.array_equal(batch.scene_samples(batch.advance(2), 3), dev.advance(2))
    assert_same_fields(k, dev, batch, 3)


def test_flavour_is_the_contexts_own():
    """A flavour chooses nothing and is reported back; one context's does not reach others
    through the launch shapes kept per plan (a plan that is tuned here for the first
    time: no other test has a domain of its size)."""
    ctx = [C.c_void_p(), C.c_void_p()]
    for c in ctx:
        assert lib().pstd_ctx_create(0, C.byref(c)) == T.PSTD_OK
    try:
        dom = (Domain * 1)(Domain(nx=123, ny=71, rho=1.2))
        seg = (T.pstd_plan_segment * 1)()
        for name, v in dict(domain=0, line_end=71, side1=-1, side2=-1, wlen=32, table_len=256, c_main1=1.0,
                            c_main2=1.0).items():
            setattr(seg[0], name, v)
        plan = Plan(n_domains=1, domains=dom, n_segments=1, segments=seg, dx=0.2, dt=1e-4, c1=340.0, patch_error=70.0)
        assert lib().pstd_ctx_set_kernel_flavour(ctx[0], 0) == T.PSTD_OK
        for c, want in zip(ctx, (0, 1)):
            assert lib().pstd_ctx_upload_plan(c, C.byref(plan)) == T.PSTD_OK
            got = C.c_int32(-1)
            assert lib().pstd_ctx_get_tuning(c, C.byref(got), None, None) == T.PSTD_OK
            assert got.value == want
    finally:
        for c in ctx:
            lib().pstd_ctx_destroy(c)
