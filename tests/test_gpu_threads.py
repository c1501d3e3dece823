"""One solver used from several threads: calls take turns, so what a thread reads is
the state after a whole number of steps, and reading disturbs no step.  Sizes on
both sides of 256 KiB, up to which reads pass through pinned memory."""
import threading

import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W

pytestmark = pytest.mark.gpu
FIELDS = ("p0", "px0", "py0", "vx0", "vy0")


def solver(nx, ny, form):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, 100)
    conf.Domains = [W.domain(0, 0, nx, ny, 1.0)]
    conf.Speakers = [(W._world_pos(nx / 3), W._world_pos(ny / 2), 0.0)]
    conf.Receivers = [(W._world_pos(x + 0.25), W._world_pos(ny / 2 + 0.25), 0.0) for x in (3, nx // 2, nx - 2)]
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    k.set_form(form)
    return k, k.prepare()


@pytest.mark.parametrize("nx, ny, form, per_call", [
    (40, 41, "fft", 1), (255, 256, "fft", 2), (300, 219, "fft", 1), (1300, 1001, "fft", 21), (256, 300, "gemm_f16", 1)])
def test_reads_from_other_threads_see_whole_steps(nx, ny, form, per_call):
    calls = 24
    k, ref = solver(nx, ny, form)
    ref.advance(1)
    states, series = [{f: ref.field(0, f) for f in FIELDS}], []
    for _ in range(calls):
        series.append(ref.advance(per_call))
        states.append({f: ref.field(0, f) for f in FIELDS})
    _, dev = solver(nx, ny, form)
    dev.advance(1)
    done = threading.Event()
    reads = {f: [] for f in FIELDS}
    failed = []

    def read(f):
        try:
            while not done.is_set() and len(reads[f]) < 60:
                reads[f].append(dev.field(0, f))
            reads[f].append(dev.field(0, f))
        except Exception as e:  # noqa: BLE001 (a thread's exception is the test's)
            failed.append(e)

    threads = [threading.Thread(target=read, args=(f,)) for f in FIELDS]
    for t in threads:
        t.start()
    got = [dev.advance(per_call) for _ in range(calls)]
    done.set()
    for t in threads:
        t.join()
    assert not failed, failed
    for n in range(calls):
        assert np.array_equal(got[n], series[n]), n
    for f in FIELDS:
        at = 0
        for values in reads[f]:  # (the states in their order)
            while at <= calls and not np.array_equal(values, states[at][f]):
                at += 1
            assert at <= calls, f
        assert np.array_equal(dev.field(0, f), states[calls][f]), f
