"""Pinned memory passes from solvers that are gone to those that read next: more solvers
than are kept, alive together and one after the other, from several threads; each
read is its own solver's."""
import threading

import numpy as np
import pytest

import openpstd_amd as P
from openpstd_amd import workloads as W

pytestmark = pytest.mark.gpu


def solver(n):
    conf = P.PSTDConfiguration()
    W.base_settings(conf, 9)
    conf.Domains = [W.domain(0, 0, 41 + 2 * n, 57, 1.0)]
    conf.Receivers = [(W._world_pos(20.25), W._world_pos(20.25), 0.0)]
    k = P.PSTDKernel(GPU=True)
    k.initialize_kernel(conf)
    return k, k.prepare()


def check(k, dev, seed):
    v = np.random.RandomState(seed).uniform(-1, 1, dev.field(0, "vy0").shape).astype(np.float32)
    dev.set_field(0, "vy0", v)
    assert np.array_equal(dev.field(0, "vy0"), v)
    s = dev.advance(1)
    assert s[0, 0] == dev.field(0, "p0")[20, 20]


def test_reads_of_solvers_alive_together_and_in_turn():
    for round_ in range(2):
        some = [solver(n) for n in range(7)]
        for n, (k, dev) in enumerate(some):
            check(k, dev, 10 * round_ + n)
        for n, (k, dev) in enumerate(reversed(some)):
            check(k, dev, 100 + n)
    failed = []

    def work(n):
        try:
            for i in range(6):
                check(*solver(n), 1000 * n + i)
        except Exception as e:  # noqa: BLE001 (a thread's exception is the test's)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
