"""Large transfers of a process that may run on one, two or three CPUs: what comes
back is compared byte for byte, and no upload takes many times what it does with
all CPUs.  (Copy threads that wait for each other's time slices on one CPU took 15
times as long; the runtime's own copy, which one CPU gets, takes 1.4 times, and 3.4
where another process shares that CPU.  Medians of nine, bound by a factor of
eight.)"""
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _allow(cpus):
    for t in os.listdir("/proc/self/task"):
        os.sched_setaffinity(int(t), cpus)


def test_transfers_on_few_cpus():
    from ib3d_amd.native import Solver
    every = os.sched_getaffinity(0)
    if len(every) < 4:
        pytest.skip("needs four CPUs to compare with")
    s = Solver(256, 192, 192)
    try:
        src = np.random.default_rng(2).standard_normal(258 * 194 * 194)
        took = {}
        for k in (len(every), 1, 2, 3):
            _allow(set(sorted(every)[:k]))
            print(f"[gpu] transfers on {k} CPUs", flush=True)
            up, down = [], []
            for q in range(9):
                t0 = time.perf_counter()
                s.upload("u", src)
                t1 = time.perf_counter()
                back = s.download("u")
                t2 = time.perf_counter()
                up.append(t1 - t0)
                down.append(t2 - t1)
                assert back.tobytes() == src.tobytes()
            took[k] = (sorted(up)[4], sorted(down)[4])
        _allow(every)
        print({k: tuple(f"{1e3 * t:.1f} ms" for t in v) for k, v in took.items()}, flush=True)
        for k in (1, 2, 3):
            assert took[k][0] < 8.0 * took[len(every)][0], took
    finally:
        _allow(every)
        s.close()
