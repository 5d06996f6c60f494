"""Contexts that come and go in several threads, with large batches and without, share the
device's lanes (tm_groups.h) and its download staging (tm_hostcopy.h): every life's rows and
fields are those of the same batch alone."""
import threading

import numpy as np
import pytest

from tests.test_gpu_groups import _instances, _open

pytestmark = pytest.mark.gpu


def _life(tm, name, steps):
    with _open(tm, name, _instances(tm)) as ctx:
        ctx.set_launch(-1, 100)
        rows = [ctx.run(n) for n in steps]
        return [*rows, ctx.download(63), ctx.download(0)]


def _small(tm):
    with tm.Context() as ctx:
        ctx.configure(tm.MODEL_DP, tm.F64, tm.DPParams(), [tm.Instance(600, 0, 2, 0)])
        ctx.init_uniform([0.0], [1.0])
        return [ctx.run(3), ctx.download(0)]


def test_lives_in_several_threads(tm):
    names, steps = ["dp2", "rk_f64", "dp_f64"], (30, 2)
    want = {n: _life(tm, n, steps) for n in names}
    small = _small(tm)
    bad = []

    def work(k):
        try:
            for life in range(4):
                n = names[(k + life) % len(names)]
                got = _life(tm, n, steps) if (k + life) % 4 else _small(tm)
                ref = want[n] if (k + life) % 4 else small
                if not all(np.array_equal(a, b) for a, b in zip(got, ref)):
                    bad.append((k, life, n))
        except Exception as e:   # a thread's exception would not fail the test
            bad.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    assert all(np.array_equal(a, b) for a, b in zip(_life(tm, "dp2", steps), want["dp2"]))
