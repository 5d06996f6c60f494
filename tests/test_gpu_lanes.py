"""Runs long enough for two instance groups on two streams (tm_groups.h): fields, rho(t)
rows and the reported fault are those of the same instances in a batch too small to be
grouped, bit for bit, in blocks of any length."""
import numpy as np
import pytest

from tests.test_gpu_groups import CASES, PICK, _instances, _open

pytestmark = pytest.mark.gpu

# 499760 cells: steps from which a run of each model is grouped, and a few more
STEPS = {"dp_f64": 22, "dp_f32": 125, "rk_f64": 25, "rk_f32": 57, "dp2": 11, "dp3": 9, "fke2": 10, "fke3": 9}


@pytest.fixture(scope="module", autouse=True)
def lanes(tm):
    """A context whose runs have been long enough for the device's lanes to be made."""
    with _open(tm, "dp2", _instances(tm)) as ctx:
        ctx.set_launch(-1, 100)
        ctx.run(2500, rows=False)
        yield ctx


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("block", [4, 100])
def test_long_runs_equal_one_group(tm, name, block):
    insts, n = _instances(tm), STEPS[name]
    print(f"lanes {name} blocks of {block}", flush=True)
    with _open(tm, name, insts) as ctx:
        variant = ctx.launch()[0]
        ctx.set_launch(variant, block)
        rows = [ctx.run(n), ctx.run(1), ctx.run(n)]   # a short run between two grouped ones
        big = [(ctx.download(k), *[r[k] for r in rows]) for k in PICK]
    with _open(tm, name, [insts[k] for k in PICK], variant) as ctx:
        rows = [ctx.run(n), ctx.run(1), ctx.run(n)]
        small = [(ctx.download(j), *[r[j] for r in rows]) for j in range(len(PICK))]
    for b, s in zip(big, small):
        for x, y in zip(b, s):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("name", ["dp_f64", "dp_f32"])
def test_long_runs_report_the_first_fault(tm, oracle, name):
    """As test_groups_report_the_first_fault, over a whole grouped run."""
    insts = _instances(tm)
    for plant in ([63], [63, 33], [63, 2], [2]):
        with _open(tm, name, insts) as ctx:
            for k in range(64):
                f = np.zeros((1, insts[k].L, insts[k].L))
                if k in plant:
                    f[0, 5, 7] = 100.0
                ctx.upload(k, f)
            with pytest.raises(tm.NumericFault):
                ctx.run(STEPS[name])
            first = insts[min(plant)]
            f = np.zeros((1, first.L, first.L))
            f[0, 5, 7] = 100.0
            ref = oracle.dp_run(oracle.dp_params(), f, first.L, first.seed, first.instance_id, 0, 1)
            assert ctx.fault_info() == (min(plant), ref["fault_cell"], 0)
