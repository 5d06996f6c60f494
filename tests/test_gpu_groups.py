"""Large batches run as two instance groups on two streams (tm_groups.h): fields,
rho(t) rows and the reported fault are those of the same instances in a batch too
small to be grouped, bit for bit (the groups change where launches run, not what
they compute), also while another context's run takes the streams away."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDES = [97, 33, 64, 129]            # 16 of each: 499760 cells, every model's batch is grouped
PICK = [0, 1, 30, 31, 32, 33, 63]    # around the cut, the first and the last (56 thousand cells)

CASES = {
    "dp_f64": ("MODEL_DP", "F64", lambda tm: tm.DPParams(), [1.0]),
    "dp_f32": ("MODEL_DP", "F32", lambda tm: tm.DPParams(), [1.0]),
    "rk_f64": ("MODEL_RIETKERK", "F64", lambda tm: tm.RietkerkParams(), [4.0, 8.0, 10.0]),
    "rk_f32": ("MODEL_RIETKERK", "F32", lambda tm: tm.RietkerkParams(), [4.0, 8.0, 10.0]),
    "dp2": ("MODEL_DP2", "F64", lambda tm: tm.DPCParams(a=1e-5), [20.0, 2.0, 0.0]),
    "dp3": ("MODEL_DP3", "F64", lambda tm: tm.DPCParams(a=1e-5), [20.0, 2.0, 0.5, 0.0, 0.0]),
    "fke2": ("MODEL_FKE2", "F64", lambda tm: tm.FKEParams(), [20.0, 2.0, 8.0, 10.0, 0.0]),
    "fke3": ("MODEL_FKE3", "F64", lambda tm: tm.FKEParams(), [20.0, 2.0, 0.5, 8.0, 10.0, 0.0, 0.0]),
}


def _instances(tm):
    return [tm.Instance(SIDES[k % 4], 0, 5, k) for k in range(64)]


def _open(tm, name, insts, like=None):
    model, prec, params, hi = CASES[name]
    ctx = tm.Context()
    ctx.configure(getattr(tm, model), getattr(tm, prec), params(tm), insts)
    # blocks of 4 steps: each run forks and joins the groups several times
    ctx.set_launch(ctx.launch()[0] if like is None else like, 4)
    ctx.init_uniform([0.0] * len(hi), hi)
    return ctx


@pytest.mark.parametrize("name", list(CASES))
def test_groups_equal_one_group(tm, name):
    insts = _instances(tm)
    print(f"groups {name}", flush=True)
    with _open(tm, name, insts) as ctx:
        variant = ctx.launch()[0]
        rows = [ctx.run(11), ctx.run(2)]
        big = [(ctx.download(k), rows[0][k], rows[1][k]) for k in PICK]
    with _open(tm, name, [insts[k] for k in PICK], variant) as ctx:
        rows = [ctx.run(11), ctx.run(2)]
        small = [(ctx.download(j), rows[0][j], rows[1][j]) for j in range(len(PICK))]
    for b, s in zip(big, small):
        for x, y in zip(b, s):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("name", ["dp_f64", "dp_f32"])
def test_groups_report_the_first_fault(tm, oracle, name):
    """100 and its neighbours' share of it turn negative under the explicit Euler step; the
    first such cell of the smallest instance is reported, whichever group it is in."""
    insts = _instances(tm)
    for plant in ([63], [63, 33], [63, 2], [2]):
        with _open(tm, name, insts) as ctx:
            for k in range(64):
                f = np.zeros((1, insts[k].L, insts[k].L))
                if k in plant:
                    f[0, 5, 7] = 100.0
                ctx.upload(k, f)
            with pytest.raises(tm.NumericFault):
                ctx.run(1)
            first = insts[min(plant)]
            f = np.zeros((1, first.L, first.L))
            f[0, 5, 7] = 100.0
            ref = oracle.dp_run(oracle.dp_params(), f, first.L, first.seed, first.instance_id, 0, 1)
            assert ctx.fault_info() == (min(plant), ref["fault_cell"], 0)


def test_groups_beside_other_runs(tm):
    insts = _instances(tm)
    names = ["dp2", "rk_f64", "dp_f64"]
    alone, beside = {}, {}
    for name in names:
        with _open(tm, name, insts) as ctx:
            alone[name] = (ctx.run(40), ctx.download(63))
    ctxs = {name: _open(tm, name, insts) for name in names}

    def work(name):
        beside[name] = (ctxs[name].run(40), ctxs[name].download(63))

    threads = [threading.Thread(target=work, args=(n,)) for n in names]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for ctx in ctxs.values():
        ctx.close()
    for name in names:
        for x, y in zip(alone[name], beside[name]):
            assert np.array_equal(x, y)
