"""Output layer with device fields: FRAME text straight from a context, and
snapshots that save, convert and resume a run exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["F64", "F32"])
def test_frame_csv_and_snapshot_round_trip(tm, tmp_path, precision):
    prec = getattr(tm, precision)
    insts = [tm.Instance(48, 0, 2, 7), tm.Instance(33, 0, 2, 8)]
    header = tm.FRAME_HEADER[tm.MODEL_RIETKERK]
    print(f"frame csv + snapshot, {precision}", flush=True)
    with tm.Context() as ctx:
        ctx.configure(tm.MODEL_RIETKERK, prec, tm.RietkerkParams(R=1.1), insts)
        ctx.init_gauss([5.0, 1.0, 1.0], 1)
        ctx.run(4)
        f1 = ctx.download(1)
        ctx.write_frame_csv(1, tmp_path / "dev.csv", 1.1, header)
        ctx.save_snapshot(1, tmp_path / "s.tms")
    tm.format_frame_csv(tmp_path / "host.csv", f1, 1.1, header)
    assert (tmp_path / "dev.csv").read_bytes() == (tmp_path / "host.csv").read_bytes()
    tm.snapshot_to_frame_csv(tmp_path / "s.tms", tmp_path / "conv.csv", 1.1, header)
    assert (tmp_path / "conv.csv").read_bytes() == (tmp_path / "host.csv").read_bytes()
    with tm.Context() as ctx:
        ctx.configure(tm.MODEL_RIETKERK, prec, tm.RietkerkParams(R=1.1), insts)
        assert ctx.load_snapshot(1, tmp_path / "s.tms") == 4
        assert np.array_equal(ctx.download(1), f1)
        with pytest.raises(tm.TMError):
            ctx.load_snapshot(0, tmp_path / "s.tms")          # L = 48 != 33


def test_snapshot_resume_is_exact(tm, tmp_path):
    """Run 6 steps; or run 3, snapshot, load into a fresh context whose instance
    starts at the recorded step, run 3 more: the same fields (FP64)."""
    p = tm.DPParams(a=1.0)
    print("snapshot resume, DP F64", flush=True)
    with tm.Context() as ctx:
        ctx.configure(tm.MODEL_DP, tm.F64, p, [tm.Instance(64, 0, 12, 5)])
        ctx.init_uniform([0.0], [1.0])
        ctx.run(3)
        ctx.save_snapshot(0, tmp_path / "mid.tms")
        ctx.run(3)
        straight = ctx.download(0)
    with tm.Context() as ctx:
        ctx.configure(tm.MODEL_DP, tm.F64, p, [tm.Instance(64, 0, 12, 5, 3)])   # step0 = 3
        assert ctx.load_snapshot(0, tmp_path / "mid.tms") == 3
        ctx.run(3)
        resumed = ctx.download(0)
    assert np.array_equal(straight, resumed)


@pytest.mark.parametrize("prec,L", [("f64", 181), ("f64", 182), ("f64", 601), ("f32", 257), ("f32", 1023)])
def test_large_downloads_through_staging(tm, prec, L):
    """Downloads from 256 KiB on go through pinned staging in 32 KiB pieces and 2 MiB
    halves: sides that leave ragged pieces and start an instance at any dword, one and
    several halves, equal to the snapshot of the same fields (a plain copy), from two
    contexts in turn and from two threads at once."""
    import threading
    P = tm.F64 if prec == "f64" else tm.F32
    insts = [tm.Instance(7, 0, 3, 0), tm.Instance(L, 0, 3, 1), tm.Instance(L, 0, 3, 2)]

    def fields(ctx, k, path):
        ctx.save_snapshot(k, path)
        raw = open(path, "rb").read()
        return np.frombuffer(raw, np.float64 if prec == "f64" else np.float32, offset=64).astype(np.float64).reshape(1, L, L)

    import tempfile
    with tempfile.TemporaryDirectory() as d, tm.Context() as a, tm.Context() as b:
        for c in (a, b):
            c.configure(tm.MODEL_DP, P, tm.DPParams(), insts)
            c.init_uniform([0.0], [1.0])
            c.run(2)
        want = [fields(a, k, f"{d}/s{k}") for k in (1, 2)]
        for c in (a, b, a):
            for k in (1, 2):
                assert np.array_equal(c.download(k), want[k - 1])
        got = {}

        def many(name, c):
            got[name] = [c.download(k) for _ in range(6) for k in (1, 2)]

        ts = [threading.Thread(target=many, args=(n, c)) for n, c in (("a", a), ("b", b))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for r in got.values():
            assert len(r) == 12 and all(np.array_equal(x, want[i % 2]) for i, x in enumerate(r))


@pytest.mark.parametrize("prec,L", [("f64", 181), ("f64", 182), ("f64", 601), ("f32", 257), ("f32", 1023)])
def test_downloads_while_the_staging_is_there(tm, tmp_path, prec, L):
    """The staging is made at 8 MiB of downloads and shared: with a context that holds it,
    every download from 256 KiB on passes through it, whatever its size and its start."""
    P = tm.F64 if prec == "f64" else tm.F32
    with tm.Context() as holder, tm.Context() as ctx:
        holder.configure(tm.MODEL_DP, tm.F64, tm.DPParams(), [tm.Instance(1500, 0, 1, 0)])
        holder.init_uniform([0.0], [1.0])
        held = holder.download(0)
        ctx.configure(tm.MODEL_DP, P, tm.DPParams(), [tm.Instance(7, 0, 3, 0), tm.Instance(L, 0, 3, 1), tm.Instance(L, 0, 3, 2)])
        ctx.init_uniform([0.0], [1.0])
        ctx.run(2)
        for k in (1, 2):
            ctx.save_snapshot(k, tmp_path / "s")
            want = np.frombuffer((tmp_path / "s").read_bytes(), np.float64 if prec == "f64" else np.float32, offset=64)
            for _ in range(3):
                assert np.array_equal(ctx.download(k).ravel(), want.astype(np.float64))
        assert np.array_equal(holder.download(0), held)
