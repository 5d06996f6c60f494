"""Timing cases: what a user of this integrator has it do, one call path per kind.

A case is a dict of plain values; `prepare` builds what a program holds before the
call (a configured Context, or device arrays), `run` makes one pass through the
public entry points and returns everything the pass produces.  A batch pass is one
fresh replicate of the batch (rewind, initial frame, steps with the rho(t) rows, the
final fields); an operator pass is one call on device arrays.

Kinds
  dp      directed-percolation Langevin batches, FP32 or FP64
  rk      Rietkerk (P, W, O) batches, FP32 or FP64
  sweep   a Rietkerk parameter sweep: measured series and replicate statistics
  dpc     vegetation + grazer (+ predator) DP batches, FP64
  fke     Rietkerk vegetation + grazer (+ predator) batches, FP64
  move    the consumers' Fokker-Planck movement on device arrays
  rk4     the consumer model's RK4 on device arrays
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import trophic_maelstorm_amd as tm

PREC = {"f32": tm.F32, "f64": tm.F64}
SCHEME = {"euler": tm.DP_EULER, "rk4": tm.DP_RK4, "exact": tm.DP_EXACT}
SAMPLER = {"exact": tm.SAMPLER_EXACT, "compat": tm.SAMPLER_COMPAT}
CONSUMER_MODEL = {("dpc", 2): tm.MODEL_DP2, ("dpc", 3): tm.MODEL_DP3,
                  ("fke", 2): tm.MODEL_FKE2, ("fke", 3): tm.MODEL_FKE3}


def listed():
    return [
        # The smallest call: one little FP64 lattice for a few steps, as a program that
        # probes a parameter point makes it.  Launch and call latency count here.
        {"name": "dp_one_f64", "kind": "dp", "prec": "f64", "sizes": "33x1", "steps": 10, "a0": 0.72, "a1": 0.72,
         "points": 1, "scheme": "euler", "sampler": "exact"},
        # The reference's own CPU configuration: 8 replicates of 128^2.
        {"name": "dp_replicates_f64", "kind": "dp", "prec": "f64", "sizes": "128x8", "steps": 200, "a0": 0.72,
         "a1": 0.72, "points": 1, "scheme": "euler", "sampler": "exact"},
        # The benchmark's uneven batch, the live part of its quench (35.7 M cells a step).
        {"name": "dp_quench_f32", "kind": "dp", "prec": "f32", "sizes": "128x128,256x64,512x48,1024x16",
         "steps": 400, "a0": 0.72, "a1": 0.72, "points": 1, "scheme": "euler", "sampler": "exact"},
        # One plain FP64 Rietkerk lattice, stepped between two frames.
        {"name": "rk_one_f64", "kind": "rk", "prec": "f64", "sizes": "256x1", "steps": 200, "a0": 1.0, "a1": 1.0,
         "points": 1, "sampler": "exact"},
        # FP64 Rietkerk replicates of odd sides, under the reference's Gaussian shortcuts.
        {"name": "rk_odd_compat_f64", "kind": "rk", "prec": "f64", "sizes": "129x8,187x4,250x4", "steps": 60,
         "a0": 0.5, "a1": 1.5, "points": 4, "sampler": "compat"},
        # The FP64 Rietkerk batch with exact draws (the precision the reference runs in).
        {"name": "rk_batch_f64", "kind": "rk", "prec": "f64", "sizes": "512x16", "steps": 100, "a0": 0.5, "a1": 1.5,
         "points": 16, "sampler": "exact"},
        # The FP32 Rietkerk sweep: 16 rainfalls x 4 replicates of 512^2, series and statistics.
        {"name": "rk_sweep_f32", "kind": "sweep", "prec": "f32", "sizes": "512x64", "steps": 300, "a0": 0.5,
         "a1": 1.5, "points": 16, "sampler": "exact"},
        # Vegetation + grazer DP replicates.
        {"name": "dp2_f64", "kind": "dpc", "species": 2, "sizes": "256x16", "steps": 100, "a0": 5e-6, "a1": 2e-5,
         "points": 4, "pr": 0.521425, "sampler": "exact"},
        # ... with the predator, odd sides.
        {"name": "dp3_odd_f64", "kind": "dpc", "species": 3, "sizes": "101x4,193x4,250x4", "steps": 60, "a0": 5e-6,
         "a1": 2e-5, "points": 4, "pr": 0.521425, "sampler": "exact"},
        # Rietkerk vegetation + grazer + predator: 4 rainfalls x 4 replicates of 256^2.
        {"name": "fke3_f64", "kind": "fke", "species": 3, "sizes": "256x16", "steps": 100, "a0": 0.8, "a1": 1.6,
         "points": 4, "sampler": "exact"},
        # The movement step of two consumers on one large lattice.
        {"name": "move_1024", "kind": "move", "species": 2, "L": 1024, "sigma1": 1.0, "sigma2": 3.0, "fill": 0.5},
        # The consumer model's RK4 on one lattice.
        {"name": "rk4_512", "kind": "rk4", "species": 2, "L": 512, "dt": 0.1},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, lo, hi, cells_lo, cells_hi, groups):
    """1 .. groups lattice sides in [lo, hi] sharing a random number of cells."""
    n = rng.randint(1, groups)
    total = math.exp(rng.uniform(math.log(cells_lo), math.log(cells_hi)))
    out = []
    for _ in range(n):
        L = _logint(rng, lo, hi)
        out.append(f"{L}x{max(1, min(256, int(total / n / (L * L))))}")
    return ",".join(out)


def _steps(rng, sizes, lo, hi, budget):
    cells = sum(L * L for L in _sides(sizes))
    return max(1, min(_logint(rng, lo, hi), int(budget / cells)))


def draw(rng):
    kind = rng.choice(["dp", "rk", "sweep", "dpc", "fke", "move", "rk4"])
    if kind == "move":
        L = _logint(rng, 48, 1536)
        return {"kind": kind, "species": rng.choice([1, 2]), "L": L, "sigma1": round(rng.uniform(0.6, 2.0), 3),
                "sigma2": round(rng.uniform(1.0, 4.0), 3), "fill": round(rng.uniform(0.2, 1.0), 3)}
    if kind == "rk4":
        return {"kind": kind, "species": rng.choice([1, 2]), "L": _logint(rng, 24, 1024),
                "dt": round(rng.uniform(0.02, 0.12), 4)}
    if kind == "dp":
        prec = rng.choice(["f32", "f64"])
        sizes = _batch(rng, 17, 1024, 1e3, 2e7 if prec == "f32" else 4e6, 4)
        a = round(rng.uniform(0.6, 1.0), 3)
        return {"kind": kind, "prec": prec, "sizes": sizes,
                "steps": _steps(rng, sizes, 8, 400, 8e9 if prec == "f32" else 1e9), "a0": a, "a1": round(a + 0.1, 3),
                "points": rng.choice([1, 2, 4]), "scheme": rng.choice(["euler", "rk4", "exact"]),
                "sampler": rng.choice(["exact", "exact", "compat"])}
    if kind in ("rk", "sweep"):
        prec = rng.choice(["f32", "f64"])
        sizes = _batch(rng, 24, 768, 2e3, 1.2e7 if prec == "f32" else 3e6, 3)
        return {"kind": kind, "prec": prec, "sizes": sizes,
                "steps": _steps(rng, sizes, 8, 300, 3e9 if prec == "f32" else 3e8),
                "a0": round(rng.uniform(0.5, 0.9), 3), "a1": round(rng.uniform(0.9, 1.5), 3),
                "points": rng.choice([1, 2, 4]), "sampler": rng.choice(["exact", "exact", "compat"])}
    if kind == "dpc":
        sizes = _batch(rng, 24, 384, 2e3, 1.5e6, 3)
        return {"kind": kind, "species": rng.choice([2, 3]), "sizes": sizes, "steps": _steps(rng, sizes, 4, 100, 8e7),
                "a0": 5e-6, "a1": 2e-5, "points": rng.choice([1, 2, 4]), "pr": round(rng.uniform(0.15, 0.95), 4),
                "sampler": "exact"}
    sizes = _batch(rng, 32, 384, 2e3, 1.2e6, 3)
    return {"kind": "fke", "species": rng.choice([2, 3]), "sizes": sizes, "steps": _steps(rng, sizes, 4, 100, 8e7),
            "a0": 0.8, "a1": 1.6, "points": rng.choice([1, 2, 4]), "sampler": rng.choice(["exact", "exact", "compat"])}


def _sides(sizes):
    out = []
    for part in sizes.split(","):
        L, n = part.split("x")
        out += [int(L)] * int(n)
    return out


def _instances(case, seed):
    sides = _sides(case["sizes"])
    return [tm.Instance(L, k % case["points"], seed & 0xFFFFFFFF, k) for k, L in enumerate(sides)]


def _points(case):
    if case["points"] == 1:
        return [case["a0"]]
    return [float(a) for a in np.linspace(case["a0"], case["a1"], case["points"])]


def _batch_state(case, seed):
    kind = case["kind"]
    smp = SAMPLER[case["sampler"]]
    ctx = tm.Context(0)
    if kind == "dp":
        ps = [tm.DPParams(a=a, a_end=a - 0.02, ramp_steps=10_000, scheme=SCHEME[case["scheme"]], sampler=smp)
              for a in _points(case)]
        ctx.configure(tm.MODEL_DP, PREC[case["prec"]], ps, _instances(case, seed))
        lo, hi = [0.0], [1.0]
    elif kind in ("rk", "sweep"):
        ps = [tm.RietkerkParams(R=a, sampler=smp) for a in _points(case)]
        ctx.configure(tm.MODEL_RIETKERK, PREC[case["prec"]], ps, _instances(case, seed))
        lo, hi = [0.0, 0.0, 0.0], [90.0, 1.0, 1.0]
    elif kind == "dpc":
        ps = [tm.DPCParams(a=a, b=1e-6, pR=(0.0, case["pr"], case["pr"]), sampler=smp) for a in _points(case)]
        ctx.configure(CONSUMER_MODEL["dpc", case["species"]], tm.F64, ps, _instances(case, seed))
        hi = [20.0, 2.0, 0.0] if case["species"] == 2 else [20.0, 2.0, 0.5, 0.0, 0.0]
        lo = [0.0] * len(hi)
    else:
        ps = [tm.FKEParams(a=a / 24.0, sampler=smp) for a in _points(case)]
        ctx.configure(CONSUMER_MODEL["fke", case["species"]], tm.F64, ps, _instances(case, seed))
        hi = [60.0, 3.0, 2.0, 2.0, 0.0] if case["species"] == 2 else [60.0, 3.0, 0.5, 2.0, 2.0, 0.0, 0.0]
        lo = [0.0] * len(hi)
    # the program's host buffer of the batch, instance blocks [nf][L * L] back to back
    sizes = [ctx.nfields * i.L * i.L for i in ctx.instances]
    host = np.zeros(sum(sizes))
    ends = np.cumsum([0] + sizes)
    at = [host[ends[i]:].ctypes.data_as(C.POINTER(C.c_double)) for i in range(len(sizes))]
    st = {"kind": kind, "ctx": ctx, "lo": lo, "hi": hi, "steps": case["steps"], "host": host, "at": at}
    if kind == "sweep":   # the reference's log-spaced measurement times up to the last step
        dt = ps[0].dt
        meas = tm.measure_steps(tm.sweep_times(25.0, dt), dt)
        st["meas"] = np.append(meas[meas < case["steps"]], np.int64(case["steps"]))
    return st


def _move_inputs(case, seed, device):
    """rho (partly empty), gamma and the drawn velocities of the grazer and predator."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    ns, L = case["species"], case["L"]
    rho = 2.0 * torch.rand((ns, L, L), generator=g, dtype=torch.float64)
    rho *= torch.rand((ns, L, L), generator=g, dtype=torch.float64) < case["fill"]
    gam = torch.rand((ns, L, L), generator=g, dtype=torch.float64)
    th = 2.0 * math.pi * torch.rand((ns, L, L), generator=g, dtype=torch.float64)
    speed = torch.tensor([0.45427, 0.40587][:ns], dtype=torch.float64).view(ns, 1, 1)
    v = torch.stack([speed * torch.cos(th), speed * torch.sin(th)], dim=-1)
    return rho.to(device), gam.to(device), v.contiguous().to(device)


def _move_constants(case):
    """(rD, rV, prefactor), the two half-stencils: of each consumer, dt = 0.1 hr, dx = 0.1 km."""
    D, v, s = [0.0298, 0.05221], [0.45427, 0.40587], [case["sigma1"], case["sigma2"]]
    return [tm.fke_move_constants(D[k], v[k], s[k], 0.1, 0.1) for k in range(case["species"])]


def _rk4_inputs(case, seed, device):
    g = torch.Generator(device="cpu").manual_seed(seed)
    ns, L = case["species"], case["L"]
    top = [60.0, 3.0] + ([0.5] if ns == 2 else []) + [2.0, 2.0]
    f = torch.rand((ns + 3, L, L), generator=g, dtype=torch.float64)
    return (f * torch.tensor(top, dtype=torch.float64).view(-1, 1, 1)).to(device)


def _rk4_params(case):
    d = tm.FKEParams()
    return tm.FKERKParams(a=d.a, c=d.c, gmax=d.gmax, alpha=d.alpha, rW=d.rW, W0=d.W0, K=d.K, A=d.A, H=d.H, E=d.E,
                          M=d.M, D_W=d.D_W, D_O=d.D_O, dt=case["dt"], dt_rk=1.1817455 * case["dt"], dx=d.dx)


def prepare(case, seed):
    if case["kind"] == "move":
        rho, gam, v = _move_inputs(case, seed, "cuda")
        consts = _move_constants(case)
        sp = (tm._MoveSpecies * case["species"])(*[tm._MoveSpecies(*c[0]) for c in consts])
        sd = torch.from_numpy(np.concatenate([c[1] for c in consts])).to("cuda")   # device arrays, as the fields
        sv = torch.from_numpy(np.concatenate([c[2] for c in consts])).to("cuda")
        return {"kind": "move", "ns": case["species"], "L": case["L"], "sp": C.cast(sp, C.c_void_p), "keep": sp,
                "sd": sd, "sv": sv, "rho": rho, "gam": gam, "v": v, "out": torch.empty_like(rho)}
    if case["kind"] == "rk4":
        f = _rk4_inputs(case, seed, "cuda")
        p = _rk4_params(case)._c()
        return {"kind": "rk4", "ns": case["species"], "L": case["L"], "f0": f, "f": torch.empty_like(f), "keep": p,
                "p": C.cast(C.byref(p), C.c_void_p), "bad": C.c_int64(0)}
    return _batch_state(case, seed)


def _status(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what} returned {rc}")


def run(state):
    kind = state["kind"]
    if kind == "move":
        s = state
        _status(tm.lib().tm_fke_movement(s["ns"], s["L"], s["sp"], s["sd"].data_ptr(), s["sv"].data_ptr(),
                                         s["rho"].data_ptr(), s["gam"].data_ptr(), s["v"].data_ptr(),
                                         s["out"].data_ptr(), torch.cuda.current_stream().cuda_stream),
                "tm_fke_movement")
        return s["out"]
    if kind == "rk4":   # in place: from the inputs every time
        s = state
        s["f"].copy_(s["f0"])
        _status(tm.lib().tm_fke_rk4(s["ns"], s["L"], s["p"], s["f"].data_ptr(), C.byref(s["bad"]),
                                    torch.cuda.current_stream().cuda_stream), "tm_fke_rk4")
        return {"fields": s["f"], "n_bad": int(s["bad"].value)}
    ctx = state["ctx"]
    ctx.reset()
    ctx.init_uniform(state["lo"], state["hi"])
    out = {}
    if kind == "sweep":
        out["series"] = ctx.run_series(state["meas"])
        out["stats"] = ctx.replicate_stats(tm.STATS_REFERENCE)
    else:
        out["rows"] = ctx.run(state["steps"])
    if kind == "fke":
        out["mov"] = ctx.mov_stats()
    for i, at in enumerate(state["at"]):   # every instance into the program's host buffer
        _status(tm.lib().tm_download_fields(ctx._h, i, at), "tm_download_fields")
    out["fields"] = state["host"]
    return out


def work(case):
    """Bytes: every input of the pass read once and every output written once (a batch
    starts from a generated frame: its final fields on the device and, in FP64, for the
    program, and its rho(t) rows).  Operations: floating-point and generator operations
    of one cell's step, counted from the algorithms (ten Philox rounds, one Poisson and
    one Gamma trial, the RK4 stages, the perception and movement sums)."""
    kind = case["kind"]
    if kind == "move":
        N = case["species"] * case["L"] ** 2
        taps = sum(2 * (2 * c[0][0] + 1) * 3 + 2 * (2 * c[0][1] + 1) * 3 for c in _move_constants(case))
        return {"bytes": N * 8.0 * 5, "flops": N * (20.0 + taps / case["species"])}
    if kind == "rk4":
        N, nf = case["L"] ** 2, case["species"] + 3
        return {"bytes": N * 16.0 * nf * 2, "flops": N * 4.0 * (45 + 4 * nf)}
    cells = float(sum(L * L for L in _sides(case["sizes"])))
    if kind == "dp":
        nf, ops = 1, 150.0
    elif kind in ("rk", "sweep"):
        nf, ops = 3, 350.0
    elif kind == "dpc":
        R = int(case["pr"] / 0.1)
        nf, ops = 2 * case["species"] - 1, case["species"] * 250.0 + (case["species"] - 1) * math.pi * R * R
    else:
        nf, ops = 2 * case["species"] + 1, 500.0 + 300.0 * (case["species"] - 1)
    es = 4 if case.get("prec") == "f32" else 8
    rows = 16.0 * nf * len(_sides(case["sizes"])) * case["steps"]
    return {"bytes": cells * nf * (es + 8.0) + rows, "flops": cells * ops * case["steps"]}


def _exact_move(case, seed):
    """The four-term spread of every source, by rows and columns, in plain torch FP64."""
    rho, gam, v = _move_inputs(case, seed, "cuda")
    L = case["L"]
    idx = torch.arange(L, device="cuda", dtype=torch.float64)
    outs = []
    for s, ((rD, rV, pref), SD, SV) in enumerate(_move_constants(case)):
        r = torch.where(rho[s] < 1e-10, torch.zeros_like(rho[s]), rho[s])
        g = gam[s]
        # round half away from zero, as C's round
        def rnd(x):
            return torch.sign(x) * torch.floor(torch.abs(x) + 0.5)
        mx = torch.remainder(rnd(idx[:, None] + v[s, :, :, 0] * pref).long(), L)
        my = torch.remainder(rnd(idx[None, :] + v[s, :, :, 1] * pref).long(), L)
        row = torch.arange(L, device="cuda")[:, None].expand(L, L)
        col = torch.arange(L, device="cuda")[None, :].expand(L, L)

        def put(w, p, q):
            return torch.zeros(L * L, dtype=torch.float64, device="cuda").index_add_(
                0, (p * L + q).reshape(-1), w.reshape(-1)).view(L, L)

        def conv(x, st, dim):
            y = st[0] * x
            for k in range(1, len(st)):
                y = y + st[k] * (torch.roll(x, k, dim) + torch.roll(x, -k, dim))
            return y
        cx = g * g * r
        y1 = put((g - g * g) * r, row, my)
        y2 = put((g - g * g) * r, mx, col)
        z = put((1 - g) * (1 - g) * r, mx, my)
        P = conv(cx, SD, 1) + conv(y1, SV, 1)
        Q = conv(y2, SD, 1) + conv(z, SV, 1)
        outs.append(conv(P, SD, 0) + conv(Q, SV, 0))
    return torch.stack(outs)


def _exact_rk4(case, seed):
    """RK4 of the consumer model's trophic and water terms in plain torch FP64."""
    y0 = _rk4_inputs(case, seed, "cuda")
    p = _rk4_params(case)
    ns = case["species"]
    W, O = ns + 1, ns + 2
    A01, A12 = p.A[0][1], p.A[1][2]
    h01, h12 = p.H[0][1], p.H[1][2]

    def lap(x):
        return torch.roll(x, 1, 0) + torch.roll(x, -1, 0) + torch.roll(x, 1, 1) + torch.roll(x, -1, 1) - 4 * x

    def f(y):
        P, G, w, o = y[0], y[1], y[W], y[O]
        d = torch.empty_like(y)
        inf = p.alpha * (P + p.K[2] * p.W0) / (P + p.K[2]) * o
        eat = A01 * P / (1 + A01 * h01 * P) * G
        up = p.gmax * w * P / (w + p.K[1])
        d[0] = p.c * up - eat
        d[1] = p.E[1] * eat - p.M[1] * G
        if ns == 2:
            eat2 = A12 * G / (1 + A12 * h12 * G) * y[2]
            d[1] -= eat2
            d[2] = p.E[2] * eat2 - p.M[2] * y[2]
        d[W] = inf - up - p.rW * w + p.D_W / p.dx ** 2 * lap(w)
        d[O] = p.a - inf + p.D_O / p.dx ** 2 * lap(o)
        return d

    h = p.dt_rk
    k1 = f(y0)
    k2 = f(y0 + h / 2 * k1)
    k3 = f(y0 + h / 2 * k2)
    k4 = f(y0 + p.dt * k3)
    y = y0 + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    return {"fields": y, "n_bad": int(((y < 0) | ~torch.isfinite(y)).sum())}


def exact(case, seed):
    """The operators' results in plain torch FP64.  A batch's fields are draws of this
    library's own random stream and samplers: no value exists for them outside it."""
    if case["kind"] == "move":
        return _exact_move(case, seed)
    if case["kind"] == "rk4":
        return _exact_rk4(case, seed)
    return None
