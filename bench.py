"""Benchmark of the fused GEMM+epilogue hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload C2]
                    [--configs C2,C3,C4,C5] [--no-cpu] [--no-eager] [--no-compile]

Headline (the driver's contract).  A step is one forward of the headline
workload (default C2, the MLP block: GEMM1+bias+GELU and GEMM2+bias+residual,
two launches of the gfx950 kernel family through the C ABI) on synthetic
seeded inputs resident in HBM.  W untimed steps, then exactly K timed steps
bracketed by ``torch.cuda.synchronize()``; ``value`` = wall ms per step.
Rank 0 prints one JSON line carrying (of ``configs`` and ``reference_presets`` the
times, speedups and check results; the records whole go to stderr):

* ``roofline`` — the dominant kernel's algorithmic FLOPs per launch over its
  average launch duration (HIP events on the launch stream, inside the timed
  region), against the 2.5 PFLOP/s bf16 dense spec and against
  ``peak_measured``, the MFMA-only rate this device sustains at its
  power-limited clock (``fuseml_mfma_peak_probe``, run in this process);
  ``traffic`` from the committed rocprofv3 FETCH_SIZE/WRITE_SIZE summary;
* ``configs`` — every benchmark config (C2..C5): the fused step, the same
  module under PyTorch eager and under ``torch.compile(model,
  backend=FuseMLCompiler())``, each the median (and quartiles) of HIP-event
  timed iterations (at least ``--min-iters`` and ``--min-seconds``, the
  reference's harness times >= 5 s, benchmarks/bench_mlp_block.py:544-590),
  a cache-cold median (1 GiB written between iterations: more than the 256 MB
  Infinity Cache), per-kernel rates, and a correctness gate: the timed fused
  output at sampled rows against a float32 PyTorch reference (tiles rtol/atol
  2e-2, reductions 1e-2 relative; bench_mlp_block.py:453-485), with eager
  bf16's own error beside it as calibration;
* ``reference_presets`` — the presets the reference publishes its speedups on
  (bench_mlp_block.py:64-153, README.md:85-96): each timed as the reference's
  harness times it (events around one forward, a synchronisation after each,
  median), eager against ``torch.compile(backend=FuseMLCompiler())`` with the
  default cost model, against every group fused (cost model off) and against
  the single-kernel MLP block where it applies, and against the default
  options replayed from a HIP graph (``hip_graph=True``), with a correctness gate
  (atol 5e-2, rtol 2e-2 against a float32 forward, the reference's gate) and
  the whole-forward HBM bytes of each path counted from the shapes; each path
  also timed on the device alone (20 forwards captured into one HIP graph and
  replayed: no host dispatch in the time), with its TFLOP/s and compulsory-byte
  GB/s against the bf16 MFMA and HBM specs (``device``);
* ``fp32_block`` — the C2 block in fp32 (not a benchmark config): compiled,
  both groups as bf16 split products, against eager fp32, with errors
  against float64 at sampled rows;
* ``cpu_baseline`` — the same eager module on this host's CPU cores (bf16,
  full batch, all cores, median of timed forwards): the reference's eager
  path, reported, not a target.

One GPU only: ``--gpus`` above 1 exits with an explanation.
"""

from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
if REPO not in sys.path:
    sys.path.insert(0, REPO)

import torch  # noqa: E402

MFMA_BF16_PEAK_TFLOPS = 2500.0  # MI355X dense bf16 spec
HBM_PEAK_GBS = 8000.0

WORKLOAD_DESC = {
    "C2": "MLP block memory_bound bf16: x[16384,1024] -> addmm(1024->4096)+b1 -> GELU -> addmm(4096->1024)+b2 + residual x",
    "C3": "Activation-heavy bf16: x[16384,1024] -> addmm(1024->4096)+b -> ReLU -> *g[16384,4096] -> Sigmoid -> +row[4096]",
    "C4": "GEMM + fused row reductions bf16: x[8192,2048] @ W[8192,2048]^T -> ReLU -> tile + row sum/amax/mean fp32",
    "C5": "Stacked MLP x4 bf16: x[8192,4096], 4 x (addmm(4096->16384)+GELU -> addmm(16384->4096)+b2+residual)",
}

RTOL = ATOL = 2e-2
RED_RTOL = 1e-2


def _parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=100)
    p.add_argument("--warmup", type=int, default=5)
    p.add_argument("--workload", default="C2", choices=sorted(WORKLOAD_DESC), help="headline workload")
    p.add_argument("--configs", default="C2,C3,C4,C5",
                   help="comma-separated configs for the per-config section ('' to skip)")
    p.add_argument("--min-iters", type=int, default=200)
    p.add_argument("--min-seconds", type=float, default=1.0)
    p.add_argument("--max-seconds", type=float, default=5.0)
    p.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    p.add_argument("--no-eager", action="store_true", help="skip the eager GPU comparison")
    p.add_argument("--no-compile", action="store_true", help="skip torch.compile timing")
    p.add_argument("--no-fp32", action="store_true", help="skip the fp32 block (split-product path)")
    p.add_argument("--eager-only", action="store_true",
                   help="run only the eager leg of --workload (rocprof counter runs of the eager module)")
    p.add_argument("--cpu-iters", type=int, default=5)
    p.add_argument("--presets", default="small,memory_bound,medium,activation_heavy_memory_bound,"
                   "activation_heavy_medium,stacked_memory_bound,stacked_medium",
                   help="reference presets to time ('' to skip; --configs '' skips them too)")
    p.add_argument("--settle-s", type=float, default=0.5,
                   help="untimed seconds of the step before its warm-up steps (the clock ramps up "
                        "over the first ~100 ms of load)")
    p.add_argument("--all-hip-headline", action="store_true",
                   help="time the all-HIP pipeline as the headline and skip the compiled module "
                        "(rocprof runs of the fused kernels alone)")
    p.add_argument("--calib-copy-mb", type=int, default=0,
                   help="after timing, run device copies of this size (rocprof counter calibration)")
    return p.parse_args()


# ---------------------------------------------------------------------------
# Fused pipelines: one list of (label, launcher, arg-builder, out key, gemm) per workload
# ---------------------------------------------------------------------------


def _build_pipeline(name: str, wl):
    from fuseml_amd.epilogue import EpilogueSpec, EpiOp
    from fuseml_amd.launcher import HipKernelLauncher

    dt = wl.dtype
    m = wl.model
    stages = []

    def mlp_block(prefix, blk, gemms):
        g1 = HipKernelLauncher(EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("gelu_erf")), dt), 3)
        g2 = HipKernelLauncher(EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("add", 3)), dt), 4)
        w1t, b1 = blk.linear1.weight.t(), blk.linear1.bias
        w2t, b2 = blk.linear2.weight.t(), blk.linear2.bias
        stages.append((f"{prefix}G1 addmm+bias+gelu", g1, lambda s: (b1, s["x"], w1t), "h", gemms[0]))
        stages.append((f"{prefix}G2 addmm+bias+residual", g2, lambda s: (b2, s["h"], w2t, s["x"]), "x", gemms[1]))

    if name == "C2":
        mlp_block("", m, wl.gemms)
    elif name == "C5":
        for i, blk in enumerate(m.blocks):
            mlp_block(f"B{i} ", blk, wl.gemms[2 * i: 2 * i + 2])
    elif name == "C3":
        lin = m.linear
        spec = EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("relu"), EpiOp("mul", 3), EpiOp("sigmoid"),
                                   EpiOp("add", 4)), dt)
        g = HipKernelLauncher(spec, 5)
        stages.append(("addmm+bias+relu*g+sigmoid+row", g,
                       lambda s: (lin.bias, s["x"], lin.weight.t(), s["g"], m.row), "y", wl.gemms[0]))
    elif name == "C4":
        # the spec FuseMLCompiler(fuse_sibling_reductions=True) derives for this module
        spec = EpilogueSpec(0, 1, (EpiOp("relu"),), dt, store_tile=True,
                            reductions=("sum", "amax", "mean"), reduce_axis=1,
                            reduce_dtypes=(torch.float32,) * 3,
                            outputs=(("red", "sum"), ("red", "amax"), ("red", "mean"), ("tile",)))
        g = HipKernelLauncher(spec, 2)
        wt = m.linear.weight.t()
        stages.append(("mm+relu+rowsum/amax/mean", g, lambda s: (s["x"], wt), "y", wl.gemms[0]))
    return stages


def _run_pipeline(stages, state, events=None, io=None):
    for i, (_, launcher, args, out_key, _) in enumerate(stages):
        if events is not None:
            events[i][0].record()
        a = args(state)
        out = launcher(*a)
        if events is not None:
            events[i][1].record()
        if io is not None:
            io.append((a, out))
        state[out_key] = out
    return state


def _final(name, state):
    return state["y"] if name in ("C3", "C4") else state["x"]


def _initial_state(name, wl):
    st = {"x": wl.inputs[0]}
    if name == "C3":
        st["g"] = wl.inputs[1]
    return st


def _algorithmic_bytes(args, out):
    """HBM bytes a launch must move at least: every distinct input tensor read
    once (a [K,N] weight view counts its K*N elements) and every output written
    once."""
    seen, total = set(), 0
    outs = out if isinstance(out, (tuple, list)) else (out,)
    for t in list(args) + list(outs):
        if isinstance(t, torch.Tensor) and (t.data_ptr(), t.numel()) not in seen:
            seen.add((t.data_ptr(), t.numel()))
            total += t.numel() * t.element_size()
    return total


# ---------------------------------------------------------------------------
# Timing
# ---------------------------------------------------------------------------


def _quartiles(xs):
    xs = sorted(xs)
    q = statistics.quantiles(xs, n=4) if len(xs) >= 2 else [xs[0]] * 3
    return {"median_ms": round(q[1], 4), "p25_ms": round(q[0], 4), "p75_ms": round(q[2], 4), "iters": len(xs)}


def _time_events(fn, args, flush=None, warmup=25):
    """HIP-event time of each fn() call on the current stream, over at least
    args.min_iters calls and args.min_seconds (at most args.max_seconds once
    min_iters are done).  `flush`, if given, runs untimed before each call."""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    times = []
    t0 = time.perf_counter()
    while True:
        batch = []
        for _ in range(10):
            if flush is not None:
                flush()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            fn()
            e.record()
            batch.append((s, e))
        torch.cuda.synchronize()
        times += [s.elapsed_time(e) for s, e in batch]
        el = time.perf_counter() - t0
        if len(times) >= args.min_iters and (el >= args.min_seconds or el >= args.max_seconds):
            break
    return _quartiles(times)


class _Flush:
    """Writes 1 GiB between timed iterations: more than the 256 MB Infinity
    Cache plus the L2s, so every operand is re-read from HBM (the reference
    flushes 128 MB, bench_mlp_block.py:436-445, sized for a 4050 Laptop's L2)."""

    def __init__(self, dev):
        self.buf = torch.empty(1 << 28, dtype=torch.float32, device=dev)
        self.k = 0

    def __call__(self):
        self.k += 1
        self.buf.fill_(float(self.k))


# ---------------------------------------------------------------------------
# Correctness gate: fused output at sampled rows against float32 PyTorch
# ---------------------------------------------------------------------------


def _sample_rows(M, n=64, seed=0):
    g = torch.Generator().manual_seed(seed)
    rows = torch.randint(0, M, (n,), generator=g)
    return torch.unique(torch.cat([torch.tensor([0, M - 1]), rows]))


def _reference_rows(name, wl, rows):
    """Float32 PyTorch forward of the workload at `rows` (rows are independent)."""
    f = lambda t: t.float()  # noqa: E731
    m = wl.model
    with torch.no_grad():
        x = f(wl.inputs[0][rows])
        if name == "C2":
            h = torch.nn.functional.gelu(x @ f(m.linear1.weight).t() + f(m.linear1.bias))
            return {"tile": h @ f(m.linear2.weight).t() + f(m.linear2.bias) + x}
        if name == "C3":
            g = f(wl.inputs[1][rows])
            h = torch.relu(x @ f(m.linear.weight).t() + f(m.linear.bias))
            return {"tile": torch.sigmoid(h * g) + f(m.row)}
        if name == "C4":
            h = torch.relu(x @ f(m.linear.weight).t())
            return {"tile": h, "sum": h.sum(-1), "amax": h.amax(-1), "mean": h.mean(-1)}
        y = x
        for blk in m.blocks:
            h = torch.nn.functional.gelu(y @ f(blk.linear1.weight).t() + f(blk.linear1.bias))
            y = h @ f(blk.linear2.weight).t() + f(blk.linear2.bias) + y
        return {"tile": y}


def _as_parts(name, out):
    """Module-shaped output -> {"tile", and for C4 "sum", "amax", "mean"}."""
    if name == "C4":
        if isinstance(out, dict):
            return out
        h, s, mx, mean = out
        return {"tile": h, "sum": s, "amax": mx, "mean": mean}
    return {"tile": out}


def _check(parts, ref, rows):
    res = {"rows_checked": int(len(rows)), "ok": True}
    for k, r in ref.items():
        got = parts[k][rows].float()
        err = (got - r).abs()
        if k == "tile":
            ok = bool(torch.all(err <= ATOL + RTOL * r.abs()))
        else:
            ok = bool(torch.all(err <= RED_RTOL * r.abs() + 1e-6))
        res[f"{k}_max_abs_err"] = float(err.max())
        res["ok"] = res["ok"] and ok
    return res


# ---------------------------------------------------------------------------
# Per-config section
# ---------------------------------------------------------------------------


def _c4_fused_parts(state):
    s, mx, mean, h = state["y"]
    return {"tile": h, "sum": s, "amax": mx, "mean": mean}


def _config_detail(name, args, dev, peak_tflops, flush):
    from fuseml_amd.compiler import FuseMLCompiler
    from fuseml_amd.workloads import WORKLOADS

    wl = WORKLOADS[name]()
    wl.to(dev)
    rows = _sample_rows(wl.inputs[0].shape[0]).to(dev)
    ref = _reference_rows(name, wl, rows)
    stages = _build_pipeline(name, wl)
    st0 = _initial_state(name, wl)
    last = {}

    def fused():
        last["state"] = _run_pipeline(stages, dict(st0))

    out = {"workload": WORKLOAD_DESC[name], "gemms_MNK": wl.gemms, "gflop": round(wl.flops / 1e9, 1)}
    with torch.no_grad():
        out["fused"] = _time_events(fused, args)
        state = last["state"]
        parts = _c4_fused_parts(state) if name == "C4" else {"tile": _final(name, state)}
        out["fused"]["check"] = _check(parts, ref, rows)
        out["fused"]["tflops"] = round(wl.flops / (out["fused"]["median_ms"] * 1e-3) / 1e12, 1)
        out["fused_cold"] = _time_events(fused, args, flush=flush)

        # per-kernel event times (the same launches, 50 steps)
        n = 50
        ev = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in stages]
              for _ in range(n)]
        for k in range(n):
            _run_pipeline(stages, dict(st0), ev[k])
        torch.cuda.synchronize()
        kernels = []
        for i, (label, _, _, _, (Mg, Ng, Kg)) in enumerate(stages):
            avg = sum(ev[k][i][0].elapsed_time(ev[k][i][1]) for k in range(n)) / n
            tf = 2.0 * Mg * Ng * Kg / (avg * 1e-3) / 1e12
            kernels.append({"kernel": label, "avg_ms": round(avg, 4), "tflops": round(tf, 1),
                            "frac_spec": round(tf / MFMA_BF16_PEAK_TFLOPS, 4),
                            "frac_measured_peak": round(tf / peak_tflops, 4) if peak_tflops else None})
        if name == "C5":  # blocks repeat the same two shapes: report one of each
            kernels = kernels[:2]
        out["kernels"] = kernels
        dom = max(kernels, key=lambda k: k["avg_ms"])
        out["dominant_frac_spec"] = dom["frac_spec"]

        if name == "C2":
            # the opt-in single-kernel MLP block (h kept on chip), same inputs
            from fuseml_amd.mlp import HipMlpLauncher

            mlp = HipMlpLauncher()
            m = wl.model
            margs = (wl.inputs[0], m.linear1.weight.t(), m.linear1.bias, m.linear2.weight.t(), m.linear2.bias,
                     wl.inputs[0])

            def single():
                last["mlp"] = mlp(*margs)

            t = _time_events(single, args)
            t["check"] = _check({"tile": last["mlp"]}, ref, rows)
            t["tflops"] = round(wl.flops / (t["median_ms"] * 1e-3) / 1e12, 1)
            t["frac_spec"] = round(t["tflops"] / MFMA_BF16_PEAK_TFLOPS, 4)
            out["fused_mlp_block"] = t
        if not args.no_eager:
            out["eager"] = _time_events(lambda: wl.model(*wl.inputs), args)
            eo = wl.model(*wl.inputs)
            out["eager"]["check"] = _check(_as_parts(name, eo), ref, rows)
            out["speedup_vs_eager"] = round(out["eager"]["median_ms"] / out["fused"]["median_ms"], 3)
        if not args.no_compile:
            torch._dynamo.reset()
            be = FuseMLCompiler(fuse_sibling_reductions=(name == "C4"))
            compiled = torch.compile(wl.model, backend=be)
            t0 = time.perf_counter()
            co = compiled(*wl.inputs)
            torch.cuda.synchronize()
            comp = {"first_call_s": round(time.perf_counter() - t0, 2),
                    "fusion_strategy": be.fusion_strategy,
                    "hip_launchers": len({id(x) for x in be.launchers})}
            comp.update(_time_events(lambda: compiled(*wl.inputs), args))
            comp["check"] = _check(_as_parts(name, co), ref, rows)
            out["compiled"] = comp
    del wl, stages, st0, last
    torch.cuda.empty_cache()
    return out


def preset_traffic(kind: str, M: int, D: int, I: int, blocks: int) -> dict:
    """HBM bytes of one forward of a reference preset (bf16, every tensor read
    or written once per kernel that touches it), per path:

    * eager: addmm (x, W1, b1 -> t), GELU (t -> t), for the activation-heavy
      block * 0.5 and + 0.125 (t -> t each), addmm (t, W2, b2 -> u), + x (u, x -> y);
    * fused (two launches per block): (x, W1, b1 -> h), (h, W2, b2, x -> y);
    * single-kernel MLP: (x, W1, b1, W2, b2 -> y), x read once as input and residual
      (the activation-heavy block's scale and shift run inside it);
    * compulsory: the forward's input, every weight and bias, its output.

    "eliminated" is 1 - (path - compulsory) / (eager - compulsory): the share
    of the intermediate traffic the path removes."""
    e = 2  # bf16
    wts = D * I + I + I * D + D
    mi, md = M * I, M * D
    extra_eager_passes = 2 if kind == "activation_heavy" else 0
    eager = (md + D * I + I + mi) + 2 * mi + extra_eager_passes * 2 * mi + (mi + I * D + D + md) + 3 * md
    fused = (md + D * I + I + mi) + (mi + I * D + D + md + md)
    single = md + wts + md
    eager, fused, single = blocks * eager * e, blocks * fused * e, blocks * single * e
    comp = (md + blocks * wts + md) * e
    out = {"eager_bytes": eager, "fused_bytes": fused, "compulsory_bytes": comp,
           "fused_eliminated": round(1 - (fused - comp) / (eager - comp), 4),
           "fused_total_saved": round(1 - fused / eager, 4)}
    out.update(single_kernel_bytes=single, single_kernel_eliminated=round(1 - (single - comp) / (eager - comp), 4))
    return out


def _time_sync(fn, args, warmup=25):
    """The reference harness's timing (bench_mlp_block.py:544-590): an event
    pair around one call and a synchronisation after each; median over at
    least args.min_iters calls and args.min_seconds."""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    times = []
    t0 = time.perf_counter()
    while True:
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        fn()
        e.record()
        torch.cuda.synchronize()
        times.append(s.elapsed_time(e))
        el = time.perf_counter() - t0
        if len(times) >= args.min_iters and (el >= args.min_seconds or el >= args.max_seconds):
            break
    return _quartiles(times)


def _device_ms(fn, reps=20, repeats=7):
    """GPU time per fn() call with the host's dispatch out of the measurement:
    ``reps`` calls captured back to back into one HIP graph, which is replayed
    between an event pair; median over ``repeats`` replays.  The calls' inputs
    stay as they are (warm caches, as in the per-call timing)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(reps):
            fn()
    g.replay()
    torch.cuda.synchronize()
    times = []
    for _ in range(repeats):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        g.replay()
        e.record()
        torch.cuda.synchronize()
        times.append(s.elapsed_time(e) / reps)
    del g
    return statistics.median(times)


def preset_roofline(ms: float, flops: float, compulsory_bytes: int) -> dict:
    """A forward's device time against both rooflines: its flops over the bf16
    MFMA spec and its compulsory bytes (input, weights, output) over the HBM
    spec.  ``bound`` names the roofline whose floor is the longer one: a
    shape whose flops per compulsory byte exceed the ridge point (2.5 PFLOP/s /
    8 TB/s = 312.5) cannot reach the HBM rate even at full MFMA speed."""
    tflops = flops / (ms * 1e-3) / 1e12
    gbps = compulsory_bytes / (ms * 1e-3) / 1e9
    floor_mfma = flops / (MFMA_BF16_PEAK_TFLOPS * 1e12) * 1e3
    floor_hbm = compulsory_bytes / (HBM_PEAK_GBS * 1e9) * 1e3
    return {"device_ms": round(ms, 4), "tflops": round(tflops, 1), "frac_mfma": round(tflops / MFMA_BF16_PEAK_TFLOPS, 4),
            "GBps": round(gbps, 1), "frac_hbm": round(gbps / HBM_PEAK_GBS, 4),
            "bound": "mfma" if floor_mfma >= floor_hbm else "hbm",
            "frac_of_bound": round(max(floor_mfma, floor_hbm) / ms, 4)}


def _presets(args, dev):
    """The reference's presets: eager, compiled (default cost model), every group
    fused, and the single-kernel MLP block, timed and checked the reference's way."""
    from fuseml_amd.compiler import FuseMLCompiler
    from fuseml_amd.mlp import HipMlpLauncher
    from fuseml_amd.workloads import REFERENCE_PRESETS, reference_preset

    out = {}
    for name in [p for p in args.presets.split(",") if p]:
        print(f"[bench] preset {name}", file=sys.stderr, flush=True)
        kind, M, D, I, blocks = REFERENCE_PRESETS[name]
        wl = reference_preset(name).to(dev)
        x = wl.inputs[0]
        m = wl.model
        res = {"workload": kind, "M": M, "d_model": D, "d_intermediate": I, "blocks": blocks,
               "gflop": round(wl.flops / 1e9, 1), "traffic": preset_traffic(kind, M, D, I, blocks)}
        with torch.no_grad():
            ref = m.float()(x.float())
            m.to(torch.bfloat16)

            def gate(y):
                err = (y.float() - ref).abs()
                ok = bool((err <= 5e-2 + 2e-2 * ref.abs()).all())
                return {"max_abs_err": round(float(err.max()), 4), "pass": ok}

            res["eager"] = _time_sync(lambda: m(x), args)
            res["eager"]["check"] = gate(m(x))
            comp_bytes = res["traffic"]["compulsory_bytes"]
            res["eager"]["device"] = preset_roofline(_device_ms(lambda: m(x)), wl.flops, comp_bytes)
            # all_fused: every group as its own launch (no single-kernel MLP)
            paths = {"compiled": {}, "all_fused": dict(k_per_epilogue_pass=0, min_tiles_long_k=0,
                                                       min_output_elements=0, fuse_mlp_block=False)}
            paths["single_kernel_mlp"] = dict(fuse_mlp_block=True, k_per_epilogue_pass=0, min_tiles_long_k=0,
                                              min_output_elements=0)
            # the default options, replayed from a HIP graph (static outputs)
            paths["compiled_hip_graph"] = dict(hip_graph=True)
            for label, kw in paths.items():
                torch._dynamo.reset()
                be = FuseMLCompiler(**kw)
                c = torch.compile(m, backend=be)
                y = c(x)
                torch.cuda.synchronize()
                n_mlp = sum(1 for L in be.launchers if isinstance(L, HipMlpLauncher))
                if label == "single_kernel_mlp" and n_mlp == 0:
                    continue
                r = _time_sync(lambda: c(x), args)
                if be.graph_forwards:
                    y = c(x)  # gate a replayed output (the first calls run without the graph)
                    torch.cuda.synchronize()
                    r["hip_graph_replays"] = sum(g.replays for g in be.graph_forwards)
                r.update(check=gate(y), fusion_strategy=be.fusion_strategy,
                         fused_launchers=len({id(L) for L in be.launchers}), dispatch=be.dispatch[:1],
                         speedup_vs_eager=round(res["eager"]["median_ms"] / r["median_ms"], 3))
                if not be.graph_forwards:  # a HIP-graph forward is not captured inside another graph
                    dv = preset_roofline(_device_ms(lambda: c(x)), wl.flops, comp_bytes)
                    dv["speedup_vs_eager"] = round(res["eager"]["device"]["device_ms"] / dv["device_ms"], 3)
                    r["device"] = dv
                r["single_kernel_launchers"] = n_mlp
                res[label] = r
        out[name] = res
        del wl, m, x, ref
        torch._dynamo.reset()
        torch.cuda.empty_cache()
    return out


def _fp32_block(args, dev):
    """The C2 block in fp32 (not a benchmark config: an fp32 model's path).
    The reference fuses fp32 groups through Triton's tf32 dot
    (kernel_generator.py:1536); here both groups run as three-term bf16 split
    products (fuseml_split_bf16x3 + the fused kernel).  Compiled module against
    the same module in eager fp32 (`allow_tf32` off), HIP-event medians, and
    both against a float64 reference at sampled rows."""
    from fuseml_amd.compiler import FuseMLCompiler
    from fuseml_amd.workloads import TransformerMLP

    torch.backends.cuda.matmul.allow_tf32 = False
    torch.manual_seed(0)
    m = TransformerMLP(1024, 4096).eval().to(dev)
    x = torch.randn(16384, 1024, generator=torch.Generator().manual_seed(1)).to(dev)
    rows = _sample_rows(16384)
    with torch.no_grad():
        xr = x[rows.to(dev)].double().cpu()
        w1, b1 = m.linear1.weight.double().cpu(), m.linear1.bias.double().cpu()
        w2, b2 = m.linear2.weight.double().cpu(), m.linear2.bias.double().cpu()
        ref = torch.nn.functional.gelu(xr @ w1.t() + b1) @ w2.t() + b2 + xr
        torch._dynamo.reset()
        be = FuseMLCompiler()
        compiled = torch.compile(m, backend=be)
        y = compiled(x)
        ye = m(x)
        torch.cuda.synchronize()
        out = {"workload": "TransformerMLP fp32: x[16384,1024] -> 4096 -> 1024 + residual",
               "fusion_strategy": be.fusion_strategy,
               "hip_launchers": len({id(l) for l in be.launchers})}
        out["compiled"] = _time_events(lambda: compiled(x), args)
        out["eager_fp32"] = _time_events(lambda: m(x), args)
    out["speedup_vs_eager"] = round(out["eager_fp32"]["median_ms"] / out["compiled"]["median_ms"], 3)
    err = lambda t: float((t[rows.to(dev)].double().cpu() - ref).abs().max())  # noqa: E731
    out["max_abs_err_vs_f64"] = {"compiled": err(y), "eager_fp32": err(ye)}
    flops = 2.0 * 16384 * 1024 * 4096 * 2
    out["tflops_equivalent"] = round(flops / (out["compiled"]["median_ms"] * 1e-3) / 1e12, 1)
    del m, x, compiled, y, ye
    torch.cuda.empty_cache()
    return out


# ---------------------------------------------------------------------------
# HBM traffic per launch, from the committed rocprofv3 counter summaries
# ---------------------------------------------------------------------------

TRAFFIC_SUMMARY = os.path.join(REPO, "profiles", "traffic_{workload}.md")
EAGER_TRAFFIC_SUMMARY = os.path.join(REPO, "profiles", "traffic_eager_{workload}.md")
MFMA_BUSY_SUMMARY = os.path.join(REPO, "profiles", "mfma_busy_{workload}.md")


def _json_block(path):
    if not os.path.exists(path):
        return None
    text = open(path).read()
    if "```json" not in text:
        return None
    return json.loads(text.split("```json", 1)[1].split("```", 1)[0])


def _traffic(workload, launch):
    """Bytes per launch of the step's launch number `launch` (issue order within
    a step, as `python -m fuseml_amd.profiling traffic --per-step N` numbers
    them), or None."""
    data = _json_block(TRAFFIC_SUMMARY.format(workload=workload))
    if data is None:
        return None
    for k in data.get("kernels", []):
        if (str(k.get("kernel", "")).startswith("gemm_epilogue_kernel") and k.get("launch") == launch
                and k.get("fetch_bytes") is not None and k.get("write_bytes") is not None):
            return int(k["fetch_bytes"] + k["write_bytes"])
    return None


def _mfma_busy(workload, launch):
    """MFMA-busy fraction of the launch from the committed counter summary
    (SQ_VALU_MFMA_BUSY_CYCLES over GRBM_GUI_ACTIVE x CUs), or None."""
    data = _json_block(MFMA_BUSY_SUMMARY.format(workload=workload))
    if data is None:
        return None
    for k in data.get("kernels", []):
        if str(k.get("kernel", "")).startswith("gemm_epilogue_kernel") and k.get("launch") == launch:
            return k.get("mfma_busy_frac")
    return None


def _hbm_traffic(workload, gemms):
    """Fused step against the eager module, both from committed counter summaries.

    Final-output bytes are what any implementation must write (the last GEMM's
    bf16 tile, plus C4's three fp32 reduction vectors); written bytes beyond
    them are intermediates.  Each intermediate is written once and read back at
    least once, so the share of intermediate writes removed is the share of
    intermediate traffic removed."""
    fused, eager = _json_block(TRAFFIC_SUMMARY.format(workload=workload)), _json_block(
        EAGER_TRAFFIC_SUMMARY.format(workload=workload))
    if fused is None or eager is None:
        return None
    gemm_entries = [k for k in fused["kernels"] if str(k["kernel"]).startswith("gemm_epilogue_kernel")]
    if not gemm_entries or any(k.get("fetch_bytes") is None or k.get("write_bytes") is None
                               for k in fused["kernels"]):
        return None
    # the summaries number a step's launches modulo their count of distinct shapes
    reps = len(gemms) / len(gemm_entries)
    f_fetch = f_write = 0.0
    for k in fused["kernels"]:
        r = reps if k in gemm_entries else 1.0
        f_fetch += k["fetch_bytes"] * r
        f_write += k["write_bytes"] * r
    M, N, _ = gemms[-1]
    out_bytes = M * N * 2 + (3 * M * 4 if workload == "C4" else 0)
    e_fetch, e_write = eager["fetch_bytes_per_call"], eager["write_bytes_per_call"]
    e_int, f_int = e_write - out_bytes, max(f_write - out_bytes, 0.0)
    return {
        "eager_bytes": int(e_fetch + e_write),
        "fused_bytes": int(f_fetch + f_write),
        "saved_frac": round(1.0 - (f_fetch + f_write) / (e_fetch + e_write), 4),
        "eager_write_bytes": int(e_write),
        "fused_write_bytes": int(f_write),
        "final_output_bytes": int(out_bytes),
        "intermediate_eliminated_frac": round(1.0 - f_int / e_int, 4) if e_int > 0 else None,
        "source": f"profiles/traffic_{workload}.md, profiles/traffic_eager_{workload}.md",
    }


# ---------------------------------------------------------------------------
# Measured MFMA peak and the CPU baseline
# ---------------------------------------------------------------------------


def _mfma_peak(dev, seconds=0.3):
    """bf16 MFMA TFLOP/s that this device sustains: fuseml_mfma_peak_probe (MFMAs
    only, random register operands, every SIMD of every CU) timed with HIP
    events; the median of 5 launches of about `seconds` each."""
    import ctypes

    from fuseml_amd import _abi

    lib = _abi.load_library()
    wgs = torch.cuda.get_device_properties(dev).multi_processor_count
    sink = torch.empty(wgs * 256, dtype=torch.float32, device=dev)
    stream = torch.cuda.current_stream(dev)
    flop_per_iter = wgs * 4 * 8 * 2 * 32 * 32 * 16

    def run(iters):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        rc = lib.fuseml_mfma_peak_probe(ctypes.c_int64(iters), wgs, ctypes.c_void_p(sink.data_ptr()),
                                        ctypes.c_void_p(stream.cuda_stream))
        e.record()
        if rc != 0:
            raise RuntimeError(f"fuseml_mfma_peak_probe: {rc}")
        torch.cuda.synchronize()
        return s.elapsed_time(e) * 1e-3

    dt = run(2000)
    iters = max(2000, int(2000 * seconds / max(dt, 1e-6)))
    rates = sorted(flop_per_iter * iters / run(iters) / 1e12 for _ in range(5))
    return {"tflops": round(rates[2], 1), "kernel": "fuseml_mfma_peak_probe (v_mfma_f32_32x32x16_bf16 only)",
            "iters": iters, "workgroups": wgs}


def _cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _cpu_baseline(name, iters):
    """The workload's eager nn.Module on this host's CPU: bf16 (fp32 for C1),
    full batch, torch.set_num_threads(len(sched_getaffinity)), one warm-up
    forward then the median of `iters` timed forwards (perf_counter)."""
    from fuseml_amd.workloads import WORKLOADS

    cores = len(os.sched_getaffinity(0))
    prev = torch.get_num_threads()
    torch.set_num_threads(cores)
    try:
        wl = WORKLOADS[name]()  # CPU tensors, same seeds as the GPU run
        with torch.no_grad():
            wl.model(*wl.inputs)
            ts = []
            for _ in range(iters):
                t0 = time.perf_counter()
                wl.model(*wl.inputs)
                ts.append(time.perf_counter() - t0)
    finally:
        torch.set_num_threads(prev)
    ms = statistics.median(ts) * 1e3
    return {
        "value": round(ms, 2),
        "unit": "ms per full-batch forward",
        "cores": cores,
        "kind": "reference",
        "sample": f"{name} eager PyTorch module (the reference's bypass path, gm.forward) on the CPU, "
                  f"{str(wl.dtype).replace('torch.', '')}, full batch, torch.set_num_threads({cores}), "
                  f"1 warm-up + median of {iters} forwards ({sum(ts):.1f} s)",
        "cpu_model": _cpu_model(),
        "gflops": round(wl.flops / (ms * 1e-3) / 1e9, 1),
    }


# ---------------------------------------------------------------------------


def _calib_copy(mb, dev):
    """Device copies of `mb` MiB, the known-size reference for the rocprof
    FETCH_SIZE / WRITE_SIZE scale factors."""
    if mb <= 0:
        return
    src = torch.empty(mb * 1024 * 1024, dtype=torch.uint8, device=dev)
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    del src, dst


def _settle(fn, seconds):
    """Run fn() untimed for `seconds` (then synchronise): the device's clock rises
    over the first ~100 ms of sustained load, which would otherwise fall into
    the first timed steps."""
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < seconds:
        for _ in range(10):
            fn()
        torch.cuda.synchronize()


def _run_eager(wl, warmup, steps, settle_s=0.0):
    """The workload's module under PyTorch eager: (forward calls made, ms per timed call)."""
    with torch.no_grad():
        _settle(lambda: wl.model(*wl.inputs), settle_s)
        n_warm = max(3, warmup)
        for _ in range(n_warm):
            wl.model(*wl.inputs)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            wl.model(*wl.inputs)
        torch.cuda.synchronize()
    return n_warm + steps, (time.perf_counter() - t0) * 1e3 / steps


def main():
    args = _parse()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: this build runs the fused kernels on a single MI355X "
              "(rows shard across GPUs with no exchange, so N GPUs run N independent copies). "
              "Run with --gpus 1.", file=sys.stderr)
        sys.exit(2)
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(2)

    from fuseml_amd.workloads import WORKLOADS

    name = args.workload
    dev = torch.device("cuda:0")
    torch.backends.cuda.matmul.allow_tf32 = False

    if args.eager_only:
        wl = WORKLOADS[name]()
        wl.to(dev)
        _calib_copy(args.calib_copy_mb, dev)
        calls, eager_ms = _run_eager(wl, args.warmup, args.steps)
        print(json.dumps({"workload": name, "eager_ms": round(eager_ms, 4), "eager_calls": calls}), flush=True)
        return

    # The MFMA peak probe runs first: ~1.5 s of full MFMA load also brings the
    # device to its sustained clock before the headline's warm-up steps.
    peak = _mfma_peak(dev)

    # ---- headline: exactly K timed steps of torch.compile(model, backend=FuseMLCompiler()) ----
    # (what a FuseML user runs, and what the reference's harness times,
    # benchmarks/bench_mlp_block.py:544-590; the cost model binds each group to
    # the fused HIP kernel or to its eager ops)
    from fuseml_amd.compiler import FuseMLCompiler
    from fuseml_amd.launcher import HipKernelLauncher

    wl = WORKLOADS[name]()
    wl.to(dev)
    gemms = _gemms_of(name)
    compiled_kernels = []
    compiled_info = None
    hip = []
    if not args.all_hip_headline:
        torch._dynamo.reset()
        be = FuseMLCompiler(fuse_sibling_reductions=(name == "C4"))
        compiled = torch.compile(wl.model, backend=be)
        with torch.no_grad():
            t0 = time.perf_counter()
            compiled(*wl.inputs)
            torch.cuda.synchronize()
            compile_s = time.perf_counter() - t0
            _settle(lambda: compiled(*wl.inputs), args.settle_s)
            for _ in range(args.warmup):
                compiled(*wl.inputs)
            torch.cuda.synchronize()
            hip = list({id(x): x for x in be.launchers if isinstance(x, HipKernelLauncher)}.values())
            for L in hip:
                L.timing_events = []
                L.timing_pool = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
                                 for _ in range(4 * args.steps)]
            t0 = time.perf_counter()
            for _ in range(args.steps):
                compiled(*wl.inputs)
            torch.cuda.synchronize()
            wall = time.perf_counter() - t0
        ms_per_step = wall * 1e3 / args.steps
    for L in hip:
        recs = L.timing_events
        L.timing_events = None
        by_shape = {}
        for ev0, ev1, mnk, nbytes in recs:
            by_shape.setdefault(mnk, []).append((ev0.elapsed_time(ev1), nbytes))
        for (Mg, Ng, Kg), rs in by_shape.items():
            avg = sum(r[0] for r in rs) / len(rs)
            compiled_kernels.append({
                "kernel": f"{L.spec.describe()} {Mg}x{Ng}x{Kg}", "avg_ms": round(avg, 4), "launches": len(rs),
                "gemm_MNK": [Mg, Ng, Kg], "tflops": round(2.0 * Mg * Ng * Kg / (avg * 1e-3) / 1e12, 1),
                "algorithmic_bytes": rs[0][1], "GBps": round(rs[0][1] / (avg * 1e-3) / 1e9, 1),
                "launch": gemms.index([Mg, Ng, Kg]) if [Mg, Ng, Kg] in gemms else None})
    if not args.all_hip_headline:
        compiled_info = {"fusion_strategy": be.fusion_strategy, "first_call_s": round(compile_s, 2),
                         "hip_groups": len(hip), "kernels": compiled_kernels,
                         "eager_groups": sum(1 for x in be.launchers if not isinstance(x, HipKernelLauncher))}
        del compiled, be
        torch._dynamo.reset()
    headline_eager = None
    if not args.no_eager:
        _, headline_eager = _run_eager(wl, args.warmup, args.steps, args.settle_s)

    # ---- the all-HIP pipeline (every group on the fused kernels), K timed steps ----
    stages = _build_pipeline(name, wl)
    with torch.no_grad():
        state = _initial_state(name, wl)
        _settle(lambda: _run_pipeline(stages, dict(state)), args.settle_s)
        for _ in range(args.warmup):
            _run_pipeline(stages, dict(state))
        torch.cuda.synchronize()
        events = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
                   for _ in stages] for _ in range(args.steps)]
        t0 = time.perf_counter()
        for k in range(args.steps):
            _run_pipeline(stages, dict(state), events[k])
        torch.cuda.synchronize()
        all_hip_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    if args.all_hip_headline:
        ms_per_step = all_hip_ms
    per_kernel = []
    for i, (label, _, _, _, gemm) in enumerate(stages):
        durs = [events[k][i][0].elapsed_time(events[k][i][1]) for k in range(args.steps)]
        avg = sum(durs) / len(durs)
        Mg, Ng, Kg = gemm
        per_kernel.append({"kernel": label, "avg_ms": round(avg, 4), "gemm_MNK": [Mg, Ng, Kg],
                           "tflops": round(2.0 * Mg * Ng * Kg / (avg * 1e-3) / 1e12, 1), "launch": i})
    io = []
    with torch.no_grad():
        _run_pipeline(stages, dict(state), io=io)
    torch.cuda.synchronize()
    for pk, (a, out) in zip(per_kernel, io):
        pk["algorithmic_bytes"] = _algorithmic_bytes(a, out)
        pk["GBps"] = round(pk["algorithmic_bytes"] / (pk["avg_ms"] * 1e-3) / 1e9, 1)
    del io
    _calib_copy(args.calib_copy_mb, dev)

    # Roofline: the dominant HIP kernel of the headline's timed region, or of
    # the all-HIP pipeline when the cost model sent every group to eager.
    if compiled_kernels:
        dk = max(compiled_kernels, key=lambda k: k["avg_ms"] * k["launches"])
        roof_src = "torch.compile step (timed region of the headline)"
    else:
        dk = max(per_kernel, key=lambda k: k["avg_ms"])
        roof_src = "all-HIP pipeline (every group eager in the compiled step)"
    dom = dk["launch"]
    Mg, Ng, Kg = dk["gemm_MNK"]
    achieved = 2.0 * Mg * Ng * Kg / (dk["avg_ms"] * 1e-3) / 1e12
    del wl, stages, state
    torch.cuda.empty_cache()

    # ---- per-config section ----
    configs = {}
    flush = _Flush(dev) if args.configs else None
    for c in [c for c in args.configs.split(",") if c]:
        print(f"[bench] config {c}", file=sys.stderr, flush=True)
        configs[c] = _config_detail(c, args, dev, peak["tflops"], flush)
    del flush
    torch.cuda.empty_cache()
    presets = _presets(args, dev) if args.presets and args.configs else None
    fp32 = None
    if args.configs and not args.no_fp32:
        print("[bench] fp32 block", file=sys.stderr, flush=True)
        fp32 = _fp32_block(args, dev)

    cpu = None
    if not args.no_cpu:
        print("[bench] cpu baseline", file=sys.stderr, flush=True)
        cpu = _cpu_baseline(name, args.cpu_iters)

    line = {
        "metric": "fused MLP-block latency (ms), % HBM/MFMA roofline, speedup vs eager",
        "value": round(ms_per_step, 4),
        "unit": "ms",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "settle_s": args.settle_s,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded torch.Generator inputs, random-init nn.Linear weights)",
        "config": {"workload": f"{name}: {WORKLOAD_DESC[name]}", "gemms_MNK": _gemms_of(name),
                   "path": "all-HIP pipeline (direct launchers)" if args.all_hip_headline
                   else "torch.compile(model, backend=FuseMLCompiler())", "parallelism": "single GPU"},
        "eager_ms": None if headline_eager is None else round(headline_eager, 4),
        "speedup_vs_eager": None if headline_eager is None else round(headline_eager / ms_per_step, 3),
        "compiled": compiled_info,
        "fused_all_hip": {"ms_per_step": round(all_hip_ms, 4), "kernels": per_kernel,
                          "note": "every group of the step on the fused HIP kernels (no cost-model routing)"},
        "roofline": {
            "bound": "mfma",
            "kernel": dk["kernel"],
            "source": roof_src,
            "achieved": round(achieved, 1),
            "peak": MFMA_BF16_PEAK_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(achieved / MFMA_BF16_PEAK_TFLOPS, 4),
            "traffic": _traffic(name, dom) if dom is not None else None,
            "peak_measured": peak["tflops"],
            "frac_of_measured": round(achieved / peak["tflops"], 4),
            "peak_probe": peak,
            "mfma_busy_frac": _mfma_busy(name, dom) if dom is not None else None,
        },
        # the same dominant kernel against the HBM roofline: algorithmic bytes
        # (inputs and outputs once) over its event-timed duration
        "hbm_roofline": {"kernel": dk["kernel"], "algorithmic_bytes": dk["algorithmic_bytes"],
                         "achieved": dk["GBps"], "peak": HBM_PEAK_GBS, "unit": "GB/s",
                         "frac": round(dk["GBps"] / HBM_PEAK_GBS, 4)},
        # the all-HIP pipeline's HBM bytes against the eager module's (committed counter summaries)
        "hbm_traffic": _hbm_traffic(name, [tuple(g) for g in _gemms_of(name)]),
        "configs": configs,
        "reference_presets": presets,
        "fp32_block": fp32,
        "cpu_baseline": cpu,
    }
    details = {k: line[k] for k in ("configs", "reference_presets")}
    print(f"[bench] details {json.dumps(details)}", file=sys.stderr, flush=True)
    line["configs"], line["reference_presets"] = _summaries(configs), _summaries(presets)
    print(json.dumps(line), flush=True)


def _summaries(records):
    """The figures of each config's or preset's record that the result line carries:
    per measured form its time, the speedup over eager and the device's time where
    that was measured, and whether every check passed.  The whole records, some
    20 KB, are longer than a reader of the output's last part sees."""
    if not records:
        return records
    out = {}
    for name, r in records.items():
        forms = {k: v for k, v in r.items() if isinstance(v, dict) and "median_ms" in v}
        checks = [f["check"].get("ok", f["check"].get("pass")) for f in forms.values() if f.get("check")]
        s = out[name] = {k: r[k] for k in ("speedup_vs_eager", "dominant_frac_spec") if k in r}
        s["ok"] = all(checks) if checks else None
        for k, f in forms.items():
            s[k] = {"ms": f["median_ms"]}
            if "speedup_vs_eager" in f:
                s[k]["speedup_vs_eager"] = f["speedup_vs_eager"]
            if f.get("device"):
                s[k]["device_ms"] = f["device"]["device_ms"]
    return out


def _gemms_of(name):
    """(M, N, K) of each GEMM of one forward of `name` (no tensors built)."""
    return {
        "C2": [[16384, 4096, 1024], [16384, 1024, 4096]],
        "C3": [[16384, 4096, 1024]],
        "C4": [[8192, 8192, 2048]],
        "C5": [[8192, 16384, 4096], [8192, 4096, 16384]] * 4,
    }[name]


if __name__ == "__main__":
    main()
