"""Measure stage of the shipped deliveries on one MI355X: gate first, then paired timing.

    python3 -m tempo.plugins.gfx950.measure_shipped [gemm_fp16|gemm_w8a16] [--out DIR] [--quick]

For every configuration shape of the op (C1/C2 for gemm_fp16; C3/C4 for gemm_w8a16) it
  1. runs the shipped launcher once into a 0x7f7f-poisoned output and gates it (reference
     tempo/core/measure/correctness.py:21-27): no poison left, relL2 <= 3e-3 against the
     reference semantics computed on the GPU by the naive kernel (kernels/naive/gemm_fp16.hip,
     bit-identical to the CPU oracle's fp32 sequential-k FMA; for W8A16 the weights are first
     dequantised by tempo_dequant_tile, bit-exact), and fp64 spot cells within
     |got-ref|/(|ref|+1e-3) <= 3e-3 (kernels/shipped/gemm_fp16/sm_70/ship_probe.cu:70-79);
  2. times the shipped kernel, the library bar (torch.matmul = hipBLASLt, fp16 weights) and the
     naive kernel with HIP events, in paired rounds with the arms interleaved and the weights
     rotated through > 512 MiB, and reports the median of the per-round ratios (reference
     tempo/core/measure/ratio.py:63-73).
Rows go to DIR/rows_<op>.json; tempo.plugins.gfx950.manifest folds them into manifest.json.

Counter step (the reference's Meters stage, tempo/plugins/sm70/counters.py:84-86):

    python3 -m tempo.plugins.gfx950.measure_shipped OP --counters [--groups hbm_read hbm_write mfma]

runs one rocprofv3 --pmc pass per counter group over a child program (`--counter-pass`) that
launches the shipped kernel REPS times per configuration shape, after a calibration device copy
of known size; the dispatches are attributed to the shapes in launch order and reduced to
per-launch figures (HBM bytes from FETCH_SIZE / WRITE_SIZE scaled by the copy, MFMA utilisation,
engine clock).  The parent process never touches the GPU (it only starts the profiler); the
figures go to DIR/counters_<op>.json, which the manifest folds into the matching rows.  OP may
also be "fmha" (configuration C5) for the counter step.
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

import numpy as np

PEAK_TF = 2516.6
PEAK_GBPS = 8000.0
ROUNDS = 5

SHAPES_FP16 = [(4096, 15360, 3840)] + [(M, N, K) for (N, K) in ((15360, 3840), (3840, 15360))
                                        for M in (1, 8, 16, 32, 64, 128, 256)]
NK_W8 = [(7168, 5120), (5120, 6144), (34816, 5120), (5120, 17408), (1024, 5120), (5120, 5120)]
SHAPES_W8 = [(M, N, K) for (N, K) in NK_W8 for M in (1, 16, 32, 128, 2048)]


def _source_md5(op):
    """md5 over the delivery's signed files as they were when these figures were taken (the
    manifest keeps it beside the md5 of the files it ships; a mismatch means stale figures)."""
    if op not in ("gemm_fp16", "gemm_w8a16"):
        return None
    from .manifest import md5_of

    return md5_of(op)


def _say(*a):
    print(*a, flush=True)


def _events_ms(fn, iters, stream):
    import torch

    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for i in range(iters):
        fn(i)
    e1.record(stream)
    e1.synchronize()
    return e0.elapsed_time(e1) / iters


def _spot(A, Wf, C, cells=256):
    """fp64 dot products on sampled cells: A [M,K] fp16, Wf [N,K] fp16, C [M,N] fp16 (torch)."""
    M, N = C.shape
    t = np.arange(cells)
    m, n = (t * 37) % M, (t * 53) % N
    a = A.cpu().numpy().astype(np.float64)[m]
    w = Wf[n.tolist()].cpu().numpy().astype(np.float64)
    ref = np.einsum("ik,ik->i", a, w)
    got = C.cpu().numpy().astype(np.float64)[m, n]
    return float(np.max(np.abs(got - ref) / (np.abs(ref) + 1e-3)))


def _rel_l2(got, ref):
    import torch

    g, r = got.double(), ref.double()
    den = torch.sum(r * r).item()
    return float(torch.sqrt(torch.sum((g - r) ** 2) / den).item()) if den > 0 else 0.0


ONLY = []  # --only: restrict the configuration shapes to these (M, N, K[, fmt]) tuples


def _only_ok(case) -> bool:
    return not ONLY or any(tuple(case[:len(o)]) == o for o in ONLY)


def cases_of(op: str, quick: bool = False):
    if op == "gemm_fp16":
        cases = [(M, N, K, 0) for (M, N, K) in SHAPES_FP16]
    elif op == "gemm_w8a16":
        cases = [(M, N, K, f) for f in (1, 2) for (M, N, K) in SHAPES_W8]
    else:  # fmha: configuration C5 (B, H, Hkv, S, D) carried as (S, H, D, Hkv)
        cases = [(4096, 16, 256, 8)]
    cases = cases[::4] if quick else cases
    return [c for c in cases if _only_ok(c)]


def label_of(M, N, K, fmt):
    return "%d,%d,%d,%d" % (M, N, K, fmt)


def algorithmic_bytes(op, M, N, K, fmt):
    if op == "fmha":
        S, H, D, Hkv = M, N, K, fmt
        return 2 * (2 * H * S * D + 2 * Hkv * S * D)
    wbytes = 2 * N * K if fmt == 0 else N * K + (2 * N if fmt == 1 else 3 * N * K // 128)
    return wbytes + 2 * M * K + 2 * M * N


def algorithmic_flops(op, M, N, K, fmt):
    if op == "fmha":
        S, H, D, Hkv = M, N, K, fmt
        return 4.0 * D * H * S * (S + 1) / 2
    return 2.0 * M * N * K


CALIB_BYTES = 1 << 30
REPS = 3


def dispatches_per_launch(op, M, N, K, fmt) -> int:
    """Kernels one call dispatches with a workspace at hand: a split-K call its main kernel, then
    the reduction; a call whose N is in two parts, its two parts."""
    from cuda_tempiler_amd import capi
    from tempo.plugins.gfx950 import manifest

    if op == "fmha":
        return 1
    need = capi.workspace_bytes(fmt, M, N, K)
    if op == "gemm_w8a16":
        sel = manifest._select(op)
        row = sel.select(op, M, N, K, fmt=fmt)
        if row.get("PLAN") and M > 128 and K % 128 == 0 and sel.plan(M, N, K, fmt)[3]:
            return 2
        route = capi.route(fmt, M, N, K)
        if route.endswith("t2") and route.startswith("i8"):
            return 3 if need else 2  # whole rounds, tail (+ reduce)
    return 2 if need else 1


def counter_pass(op: str, segfile: str, quick: bool = False) -> int:
    """The program a counter pass profiles: a calibration copy (3 x 1 GiB device copies), then
    REPS launches of the shipped kernel per configuration shape (inputs generated on the device
    beforehand).  Writes the launch order to `segfile` for assign_segments()."""
    import torch

    from cuda_tempiler_amd import capi

    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    segs = []
    src = torch.ones(CALIB_BYTES, dtype=torch.uint8, device=dev)
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    segs.append(dict(label="calibration", count=3, copy_bytes=CALIB_BYTES))
    del src, dst
    for (M, N, K, fmt) in cases_of(op, quick):
        _say("counter pass %s %s" % (op, label_of(M, N, K, fmt)))
        gen.manual_seed(1000 * M + N + K + fmt)
        if op == "fmha":
            S, H, D, Hkv = M, N, K, fmt
            Q = torch.randn((1, S, H, D), generator=gen, device=dev).half()
            Kt = torch.randn((1, S, Hkv, D), generator=gen, device=dev).half()
            V = torch.randn((1, S, Hkv, D), generator=gen, device=dev).half()
            run = lambda: capi.fmha_fwd(Q, Kt, V, D ** -0.5, True)  # noqa: E731
        else:
            A = (torch.randn((M, K), generator=gen, device=dev) / K ** 0.5).half()
            C = torch.empty((M, N), dtype=torch.float16, device=dev)
            if fmt == 0:
                W = (torch.randn((N, K), generator=gen, device=dev) / K ** 0.5).half()
                run = lambda: capi.gemm_fp16(A, W, C)  # noqa: E731
            elif fmt == 1:
                W = torch.randint(-127, 128, (N, K), generator=gen, device=dev, dtype=torch.int8)
                S1 = (torch.rand(N, generator=gen, device=dev) + 0.5).div(127).half()
                run = lambda: capi.gemm_w8a16(A, W, S1, None, fmt=1, C=C)  # noqa: E731
            else:
                W = torch.randint(0, 256, (N, K), generator=gen, device=dev, dtype=torch.uint8)
                S2 = (torch.rand((N, K // 128), generator=gen, device=dev) + 0.5).div(255).half()
                Z = torch.randint(100, 157, (N, K // 128), generator=gen, device=dev,
                                  dtype=torch.uint8)
                run = lambda: capi.gemm_w8a16(A, W, S2, Z, fmt=2, C=C)  # noqa: E731
        torch.cuda.synchronize()
        try:
            run()
        except capi.NotCovered:
            continue
        for _ in range(REPS - 1):
            run()
        torch.cuda.synchronize()
        route = capi.route(fmt, M, N, K) if op != "fmha" else "k_fmha_fwd"
        per = dispatches_per_launch(op, M, N, K, fmt)
        segs.append(dict(label=label_of(M, N, K, fmt), count=REPS * per, per_launch=per,
                         route=route))
    with open(segfile, "w") as f:
        json.dump(segs, f, indent=1)
    return 0


def counters(op: str, out: str, groups, quick: bool = False) -> str:
    """Parent of the counter passes (never touches the GPU): one rocprofv3 --pmc run per group,
    then per-launch figures per configuration shape into out/counters_<op>.json."""
    from tempo.plugins.gfx950.counters import (Gfx950Meters, GROUPS, assign_segments,
                                               copy_scales, derive, kernel_name, medians)

    meters = Gfx950Meters()
    per_shape, scales, routes, per_launch, kernels = {}, {}, {}, {}, {}
    for g in groups:
        d = os.path.abspath(os.path.join(out, "pmc_%s_%s" % (op, g)))
        seg = os.path.join(d, "segments.json")
        os.makedirs(d, exist_ok=True)
        argv = [sys.executable, "-m", "tempo.plugins.gfx950.measure_shipped", op,
                "--counter-pass", seg] + (["--quick"] if quick else [])
        if ONLY:
            argv += ["--only"] + [",".join(str(x) for x in o) for o in ONLY]
        _say("counter group %s: %s" % (g, " ".join(GROUPS[g])))
        disp = meters.run_pass(argv, GROUPS[g], d)
        with open(seg) as f:
            segs = json.load(f)
        got = assign_segments(disp, segs, "tempo")
        calib = got.pop("calibration")
        scales.update(copy_scales(calib, CALIB_BYTES))
        for s in segs:
            if s["label"] in got:
                routes[s["label"]] = s.get("route")
                per_launch[s["label"]] = s.get("per_launch", 1)
                kernels[s["label"]] = [kernel_name(d["kernel"]) for d in
                                       got[s["label"]][:s.get("per_launch", 1)]]
                per_shape.setdefault(s["label"], {}).update(
                    medians(got[s["label"]], s.get("per_launch", 1)))
    rows = []
    for lab, med in per_shape.items():
        M, N, K, fmt = (int(x) for x in lab.split(","))
        fig = derive(med, scales, algorithmic_bytes(op, M, N, K, fmt))
        if med.get("_duration_ns"):
            fig["pmc_duration_us"] = med["_duration_ns"] / 1e3
        rows.append(dict(M=M, N=N, K=K, fmt=fmt, route=routes.get(lab),
                         dispatches_per_launch=per_launch.get(lab, 1),
                         kernels=kernels.get(lab),
                         algorithmic_bytes=algorithmic_bytes(op, M, N, K, fmt),
                         algorithmic_flops=algorithmic_flops(op, M, N, K, fmt),
                         counters=fig))
    path = os.path.join(out, "counters_%s.json" % op)
    with open(path, "w") as f:
        json.dump({"op": op, "groups": list(groups), "scales": scales, "reps": REPS,
                   "source_md5": _source_md5(op), "rows": rows}, f, indent=1)
    _say("wrote %s: %d shapes" % (path, len(rows)))
    return path


def render_counters(path: str) -> str:
    """A counter step's JSON (counters()) as a markdown table, one row per configuration shape:
    per-launch duration under counters, HBM bytes against the algorithmic bytes, MFMA
    utilisation at the spec clock (and, for launches of 100 us or more, against the measured
    engine clock, with that clock and the LDS utilisation), LDS bank conflicts per access."""
    from tempo.plugins.gfx950.counters import CUS, MIN_CLOCK_NS

    with open(path) as f:
        got = json.load(f)
    lines = ["| M | N | K | fmt | route | disp./launch | us (pmc) | HBM MB | traffic / alg. "
             "| MFMA util (spec clk) | MFMA util (meas. clk) | sclk GHz | LDS util "
             "| LDS confl./access |", "|" + "---|" * 14]

    def f(x, fmt):
        return "-" if x is None else fmt % x

    for r in got["rows"]:
        c = r["counters"]
        long_ = c.get("pmc_duration_us", 0) * 1e3 >= MIN_CLOCK_NS
        lds = c.get("lds_util")
        if lds is None and long_ and c.get("gui_cycles") and "SQ_LDS_IDX_ACTIVE" in c:
            lds = c["SQ_LDS_IDX_ACTIVE"] / (c["gui_cycles"] * CUS)
        confl = c.get("lds_conflicts_per_access")
        if confl is None and c.get("SQ_LDS_IDX_ACTIVE", 0) > c.get("SQ_LDS_BANK_CONFLICT", 0) > 0:
            confl = c["SQ_LDS_BANK_CONFLICT"] / (c["SQ_LDS_IDX_ACTIVE"] - c["SQ_LDS_BANK_CONFLICT"])
        elif confl is None and "SQ_LDS_BANK_CONFLICT" in c:
            confl = 0.0
        lines.append("| %d | %d | %d | %d | %s | %d | %s | %s | %s | %s | %s | %s | %s | %s |" % (
            r["M"], r["N"], r["K"], r["fmt"], r.get("route") or "-",
            r.get("dispatches_per_launch", 1), f(c.get("pmc_duration_us"), "%.1f"),
            f(c.get("hbm_bytes", 0) / 1e6 if "hbm_bytes" in c else None, "%.1f"),
            f(c.get("traffic_over_algorithmic"), "%.2f"), f(c.get("mfma_util_spec_clock"), "%.3f"),
            f(c.get("mfma_util") if long_ else None, "%.3f"),
            f(c.get("sclk_ghz") if long_ else None, "%.2f"), f(lds, "%.3f"), f(confl, "%.3f")))
    if any(r.get("kernels") for r in got["rows"]):
        lines += ["", "Kernels of one launch (the row names the shape; its plan or its other arm may "
                  "run it):", ""]
        lines += ["    %d,%d,%d,%d: %s" % (r["M"], r["N"], r["K"], r["fmt"],
                                           " + ".join(r.get("kernels") or ["-"]))
                  for r in got["rows"]]
    lines += ["", "Exact HBM bytes per launch (M,N,K,fmt: fetch, write, total, algorithmic):", ""]
    for r in got["rows"]:
        c = r["counters"]
        if "hbm_bytes" in c:
            lines.append("    bytes %d,%d,%d,%d: fetch %d write %d traffic %d algorithmic %d" % (
                r["M"], r["N"], r["K"], r["fmt"], round(c["fetch_bytes"]), round(c["write_bytes"]),
                round(c["hbm_bytes"]), r["algorithmic_bytes"]))
    return "\n".join(lines) + "\n"


STALL_FRACTIONS = (  # (label, counter): wave-cycle counters as fractions of SQ_WAVE_CYCLES
    ("waiting on anything (waitcnt, barrier)", "SQ_WAIT_ANY"),
    ("waiting to issue (dependencies, issue ports)", "SQ_WAIT_INST_ANY"),
    ("issuing any instruction", "SQ_ACTIVE_INST_ANY"),
    ("issuing VALU (MFMA included)", "SQ_ACTIVE_INST_VALU"),
    ("issuing LDS", "SQ_ACTIVE_INST_LDS"),
    ("waiting to issue LDS", "SQ_WAIT_INST_LDS"),
    ("issuing VMEM", "SQ_ACTIVE_INST_VMEM"),
    ("issuing FLAT", "SQ_ACTIVE_INST_FLAT"),
    ("issuing scalar", "SQ_ACTIVE_INST_SCA"),
    ("issuing misc (s_waitcnt, s_barrier, branches)", "SQ_ACTIVE_INST_MISC"),
)


def render_stalls(path: str) -> str:
    """The stall groups of a counter step (waves, stall, issue, fifo) per shape: where the
    wave-cycles go (each SQ wave-cycle counter over SQ_WAVE_CYCLES, both in quad-cycles summed
    over the waves), the matrix cores' busy cycles and the VALU work co-issued with them (over
    the busy cycles), and the cycles the CU's address / LDS queues were full per engine cycle
    (GRBM_GUI_ACTIVE / XCDs), summed over the units that report them."""
    from tempo.plugins.gfx950.counters import XCDS

    with open(path) as f:
        got = json.load(f)
    out = []
    for r in got["rows"]:
        c = r["counters"]
        out.append("### M=%d N=%d K=%d fmt %d, row %s (%s dispatch(es) per launch, %.1f us under "
                   "counters)" % (r["M"], r["N"], r["K"], r["fmt"], r.get("route") or "-",
                                  r.get("dispatches_per_launch", 1),
                                  c.get("pmc_duration_us", float("nan"))))
        out += ["", "| wave-cycles | fraction |", "|---|---|"]
        wc = c.get("SQ_WAVE_CYCLES")
        for label, name in STALL_FRACTIONS:
            if wc and name in c:
                out.append("| %s (%s) | %.3f |" % (label, name, c[name] / wc))
        if "SQ_WAVES" in c:
            out.append("| waves per dispatch | %d |" % c["SQ_WAVES"])
        busy, coex = c.get("SQ_VALU_MFMA_BUSY_CYCLES"), c.get("SQ_VALU_MFMA_COEXEC_CYCLES")
        if busy and coex is not None:
            out.append("| VALU cycles co-issued with MFMA / MFMA busy cycles | %.3f |" % (coex / busy))
        gui = c.get("GRBM_GUI_ACTIVE")
        if gui:
            cyc = gui / XCDS
            for name in ("SQ_VMEM_TA_ADDR_FIFO_FULL", "SQ_VMEM_TA_CMD_FIFO_FULL",
                         "SQ_LDS_DATA_FIFO_FULL", "SQ_LDS_CMD_FIFO_FULL", "SQ_INST_CYCLES_SALU",
                         "SQ_INST_CYCLES_VMEM_RD"):
                if name in c:
                    out.append("| %s per engine cycle (summed over reporting units) | %.3f |"
                               % (name, c[name] / cyc))
        out.append("")
    return "\n".join(out) + "\n"


def measure(op: str, quick: bool = False):
    import torch

    from cuda_tempiler_amd import capi

    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()
    gen = torch.Generator(device=dev)
    rows = []
    for (M, N, K, fmt) in cases_of(op, quick):
        _say("measure %s fmt=%d M=%d N=%d K=%d" % (op, fmt, M, N, K))
        gen.manual_seed(1000 * M + N + K + fmt)
        A = (torch.randn((M, K), generator=gen, device=dev) / K ** 0.5).half()
        wbytes = 2 * N * K if fmt == 0 else N * K + (2 * N if fmt == 1 else 3 * N * K // 128)
        copies = max(2, -(-(512 << 20) // wbytes) + 1)
        Ws, Ss, Zs, Fs = [], [], [], []
        for c in range(copies):
            if fmt == 0:
                Ws.append((torch.randn((N, K), generator=gen, device=dev) / K ** 0.5).half())
                Ss.append(None)
                Zs.append(None)
            elif fmt == 1:
                Ws.append(torch.randint(-127, 128, (N, K), generator=gen, device=dev,
                                        dtype=torch.int8))
                Ss.append((torch.rand(N, generator=gen, device=dev) + 0.5).div(127).half())
                Zs.append(None)
            else:
                Ws.append(torch.randint(0, 256, (N, K), generator=gen, device=dev,
                                        dtype=torch.uint8))
                Ss.append((torch.rand((N, K // 128), generator=gen, device=dev) + 0.5)
                          .div(255).half())
                Zs.append(torch.randint(100, 157, (N, K // 128), generator=gen, device=dev,
                                        dtype=torch.uint8))
        # dequantised fp16 copy of the first weight set (bit-exact dequant) for gate and library bar
        if fmt == 0:
            F0 = Ws[0]
        else:
            F0 = capi.dequant_tile(Ws[0], Ss[0], Zs[0], fmt, 0, 0, N, K)
        Fb = [F0] + [F0.clone() for _ in range(max(1, -(-(512 << 20) // (2 * N * K))))]
        C = torch.empty((M, N), dtype=torch.int16, device=dev).fill_(0x7f7f).view(torch.float16)

        def ours(i, C=C):
            if fmt == 0:
                capi.gemm_fp16(A, Ws[i % copies], C)
            else:
                capi.gemm_w8a16(A, Ws[i % copies], Ss[i % copies], Zs[i % copies], fmt=fmt, C=C)

        try:
            ours(0)
        except capi.NotCovered:
            rows.append(dict(M=M, N=N, K=K, fmt=fmt, winner=None, note="not covered: fallback"))
            continue
        torch.cuda.synchronize()
        # the timed arm: the C entry point on parameter blocks built once per weight copy (the
        # operands were validated by the call above), so a launch costs the C-ABI call only and
        # the small shapes are timed on the GPU, not on the Python wrapper's checks
        sh = capi._stream(stream)
        if fmt == 0:
            pars = [capi.TempoGemmParams(capi._ptr(A), capi._ptr(Ws[c]), capi._ptr(C), M, N, K,
                                         A.stride(0), Ws[c].stride(0), C.stride(0))
                    for c in range(copies)]
            entry = capi.lib().tempo_gemm_fp16_launch
        else:
            pars = [capi.w8a16_params(A, Ws[c], Ss[c], Zs[c], C, fmt, 128) for c in range(copies)]
            entry = capi.lib().tempo_gemm_w8a16_launch

        def ours_timed(i, pars=pars, entry=entry, sh=sh):
            entry(pars[i % copies], sh)
        poison = int((C.view(torch.int16) == 0x7f7f).sum().item())
        ref = capi.naive_gemm_fp16(A, F0)
        torch.cuda.synchronize()
        rel = _rel_l2(C, ref)
        spot = _spot(A, F0, C)
        ok = poison == 0 and rel <= 3e-3 and spot <= 3e-3
        row = dict(M=M, N=N, K=K, fmt=fmt, winner=capi.route(fmt, M, N, K), poison=poison,
                   rel_l2=rel, spot_rel=spot, gate="pass" if ok else "FAIL")
        if not ok:
            rows.append(row)
            _say("  GATE FAIL", row)
            continue
        Cl = torch.empty((M, N), dtype=torch.float16, device=dev)

        def lib_bar(i):
            torch.matmul(A, Fb[i % len(Fb)].t(), out=Cl)

        def naive(i):
            capi.naive_gemm_fp16(A, F0, Cl)

        # iteration count: ~0.3 s per arm per round (reference harness: it = clamp(300/ms, 3, 2000))
        for f in (ours_timed, lib_bar):
            for i in range(3):
                f(i)
        torch.cuda.synchronize()
        t0 = _events_ms(ours_timed, 3, stream)
        it = int(min(2000, max(3, 300.0 / max(t0, 1e-3) / 10)))
        ratios, t_ours, t_lib = [], [], []
        for r in range(ROUNDS):
            a = _events_ms(ours_timed, it, stream)
            b = _events_ms(lib_bar, it, stream)
            t_ours.append(a)
            t_lib.append(b)
            ratios.append(b / a)
        tn = _events_ms(naive, 1 if M * N * K > 1e10 else 3, stream)
        ms = statistics.median(t_ours)
        flops = 2.0 * M * N * K
        byts = wbytes + 2 * M * K + 2 * M * N
        row.update(ms=ms, tflops=flops / ms / 1e9, GBps=byts / ms / 1e6,
                   mfma_frac=flops / ms / 1e9 / PEAK_TF, hbm_frac=byts / ms / 1e6 / PEAK_GBPS,
                   ratio_vs_hipblaslt=statistics.median(ratios), ratio_min=min(ratios),
                   ratio_max=max(ratios), hipblaslt_tflops=flops / statistics.median(t_lib) / 1e9,
                   naive_tflops=flops / tn / 1e9, ratio_vs_naive=tn / ms, iters=it, rounds=ROUNDS)
        rows.append(row)
        _say("  %s" % json.dumps(row))
        del Ws, Ss, Zs, Fb, F0
        torch.cuda.empty_cache()
    return rows


def card_state():
    """The card passport (card.snapshot: clocks, power, foreign processes) plus the device's
    name, architecture and CU count as torch reports them."""
    from tempo.plugins.gfx950 import card

    out = card.snapshot(0)
    try:
        import torch

        out["name"] = torch.cuda.get_device_name(0)
        p = torch.cuda.get_device_properties(0)
        out["gcn_arch"] = getattr(p, "gcnArchName", "")
        out["cus"] = p.multi_processor_count
    except Exception as e:  # recorded, not fatal
        out["name_error"] = str(e)
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("op", nargs="?", default="gemm_fp16",
                    choices=("gemm_fp16", "gemm_w8a16", "fmha"))
    ap.add_argument("--out", default="gpurun_out")
    ap.add_argument("--quick", action="store_true")
    ap.add_argument("--counters", action="store_true",
                    help="run the counter step (rocprofv3 --pmc passes) instead of timing")
    ap.add_argument("--groups", nargs="*", default=["hbm_read", "hbm_write", "mfma"])
    ap.add_argument("--counter-pass", metavar="SEGFILE",
                    help="(internal) the program a counter pass profiles")
    ap.add_argument("--only", nargs="*", default=[], metavar="M,N,K[,fmt]",
                    help="restrict the configuration shapes to these")
    ap.add_argument("--render", metavar="COUNTERS_JSON",
                    help="print a counter step's JSON as a markdown table (no GPU)")
    ap.add_argument("--render-stalls", metavar="COUNTERS_JSON",
                    help="print the stall groups of a counter step's JSON (no GPU)")
    a = ap.parse_args()
    ONLY[:] = [tuple(int(x) for x in o.split(",")) for o in a.only]
    if a.render:
        sys.stdout.write(render_counters(a.render))
        return 0
    if a.render_stalls:
        sys.stdout.write(render_stalls(a.render_stalls))
        return 0
    os.makedirs(a.out, exist_ok=True)
    if a.counter_pass:
        return counter_pass(a.op, a.counter_pass, a.quick)
    if a.counters:
        counters(a.op, a.out, a.groups, a.quick)
        return 0
    if a.op == "fmha":
        ap.error("fmha has a counter step only (--counters)")
    before = card_state()
    rows = measure(a.op, a.quick)
    after = card_state()
    path = os.path.join(a.out, "rows_%s.json" % a.op)
    with open(path, "w") as f:
        json.dump({"op": a.op, "card_before": before, "card_after": after,
                   "source_md5": _source_md5(a.op), "rows": rows}, f, indent=1)
    bad = [r for r in rows if r.get("gate") == "FAIL"]
    _say("wrote %s: %d rows, %d gate failures" % (path, len(rows), len(bad)))
    return 1 if bad else 0


if __name__ == "__main__":
    sys.exit(main())
