#!/usr/bin/env python3
"""Generates dispatch.inc from select.py: one source of the ladder, two consumers.

    python3 gen_dispatch.py > dispatch.inc

The Python predicate is what a host tree calls once at load time; the instantiation table is
what the compiler needs.  The second is generated from the first so they cannot drift
(reference: kernels/shipped/gemm_fp16/sm_70/gen_dispatch.py:6-13).
"""
from __future__ import annotations

import importlib.util
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def _select():
    spec = importlib.util.spec_from_file_location("tempo_select_fp16_gfx950",
                                                  os.path.join(HERE, "select.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


HEAD = """// GENERATED from select.py -- do not edit.  Regenerate with:
//   python3 kernels/shipped/gemm_fp16/gfx950/gen_dispatch.py > dispatch.inc
//
// Ladder, one TEMPO_ROW(band, fit, launcher, tag) per row; launch.hip expands it twice (launch
// and route).  The first row whose band holds (M, N) and whose kernel fits the shape runs; if
// none does, the answer is hipErrorInvalidConfiguration: the caller's own path takes over
// (TEMPO_FALLBACK) -- a legal answer, not a failure.
"""


def instantiation(kind, p, epi=0):
    tail = ",%d" % epi if epi else ""
    if kind == "line" and p.get("PLAN"):
        if epi:
            raise ValueError("a line row with a plan takes the plain epilogue")
        return "launch_line_or_plan<%d,%d,%d,%d,%d,%d>" % (p["MB"], p["R"], p["D"], p.get("SN", 1),
                                                           p["W"], p.get("KS", 1))
    if kind == "line" and p.get("KS", 1) > 1:  # k slices across workgroups: a workspace row
        if epi:
            raise ValueError("k slices take the plain epilogue only")
        return "launch_line_ks<%d,%d,%d,%d,%d,%d>" % (p["MB"], p["R"], p["D"], p.get("SN", 1),
                                                      p["W"], p["KS"])
    if kind == "line":
        return "launch_line<%d,%d,%d,%d,%d%s>" % (p["MB"], p["R"], p["D"], p.get("SN", 1), p["W"],
                                                  tail)
    if kind == "shared":
        return "launch_shared<%d,%d,%d,%d,%d%s>" % (p["MB"], p["R"], p["U"], p["SN"],
                                                    p.get("TPB", 1024), tail)
    if kind == "stream":
        return "launch_stream<%d,%d,%d,%d%s>" % (p["MB"], p["R"], p["U"], p.get("A", 0), tail)
    if epi and kind == "ilv" and p.get("PLAN"):  # tile and split count by plan_tiles
        return "launch_ilv_plan_gu<%d,%d,%d>" % (p["GROUP"], p["XCD"], p["RSP"])
    if epi:
        raise ValueError("the fused gate/up epilogue exists for the stream kernels and for plans")
    if kind == "ilv" and p.get("PLAN") and not p.get("SW"):
        return "launch_ilv_plan<%d,%d,%d>" % (p["GROUP"], p["XCD"], p["RSP"])
    if kind == "ilv" and p.get("PLAN"):  # a split-K row of its own: RATE in 1/100
        return "launch_ilv_or_plan<%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d>" % (
            p["BM"], p["BN"], p["BK"], p["WM"], p["WN"], p["STAGES"], p["GROUP"], p["XCD"],
            p["RSP"], p["SW"], p["MINKT"], round(100 * p["RATE"]))
    if kind == "ilv":
        return "launch_ilv<%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d>" % (
            p["BM"], p["BN"], p["BK"], p["WM"], p["WN"], p["STAGES"], p["GROUP"], p["XCD"],
            p["RSP"], p.get("SW", 0), p.get("MINKT", 0))
    if kind == "dma" and p.get("PLAN"):
        return "launch_dma_or_plan<%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d>" % (
            p["BM"], p["BN"], p["BK"], p["WM"], p["WN"], p["STAGES"], p["SWZ"], p["GROUP"],
            p["XCD"], p.get("MS", 32), round(100 * p["RATE"]))
    if kind == "dma":
        return "launch_dma<%d,%d,%d,%d,%d,%d,%d,%d,%d,%d>" % (
            p["BM"], p["BN"], p["BK"], p["WM"], p["WN"], p["STAGES"], p["SWZ"], p["GROUP"],
            p["XCD"], p.get("MS", 32))
    return "launch_mfma<%d,%d,%d,%d,%d,%d,%d,%d,%d>" % (
        p["BM"], p["BN"], p["BK"], p["WM"], p["WN"], p["MS"], p["SWZ"], p["GROUP"], p["XCD"])


def condition(sel, kind, p, m_max, n_min=0, gate_up=False):
    if kind == "line":
        sno = p.get("SN", 1) // 2 if gate_up and p.get("SN", 1) >= 2 else p.get("SN", 1)
        fit = "(p.N %% %d) == 0 && (p.K %% %d) == 0 && p.K <= %d" % (
            sel.STREAM_N_ROWS * p["R"] * sno, sel.LINE_K_STEP, sel.LINE_K_MAX)
        if "NMAX" in p:
            fit += " && p.N < %d" % p["NMAX"]
        if "KMIN" in p:
            fit += " && p.K >= %d" % p["KMIN"]
    elif kind == "stream":
        fit = "(p.N %% %d) == 0 && (p.K %% %d) == 0" % (sel.STREAM_N_ROWS * p["R"],
                                                          sel.STREAM_K_STEP * p["U"])
    elif kind == "shared":
        spw = p["SN"] // 2 if gate_up else p["SN"]  # gate/up: the slab waves pair up
        fit = "(p.N %% %d) == 0 && (p.K %% %d) == 0" % (sel.STREAM_N_ROWS * p["R"] * spw,
                                                          sel.STREAM_K_STEP * p["U"])
    elif kind == "ilv":  # an even number of 32-k substeps; 31-bit panel byte offsets
        fit = "(p.N %% %d) == 0 && (p.K %% %d) == 0 && p.lda <= %d && p.ldb <= %d" % (
            p["BN"] // 2 if gate_up else p["BN"], max(64, p["BK"]), sel.ilv_ld_max(p),
            sel.ilv_ld_max(p))
        if "NMAX" in p:
            fit += " && p.N < %d" % p["NMAX"]
    else:
        fit = "(p.N %% %d) == 0 && (p.K %% %d) == 0" % (p["BN"], p["BK"])
        if "NMAX" in p:
            fit += " && p.N < %d" % p["NMAX"]
    band = "p.M <= %d" % m_max
    if n_min:
        band += " && p.N >= %d" % n_min
    return band, fit


HEAD_GATE_UP = """// GENERATED from select.py (LADDER_GATE_UP) -- do not edit.  Regenerate with:
//   python3 kernels/shipped/gemm_fp16/gfx950/gen_dispatch.py --gate-up > dispatch_gate_up.inc
//
// Fused gate/up ladder: p.N is the output width, the weights hold 2N rows (gate, then up).  Same
// row rule as dispatch.inc; none -> hipErrorInvalidConfiguration.
"""


def render(gate_up: bool = False) -> str:
    sel = _select()
    out = [HEAD_GATE_UP if gate_up else HEAD]
    for m_max, n_min, tag, kind, p in (sel.LADDER_GATE_UP if gate_up else sel.LADDER):
        band, fit = condition(sel, kind, p, m_max, n_min, gate_up)
        out.append("TEMPO_ROW(%s, %s,\n          (%s), \"%s\")"
                   % (band, fit, instantiation(kind, p, 1 if gate_up else 0), tag))
    out.append("TEMPO_FALLBACK_ROW")
    return "\n".join(out) + "\n"


HEAD_PREFILL = """// GENERATED from select.py -- do not edit.  Regenerate with:
//   python3 kernels/shipped/gemm_fp16/gfx950/gen_dispatch.py --prefill > prefill.inc
//
// Explicit instantiations of the interleaved prefill launchers the ladder names; included by
// launch_prefill.hip, the translation unit that builds k_gemm_ilv.
"""


def render_prefill() -> str:
    sel = _select()
    out = [HEAD_PREFILL]
    seen = set()
    for _m, _n, _tag, kind, p, epi in ([r + (0,) for r in sel.LADDER]
                                       + [r + (1,) for r in sel.LADDER_GATE_UP]):
        if kind != "ilv":
            continue
        inst = instantiation(kind, p, epi)
        if inst in seen:
            continue
        seen.add(inst)
        out.append("template hipError_t %s(const GemmParams&, hipStream_t, const Workspace&);"
                   % inst)
    if any(r[4].get("PLAN") for r in sel.LADDER):
        out.append("template bool plan_instead<8,1,8>(const GemmParams&, hipStream_t, const Workspace&, "
                   "const OwnRow&, hipError_t*);")
    return "\n".join(out) + "\n"


HEAD_PLAN = """// GENERATED from select.py (PLAN_TILES) -- do not edit.  Regenerate with:
//   python3 kernels/shipped/gemm_fp16/gfx950/gen_dispatch.py --plan > plan.inc
//
// TEMPO_TILE(index, BM, BN, BK, WM, WN, STAGES, split-K)
// TEMPO_TABLE(M_max, us a round, a split, a MB of partial sums, a million weights, tiles, {tile, us per 1000 k and round
//             (twice)} ...)
"""


def render_plan() -> str:
    sel = _select()
    out = [HEAD_PLAN, "#ifdef TEMPO_TILE"]
    out += ["TEMPO_TILE(%d, %s)" % (i, ", ".join(map(str, t))) for i, t in enumerate(sel.PLAN_TILES)]
    out += ["#endif", "#ifdef TEMPO_TABLE"]
    for m_max, rnd, split, mb, weights, rates in sel.PLAN_TABLES:
        out.append("TEMPO_TABLE(%d, %s, %s, %s, %s, %d, %s)" % (
            m_max, rnd, split, mb, weights, len(rates),
            ", ".join("{%d, {%s, %s}}" % (i, u[0], u[-1]) for i, u in rates)))
    return "\n".join(out + ["#endif"]) + "\n"


def main():
    if "--plan" in sys.argv[1:]:
        sys.stdout.write(render_plan())
    elif "--prefill" in sys.argv[1:]:
        sys.stdout.write(render_prefill())
    else:
        sys.stdout.write(render(gate_up="--gate-up" in sys.argv[1:]))
    return 0


if __name__ == "__main__":
    sys.exit(main())
