"""PLAN rows (tile and split count by an estimate of the time): what the rule says -- plan or the row's
own kernel, which tile, how many splits -- and what the library launches agree over a sweep, and the GPU results meet the oracle where a plan changes: one split and many, the
last split shorter, ragged M against every tile height, N in one 128-column tile, and without a
workspace.

Tolerance: fp32 sums in another order, one rounding to fp16 -- 2.1e-4 in the 2-norm (uniform in +-half
an ulp); the oracle rounds its own sums too, so a value whose fp32 sums differ across a rounding
boundary differs by one ulp: 5e-4 allowed.  Gate/up rounds twice on the way: 1e-3.
"""
import importlib.util
import os

import numpy as np
import pytest

from cuda_tempiler_amd import capi
from oracle import oracle as O
from tests.launch_recorder import own_kernel, record

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _select(op):
    path = os.path.join(ROOT, "kernels", "shipped", op, "gfx950", "select.py")
    spec = importlib.util.spec_from_file_location("sel_plan_" + op, path)
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


F16, W8 = _select("gemm_fp16"), _select("gemm_w8a16")
SWEEP = [(M, N, K) for M in (33, 65, 129, 192, 193, 256, 257, 500, 777, 1536, 2048, 3000)
         for N in (128, 1024, 2560, 3968, 5120, 7168, 17408, 34816) for K in (512, 1152, 5120, 17408)]


def _gate_up_need(fmt, M, N, K):
    f = capi._p(0x1000)
    if fmt == 0:
        return capi.lib().tempo_gemm_fp16_gate_up_workspace_bytes(
            capi.TempoGemmParams(f, f, f, M, N, K, K, K, N))
    return capi.lib().tempo_gemm_w8a16_gate_up_workspace_bytes(
        capi.TempoW8A16Params(f, f, f, f if fmt == 2 else None, f, M, N, K, K, K, N,
                              128 if fmt == 2 else 0, fmt))


def _own(row, M, N, K):
    """Splits of a split-K row's own tile (split_count of the frozen kernel file)."""
    if row["kind"] not in ("ilv", "ilv8") or not row.get("SW"):
        return None
    tiles, kt = -(-M // row["BM"]) * (N // row["BN"]), K // row["BK"]
    sp = min(row["SW"] // tiles, kt // row["MINKT"]) if 2 * tiles <= row["SW"] else 1
    return -(-kt // -(-kt // sp)) if sp > 1 else 1


def _kslices(wgs, K, KS):
    """line_kslices of launch.h."""
    steps, best = K // 128, 1

    def even(ks):
        return wgs * ks / (-(-wgs * ks // 256) * 256)

    for ks in range(2, KS + 1):
        if steps % ks == 0 and steps // ks >= 8 and even(ks) > even(best) + 1e-9:
            best = ks
    return best if even(best) >= even(1) + 0.08 else 1


def _line_us(M, N, K, p):
    """line_us of the fp16 launch.h."""
    sn = p.get("SN", 1)
    wgs = N // (16 * sn)
    ks = _kslices(wgs, K, p["KS"]) if p.get("KS", 1) > 1 else 1
    w = wgs * ks
    rounds = -(-w // 256)
    if p["MB"] == 1 and rounds == 1:
        return 2.5 + 1.5 * w / 256 + (0.89 + 0.037 * M) * K * 1e-3
    if p["MB"] == 1:
        return 5.8 + rounds * (1.1 + 0.029 * M) * K * 1e-3
    return 3 + 0.095 * wgs * K * 2e-6 * (16 * sn + M) * rounds * 256 / w + (5 if ks > 1 else 0)


def _choice(op, row, M, N, K):
    """What a row with a plan runs, given a workspace: (index into PLAN_TILES, splits), "tail", or
    "own"."""
    sel, f = (F16, 0) if op == 0 else (W8, op - 1)
    kind = row["kind"]
    if op and kind == "mfma" and K % 128:
        return "own"
    if kind in ("ilv8", "mfma") and "RATE" not in row:
        _, tile, sp, tail = W8.plan(M, N, K, op)
        return "tail" if tail else (tile, sp)
    plan = sel.plan_tiles(M, N, K, f)
    if kind == "ilv" and not row.get("SW"):
        return F16.plan(M, N, K)[1:]
    if plan is None:
        return "own"
    us, tile, sp = plan
    if kind == "line" and op == 0:
        own, ahead = _line_us(M, N, K, row), 0.88
        if M <= 32 and K % 8192 == 0:
            return "own"
        if row["MB"] == 1:
            bm, bn = sel.PLAN_TILES[tile][:2]
            us = max(us + 0.01 * -(-M // bm) * (N // bn) * sp, 0.46e-6 * N * K)
            ahead = 0.93
    else:
        if kind == "line":
            bm, bn, bk = 16 * row["MB"], 16 * row["R"] * row.get("SN", 1), 128
        else:
            bm, bn, bk = row["BM"], row["BN"], row["BK"]
        own_sp = _own(row, M, N, K) or 1
        rates = row["RATE"] if isinstance(row["RATE"], tuple) else (row["RATE"],)
        rates = row.get("RATES", rates) if own_sp > 1 else rates
        own = sel.tile_us(M, N, K, bm, bn, bk, rates[f], own_sp)
        ahead = 0.95
        if kind == "dma":
            ahead = (0.7 if K % 8192 == 0 else 0.85) if M <= 128 else 0.8 if sp > 1 else 0.95
    return (tile, sp) if us < ahead * own else "own"


def _check(op, shapes):
    """The library's launches against _choice; returns how often each kind of choice was met."""
    sel = F16 if op == 0 else W8
    select = (lambda M, N, K: F16.select("gemm", M, N, K)) if op == 0 else (
        lambda M, N, K: W8.select("gemm_w8a16", M, N, K, fmt=op))
    shapes = [(M, N, K, select(M, N, K)) for M, N, K in shapes]
    shapes = [x for x in shapes if x[3] and x[3].get("PLAN")]
    met = {}
    for (M, N, K, row), got in zip(shapes, record([
            dict(op=op, M=M, N=N, K=K, entry="ws") for M, N, K, _ in shapes])):
        want = _choice(op, row, M, N, K)
        what = (op, M, N, K, row["tag"], want, got)
        assert got["rc"] == 0, what
        names = [l["kernel"] for l in got["launches"]]
        reduces = sum(n.startswith("k_splitk_reduce") for n in names)
        first = got["launches"][0]
        if want == "tail":
            assert names == ["k_gemm_ilv8"] * 2 and first["args"][:2] == [256, 256], what
            key = "tail"
        elif want == "own":
            full = (None, None, row["tag"], row["kind"], row)
            name, args = own_kernel(full, op, False)
            assert names[0] == name and first["args"][:len(args)] == args, what
            key = "own " + row["kind"]
        else:
            tile, sp = want
            bm, bn = sel.PLAN_TILES[tile][:2]
            assert names[0] == ("k_gemm_ilv" if op == 0 else "k_gemm_ilv8"), what
            assert tuple(first["args"][:6]) == sel.PLAN_TILES[tile][:6], what
            assert first["grid"] == -(-M // bm) * (N // bn) * sp and reduces == (sp > 1), what
            need = capi.workspace_bytes(op, M, N, K)
            assert need == (0 if sp == 1 else sp * M * N * 4) <= W8.PLAN_WS, what
            key = "split" if sp > 1 else "unsplit"
        met[key] = met.get(key, 0) + 1
    return met


@pytest.mark.parametrize("fmt", [1, 2])
def test_w8a16_plans_agree(fmt):
    wide = [(M, N, K) for M in (33, 48, 64) for N in (12288, 15360, 17408) for K in (640, 5120)]
    met = _check(fmt, SWEEP + wide + [(200, 3840, 3904), (256, 5120, 5184)])
    own = {"own line", "own ilv8"} | ({"own mfma"} if fmt == 1 else set())  # fmt 2: whole 128 k
    assert {"split", "unsplit", "tail"} | own <= set(met), met
    for M, N, K in SWEEP:
        row = W8.select_gate_up("gemm_w8a16_gate_up", M, N, K, fmt=fmt)
        if row and row.get("PLAN"):
            _, _, sp, tail = W8.plan(M, N, K, fmt, gate_up=True)
            want = 0 if tail or sp == 1 else sp * M * 2 * N * 4
            assert _gate_up_need(fmt, M, N, K) == want <= W8.PLAN_WS, (M, N, K)


def test_fp16_plans_agree():
    few = [(M, N, K) for _, N, K in SWEEP if _ == 33 for M in (2, 8, 16, 17, 24, 32, 48)]
    # (rows 16 KiB apart; 256-row tiles with a nearly empty last round)
    met = _check(0, SWEEP + few + [(16, 4096, 8192), (32, 5120, 16384), (2048, 9216, 3840),
                                   (2048, 17408, 5120), (2048, 9216, 2560), (2048, 10240, 3840),
                                   (2048, 11264, 13824), (3000, 11008, 11008), (65, 15360, 8192)])
    assert F16.plan(2048, 9216, 3840)[1] == 2 and F16.plan(2048, 10240, 3840)[1] == 5
    assert F16.plan(2048, 11264, 13824)[1] == 2 and F16.plan(3000, 11008, 11008)[1] == 5
    assert {"split", "unsplit", "own line", "own dma", "own ilv"} <= set(met), met
    shapes = [x for x in SWEEP + [(74, 17408, 3840), (700, 14464, 4096), (384, 13440, 8192)]
              if (F16.select_gate_up("gemm_gate_up", *x) or {}).get("PLAN")
              and not (x[0] > 128 and W8.tail_split(x[0], x[1], 256, 128))]
    for (M, N, K), got in zip(shapes, record([dict(op=3, M=M, N=N, K=K, entry="ws")
                                              for M, N, K in shapes])):
        _, tile, sp = F16.plan(M, N, K, gate_up=True)
        first = got["launches"][0]
        assert tuple(first["args"][:6]) == F16.PLAN_TILES[tile][:6], (M, N, K)
        assert len(got["launches"]) == 1 + (sp > 1), (M, N, K)
        assert _gate_up_need(0, M, N, K) == (0 if sp == 1 else sp * M * 2 * N * 4), (M, N, K)
    assert F16.plan(74, 17408, 3840, True)[2] == 1 and F16.plan(700, 14464, 4096, True)[1] == 2


def test_line_row_keeps_its_uint8_rounds():
    """At 32 < M <= 64 one round of the line row streams uint8 weights at 4.4 .. 4.6 us per 1000 k at
    long K; a plan that is not faster than that stays out ((33, 14208, 12928) 57 us against 72)."""
    line = [(33, 14208, 12928), (64, 13696, 13312), (48, 14208, 17408), (50, 13824, 6144),
            (48, 12416, 12032)]
    planned = [(64, 34816, 5120), (48, 20480, 17408), (33, 27648, 13824)]
    for (M, N, K), got in zip(line + planned, record([dict(op=2, M=M, N=N, K=K, entry="pool")
                                                      for M, N, K in line + planned])):
        tag = capi.route(2, M, N, K)
        assert tag == "l4r1n4d3"
        assert (got["launches"][0]["kernel"] == "k_stream_line") == ((M, N, K) in line), (M, N, K)


def test_nearly_empty_last_round_of_256_rows():
    """Up to 48 tiles past the whole rounds 256-row tiles are the faster; past that 192-row ones."""
    shapes = [(2048, 9472, 14080), (2048, 9728, 4352), (2048, 10240, 3584)]
    for (M, N, K), rows, got in zip(shapes, (256, 256, 192), record([
            dict(op=0, M=M, N=N, K=K, entry="pool") for M, N, K in shapes])):
        assert got["launches"][0]["args"][:2] == [rows, 256], (M, N, K)


CASES = [  # M, N, K
    (9, 5120, 2560),     # 64-row tiles, most rows past M (fp16)
    (33, 5120, 1152),
    (64, 34816, 256),    # wide N, unsplit 64-row tiles
    (65, 2560, 2560),
    (128, 34816, 256),
    (129, 1024, 5120),   # one ragged tile row more, many splits
    (193, 2560, 2560),
    (256, 128, 1152),    # one column tile; K of nine 128-k tiles
    (384, 5120, 1152),   # splits of which the last is shorter
    (500, 7168, 640),    # no split
    (700, 2304, 2048),   # 2304 = 9 x 256
]


def _weights(fmt, N, K, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    if fmt == 1:
        q = g.integers(-127, 128, (N, K)).astype(np.int8)
        return q, O.f2h((g.random(N, dtype=np.float32) + 0.5) / 127), None
    q = g.integers(0, 256, (N, K)).astype(np.uint8)
    s = O.f2h((g.random((N, K // 128), dtype=np.float32) + 0.5) / 255)
    return q, s, g.integers(100, 157, (N, K // 128)).astype(np.uint8)


def _dev(gpu, *arrays):
    from tests.gpu_util import dev
    return [None if a is None else dev(a, gpu) for a in arrays]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "m%d-n%d-k%d" % c)
@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_plan_against_oracle(gpu, fmt, case):
    """The pool's workspace, torch's, and none (an unsplit plan; the rows below refuse or run
    their own way) all meet the oracle."""
    import torch
    from tests.gpu_util import host, say

    M, N, K = case
    A = O.randn_f16((M, K), 3 + M, K ** -0.5)
    if fmt == 0:
        B = O.randn_f16((N, K), 5, K ** -0.5)
        ref = O.gemm_f16(A, B)
        dA, dB = _dev(gpu, A, B)
        run = lambda ws: capi.gemm_fp16(dA, dB, workspace=ws)  # noqa: E731
    else:
        q, s, z = _weights(fmt, N, K, 7)
        ref = O.gemm_w8a16(A, q, s, z, 128, fmt)
        dA, dq, ds, dz = _dev(gpu, A, q, s, z)
        run = lambda ws: capi.gemm_w8a16(dA, dq, ds, dz, fmt=fmt, workspace=ws)  # noqa: E731
    none = torch.empty(0, dtype=torch.uint8, device=gpu)
    for ws in (None, "torch") + ((none,) if M > 256 or (fmt and M > 128) else ()):
        say("fmt", fmt, "case", case, "need", capi.workspace_bytes(fmt, M, N, K), "ws", type(ws))
        C = run(ws)
        torch.cuda.synchronize()
        r = O.rel_l2(host(C), ref)
        say("  relL2 %.3e" % r)
        assert r <= 5e-4


GU = [(33, 128, 1152), (100, 2048, 2048), (129, 4864, 1024), (300, 1280, 4096), (600, 1024, 640)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", GU, ids=lambda c: "m%d-n%d-k%d" % c)
@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_gate_up_plan_against_oracle(gpu, fmt, case):
    import torch
    from tests.gpu_util import host, say

    M, N, K = case
    A = O.randn_f16((M, K), 11 + M, K ** -0.5)
    if fmt == 0:
        B = O.randn_f16((2 * N, K), 5, 1.0)
        ref = O.gemm_gate_up_f16(A, B)
        dA, dB = _dev(gpu, A, B)
        p = lambda C: capi.TempoGemmParams(capi._ptr(dA), capi._ptr(dB), capi._ptr(C), M, N, K,  # noqa: E731
                                           K, K, N)
        run, bare = lambda: capi.gemm_fp16_gate_up(dA, dB), capi.lib().tempo_gemm_fp16_gate_up_launch
    else:
        q, s, z = _weights(fmt, 2 * N, K, 9)
        ref = O.gemm_gate_up_w8a16(A, q, s, z, 128, fmt)
        dA, dq, ds, dz = _dev(gpu, A, q, s, z)
        run = lambda: capi.gemm_w8a16_gate_up(dA, dq, ds, dz, fmt=fmt)  # noqa: E731
        bare = capi.lib().tempo_gemm_w8a16_gate_up_launch

        def p(C):
            x = capi.w8a16_params(dA, dq, ds, dz, C, fmt)
            x.N = N
            return x
    C1 = run()
    C2 = torch.empty_like(C1)
    capi._check(bare(p(C2), capi._stream(None)), "bare")
    torch.cuda.synchronize()
    for what, C in (("workspace", C1), ("none", C2)):
        r = O.rel_l2(host(C), ref)
        say("fmt", fmt, "case", case, "need", _gate_up_need(fmt, M, N, K), what, "relL2 %.3e" % r)
        assert r <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [2, 3, 7, 8, 9, 10, 11, 12, 13, 15, 16, 17, 27, 31])
def test_reduction_of_every_remainder(gpu, splits):
    """The reduction takes the splits in eights and then the rest: one 128-column tile of the 64-row
    split-K row, whose split count is K / 512."""
    import torch
    from tests.gpu_util import host, say

    M, N, K = 40, 128, 512 * splits
    assert capi.route(0, M, N, K) == "i64x128k64s4w256"
    assert capi.workspace_bytes(0, M, N, K) == splits * M * N * 4
    A = O.randn_f16((M, K), 3 + splits, K ** -0.5)
    B = O.randn_f16((N, K), 5, 1.0)
    dA, dB = _dev(gpu, A, B)
    C = capi.gemm_fp16(dA, dB)
    torch.cuda.synchronize()
    r = O.rel_l2(host(C), O.gemm_f16(A, B))
    say("splits", splits, "relL2 %.3e" % r)
    assert r <= 5e-4
