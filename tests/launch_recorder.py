"""What the library launches, recorded on the CPU: launch_recorder.c takes the place of the HIP
runtime's entry points in a process of its own, and each call's kernels come back by name.

    record([dict(op=..., M=..., N=..., K=...), ...]) -> one list of launches per call

A call: op 0 = gemm_fp16, 1 / 2 = gemm_w8a16 (formats 1, 2), 3..5 their fused gate/up forms; M, N, K;
optional `entry` ("pool" (default), "ws", "none", "noalloc"; "none" is "ws" without a workspace),
`ws_bytes` (in place of what the shape asks for), `stream` (a handle value), `capture` (true: that
stream is under capture), `pads` (elements added to lda, ldb / ldw, ldc), `odd` (bytes added to the
scale pointer).  Or an attention call: fmha=[B, Sq, Sk, H, Hkv, D, causal], entry "ws" (default) or
"none".  A launch: dict(kernel, args, grid, block, stream, thread, first): `kernel` and the list of
integer template arguments from the device symbol, `first` the first kernel argument (a split-K
reduction's workspace address).
"""
import ctypes as ct
import json
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SCRATCH = 0x7000000000  # the static array of the allocation-free entry point
WS = 0x6000000000       # the caller's workspace


class _Launch(ct.Structure):
    _fields_ = [("name", ct.c_char_p), ("first", ct.c_uint64), ("grid", ct.c_uint32),
                ("block", ct.c_uint32), ("stream", ct.c_void_p), ("thread", ct.c_int)]


def _parse(sym):
    """(name, integer template arguments) of an Itanium-mangled kernel."""
    rest, name = sym[len("_ZN"):], ""
    while rest[0].isdigit():
        n = re.match(r"\d+", rest).group(0)
        name = rest[len(n):len(n) + int(n)]
        rest = rest[len(n) + int(n):]
    args = re.match(r"I((?:L[ibj]\d+E)+)E", rest)
    return name, [int(v) for v in re.findall(r"L[ibj](\d+)E", args.group(1))] if args else []


def _child_load(shim):
    rec = ct.CDLL(shim, mode=ct.RTLD_GLOBAL)
    rec.rec_get.restype = ct.POINTER(_Launch)
    rec.rec_capture.argtypes = [ct.c_void_p]
    from cuda_tempiler_amd import capi

    return rec, capi, capi.lib()


def _child_fmha(capi, L, c):
    B, Sq, Sk, H, Hkv, D, causal = c["fmha"]
    f = 0x100000
    p = capi.TempoFmhaParams(f, f, f, f, None, B, H, Hkv, Sq, Sk, D, 0.1, int(causal),
                             Sq * H * D, H * D, D, Sk * Hkv * D, Hkv * D, D,
                             Sk * Hkv * D, Hkv * D, D, Sq * H * D, H * D, D)
    need = L.tempo_fmha_fwd_workspace_bytes(p) if c.get("entry", "ws") == "ws" else 0
    return L.tempo_fmha_fwd_launch_ws(p, WS if need else None, need, 0x50)


def _child_call(capi, L, c):
    if "fmha" in c:
        return _child_fmha(capi, L, c)
    op, M, N, K = c["op"], c["M"], c["N"], c["K"]
    base, gu = op % 3, op >= 3
    pa, pb, pc = c.get("pads", (0, 0, 0))
    f = 0x100000
    if base == 0:
        p = capi.TempoGemmParams(f, f, f, M, N, K, K + pa, K + pb, N + pc)
    else:
        p = capi.TempoW8A16Params(f, f, f + c.get("odd", 0), f if base == 2 else None, f, M, N, K,
                                  K + pa, K + pb, N + pc, 128 if base == 2 else 0, base)
    name = "tempo_gemm_" + ("fp16" if base == 0 else "w8a16") + ("_gate_up" if gu else "")
    entry, s = c.get("entry", "pool"), c.get("stream", 0x50)
    if entry == "pool":
        return getattr(L, name + "_launch")(p, s)
    if entry == "noalloc":
        return getattr(L, name + "_launch_noalloc")(p, s)
    need = getattr(L, name + "_workspace_bytes")(p) if entry == "ws" else 0
    need = c.get("ws_bytes", need)
    return getattr(L, name + "_launch_ws")(p, WS if need else None, need, s)


def _child_launches(rec):
    out = []
    for i in range(rec.rec_count()):
        l = rec.rec_get(i).contents
        kernel, args = _parse(l.name.decode())
        out.append(dict(kernel=kernel, args=args, first=l.first, grid=l.grid, block=l.block,
                        stream=l.stream or 0, thread=l.thread))
    return out


def _child_sequence(rec, capi, L, calls):
    out = []
    for c in calls:
        rec.rec_reset()
        rec.rec_capture(c.get("stream", 0x50) if c.get("capture") else None)
        rc = _child_call(capi, L, c)
        out.append(dict(rc=rc, launches=_child_launches(rec)))
    return out


def _child_threads(rec, capi, L, job):
    """Every thread makes its call `repeat` times on one stream, all at once."""
    import threading

    rec.rec_delay(job["delay_us"])
    start = threading.Barrier(len(job["calls"]))

    def work(i, c):
        rec.rec_thread(i)
        start.wait()
        for _ in range(job["repeat"]):
            _child_call(capi, L, c)

    ts = [threading.Thread(target=work, args=(i, c)) for i, c in enumerate(job["calls"])]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    return _child_launches(rec)


def _child_main():
    shim = sys.argv[1]
    job = json.load(sys.stdin)
    rec, capi, L = _child_load(shim)
    do = _child_threads if job["mode"] == "threads" else \
        lambda r, c, l, j: _child_sequence(r, c, l, j["calls"])
    json.dump(do(rec, capi, L, job), sys.stdout)


_SHIM = None


def _shim():
    global _SHIM
    if _SHIM is None:
        import atexit
        import shutil
        import tempfile

        d = tempfile.mkdtemp(prefix="launch_recorder")
        atexit.register(shutil.rmtree, d, True)
        _SHIM = os.path.join(d, "librecorder.so")
        subprocess.run(["gcc", "-std=gnu11", "-O1", "-shared", "-fPIC", "-pthread", "-o", _SHIM,
                        os.path.join(HERE, "launch_recorder.c")], check=True)
    return _SHIM


def _run(job):
    r = subprocess.run([sys.executable, "-m", "tests.launch_recorder", _shim()], cwd=ROOT,
                       input=json.dumps(job), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    return json.loads(r.stdout)


def record(calls):
    """One dict(rc, launches) per call, made one after the other in one process."""
    return _run(dict(mode="sequence", calls=calls))


def record_threads(calls, repeat=20, delay_us=500):
    """The launches of one thread per call, each making its call `repeat` times."""
    return _run(dict(mode="threads", calls=calls, repeat=repeat, delay_us=delay_us))


def own_kernel(row, fmt, gu):
    """(kernel, leading template arguments) of a row's own kernel."""
    kind, p = row[3], row[4]
    epi = int(gu)
    if kind in ("ilv", "ilv8", "dma", "mfma"):
        name = {"ilv": "k_gemm_ilv", "ilv8": "k_gemm_ilv8", "dma": "k_gemm_dma",
                "mfma": "k_gemm"}[kind]
        return name, [p[k] for k in ("BM", "BN", "BK", "WM", "WN")] + (
            [p["STAGES"]] if kind != "mfma" else [])
    if kind == "line":
        tpb = 512 if p["MB"] >= 4 else 1024
        if p.get("MT"):
            return "k_stream_line", [p["MB"], p["R"], p["D"], fmt, 0, 1, 64 * p["S"], 0]
        return "k_stream_line", [p["MB"], p["R"], p["D"], fmt, epi, p.get("SN", 1), tpb,
                                 p.get("TL", 0)]
    if kind == "phase":
        return "k_stream_phase", [p["MB"], p["NS"], p["D"], fmt, epi, int(p.get("KS", 1) > 1)]
    if kind == "stream":
        return "k_stream", [p["MB"], p["R"], p["U"], fmt]
    return "k_stream_sh", [p["MB"], p["R"], p["U"], fmt, p["SN"]]


if __name__ == "__main__":
    _child_main()
