"""W8A16 decode rows that give way to the k-sliced phase kernel (M <= 32): which shapes do, by the
workspace they ask for, and the GPU results against the oracle at its edges: a part slab at the end,
the fewest and the most slabs, slices dealt unevenly to the waves, ragged M, and without a workspace.

Tolerance: fp32 sums in another order, one rounding to fp16 -- 2.1e-4 in the 2-norm (uniform in +-half
an ulp); the oracle rounds its own sums too, so a value whose fp32 sums differ across a rounding
boundary differs by one ulp: 5e-4 allowed.
"""
import pytest

from cuda_tempiler_amd import capi
from oracle import oracle as O
from tests.launch_recorder import record
from tests.test_plan_rows import W8, _dev, _kslices, _weights

SLICED = [  # M, N, K, slices
    (2, 2048, 8192, 8),     # 64 rows a workgroup: 4 slabs
    (16, 3072, 8192, 8),    # 96 rows: 6 slabs
    (17, 4096, 5120, 4),    # 4 slabs, 10 steps over 8 waves
    (32, 5120, 5120, 4),    # 5 slabs
    (24, 3584, 18944, 4),   # 56 rows: a part slab, 37 steps
    (9, 10240, 5120, 4),    # 160 rows: 10 slabs
    (16, 11264, 8192, 2),   # 88 rows: 6 slabs, 32 steps
    (13, 10752, 13312, 2),  # 84 rows: a part slab
    (31, 11264, 5120, 2),
    (32, 10752, 5120, 2),
]
EVEN = [(16, 8192, 8192), (16, 7168, 5120), (32, 5120, 4096)]  # the line grid fills its rounds


def _slices(fmt, M, N, K):
    """phase_slices of launch.h: (slices, slabs) of the k-sliced phase kernel, or None."""
    mb = 1 if M <= 16 else 2
    for ks in (4, 2, 8):
        for ns in range(4, 11):
            if W8.phase_fits(dict(MB=mb, NS=ns, D=4, KS=ks), M, N, K, fmt):
                return ks, ns
    return None


def _choice(fmt, row, M, N, K):
    """(slices, slabs) of the phase kernel where a row runs that, else None (launch_line_or_phase,
    launch_phase_row)."""
    cut = _slices(fmt, M, N, K)
    if row["kind"] == "phase":
        return cut if cut else (row["KS"], row["NS"])
    if not cut:
        return None
    wgs = N // (16 * row["R"] * row["SN"])
    own = _kslices(wgs, K, row["KS"]) if row.get("KS", 1) > 1 else 1
    grid = wgs * own
    idle = N * K / 7.2e6 * (-(-grid // 256) * 256 - grid) / grid
    part = (own - cut[0]) * 2.0 * M * N * 4 / 2.5e6 if own > 1 else 0
    return cut if idle + part > row["PHASE"] else None


@pytest.mark.parametrize("fmt", [1, 2])
def test_sliced_rows_agree(fmt):
    """The rule above and what the library launches, over the rows that may be sliced."""
    shapes = [(M, N, K) for M in (2, 9, 16, 17, 24, 32)
              for N in (2048, 2560, 3072, 3584, 4096, 4736, 5120, 6144, 7168, 8192, 10240, 10752, 11264)
              for K in (2048, 4096, 5120, 5248, 6144, 8192, 12288, 17408, 18944)]
    rows = [(x, W8.select("gemm_w8a16", *x, fmt=fmt)) for x in shapes]
    rows = [(x, r) for x, r in rows if r and r["kind"] in ("line", "phase")
            and ("PHASE" in r or r.get("KS", 1) > 1 and r["kind"] == "phase") and not r.get("TL")]
    met = {}
    for (x, r), got in zip(rows, record([dict(op=fmt, M=M, N=N, K=K, entry="ws")
                                         for (M, N, K), _ in rows])):
        want = _choice(fmt, r, *x)
        first, what = got["launches"][0], (fmt, x, r["tag"], want, got)
        assert got["rc"] == 0, what
        if want:
            ks, ns = want
            assert first["kernel"] == "k_stream_phase", what
            assert first["args"] == [1 if x[0] <= 16 else 2, ns, 4, fmt, 0, 1], what
            assert got["launches"][1]["args"] == [ks], what
        else:
            assert first["kernel"] == "k_stream_line", what
        met[want and want[0]] = met.get(want and want[0], 0) + 1
    assert set(met) == {None, 2, 4, 8}, met


@pytest.mark.parametrize("fmt", [1, 2])
def test_which_shapes_are_sliced(fmt):
    got = record([dict(op=fmt, M=M, N=N, K=K, entry="ws") for M, N, K, _ in SLICED])
    for (M, N, K, ks), g in zip(SLICED, got):
        assert [l["kernel"] for l in g["launches"]] == ["k_stream_phase", "k_splitk_reduce"], (M, N, K)
        assert g["launches"][1]["args"] == [ks], (M, N, K)
        assert capi.workspace_bytes(fmt, M, N, K) >= ks * M * N * 4, (M, N, K)
    for M, N, K in EVEN:
        assert capi.workspace_bytes(fmt, M, N, K) == 0, (M, N, K)
    # no slice count divides this K into whole steps
    assert capi.workspace_bytes(fmt, 16, 2048, 8192 + 128) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", SLICED, ids=lambda c: "m%d-n%d-k%d-s%d" % c)
@pytest.mark.parametrize("fmt", [1, 2])
def test_sliced_against_oracle(gpu, fmt, case):
    """The pool's workspace, torch's, and scales off their 4-byte alignment (the line row runs);
    none where the line row needs none."""
    import torch
    from tests.gpu_util import host, say

    M, N, K, _ = case
    A = O.randn_f16((M, K), 3 + M, K ** -0.5)
    q, s, z = _weights(fmt, N, K, 7)
    ref = O.gemm_w8a16(A, q, s, z, 128, fmt)
    dA, dq, ds, dz = _dev(gpu, A, q, s, z)
    odd = torch.empty(ds.numel() + 1, dtype=ds.dtype, device=gpu)[1:].view(ds.shape)
    odd.copy_(ds)
    assert odd.data_ptr() % 4 == 2
    runs = [("pool", ds, None), ("torch", ds, "torch"), ("odd scale", odd, "torch")]
    row = W8.select("gemm_w8a16", M, N, K, fmt=fmt)
    if row["kind"] == "line" and (row.get("KS", 1) == 1 or _kslices(
            N // (16 * row["R"] * row["SN"]), K, row["KS"]) == 1):
        runs.append(("none", ds, torch.empty(0, dtype=torch.uint8, device=gpu)))
    for what, sc, ws in runs:
        say("fmt", fmt, "case", case, what)
        C = capi.gemm_w8a16(dA, dq, sc, dz, fmt=fmt, workspace=ws)
        torch.cuda.synchronize()
        r = O.rel_l2(host(C), ref)
        say("  relL2 %.3e" % r)
        assert r <= 5e-4


def test_int8_tail_rows_take_the_phase_kernel_where_it_is_faster():
    """M = 17 .. 32, int8: nine slabs and 4096 <= K < 12288 (gate/up: 3072)."""
    cases = [  # op, N, K, phase
        (1, 34816, 4096, True), (1, 34816, 3072, False), (1, 34816, 1024, False),
        (1, 34816, 11264, True), (1, 34816, 12288, False), (1, 36864, 5120, True),
        (1, 32768, 5120, False), (1, 34816, 4224, False),
        (4, 17408, 3072, True), (4, 17408, 2048, False), (4, 18432, 5120, True),
        (4, 17408, 12288, False), (4, 16384, 5120, False),
    ]
    got = record([dict(op=op, M=M, N=N, K=K) for op, N, K, _ in cases for M in (17, 32)])
    for i, (op, N, K, phase) in enumerate(cases):
        for g in got[2 * i:2 * i + 2]:
            assert [l["kernel"] for l in g["launches"]] == [
                "k_stream_phase" if phase else "k_stream_line"], (op, N, K)
