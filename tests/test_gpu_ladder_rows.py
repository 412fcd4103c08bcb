"""GPU parity of every row of the shipped ladders (cases in tests/ladder_cases.py, whose coverage
of the ladders tests/test_ladder_coverage.py checks on the CPU).

Each case: the compiled dispatcher must route it to the row the case names; every output cell
must be written (0x7f7f poison gone, reference harness.cu:50-57); the whole output must match the
oracle within relL2 3e-3 (the north star's bar for fp16 outputs), and fp16 GEMM cases also pass
the reference's fp64 spot rule on 256 sampled cells (ship_probe.cu:70-79).
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests import ladder_cases as LC
from tests.gpu_util import dev, host, poisoned, say

pytestmark = pytest.mark.gpu
TOL = 3e-3


def _weights(N, K, fmt, seed, G=128):
    g = np.random.Generator(np.random.PCG64(seed))
    if fmt == 1:
        q = g.integers(-127, 128, (N, K), dtype=np.int16).astype(np.int8)
        s = O.f2h(g.uniform(0.5, 1.5, N).astype(np.float32) / 127)
        return q, s, None
    q = g.integers(0, 256, (N, K), dtype=np.int16).astype(np.uint8)
    s = O.f2h(g.uniform(0.5, 1.5, (N, K // G)).astype(np.float32) / 255)
    z = g.integers(100, 157, (N, K // G), dtype=np.int16).astype(np.uint8)
    return q, s, z


def _check(got, ref, what):
    assert O.count_poison(got) == 0, what + ": unwritten cells"
    r = O.rel_l2(got, ref)
    say("  relL2 %.3e" % r)
    assert r <= TOL, what


@pytest.mark.parametrize("case", LC.FP16, ids=LC.case_id)
def test_fp16_row(gpu, case):
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K = case
    route = capi.route(0, M, N, K)
    say("fp16 row", tag, "M", M, "N", N, "K", K, "route", route)
    assert route == tag
    A = O.randn_f16((M, K), 11 + M, K ** -0.5)
    B = O.randn_f16((N, K), 77 + N, K ** -0.5)
    C = poisoned((M, N), gpu)
    capi.gemm_fp16(dev(A, gpu), dev(B, gpu), C)
    torch.cuda.synchronize()
    got = host(C)
    _check(got, O.gemm_f16(A, B), tag)
    worst, bad = O.spot_fp64(A, B, got, cells=256)
    assert bad == 0, "fp64 spot %.3e" % worst


@pytest.mark.parametrize("case", LC.FP16_STRIDED, ids=LC.case_id)
def test_fp16_row_strided(gpu, case):
    """lda > K, ldb > K, ldc > N (views into wider buffers); ldc = N + 4 leaves every other C row
    8-byte but not 16-byte aligned.  The padding columns of C must stay untouched."""
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K, pa, pb, pc = case
    say("fp16 strided row", tag, "M", M, "N", N, "K", K, "pads", pa, pb, pc)
    assert capi.route(0, M, N, K) == tag
    A = O.randn_f16((M, K), 5, K ** -0.5)
    B = O.randn_f16((N, K), 6, K ** -0.5)
    Aw = np.zeros((M, K + pa), np.float16)
    Aw[:, :K] = A
    Bw = np.zeros((N, K + pb), np.float16)
    Bw[:, :K] = B
    dA, dB = dev(Aw, gpu)[:, :K], dev(Bw, gpu)[:, :K]
    Cw = poisoned((M, N + pc), gpu)
    dC = Cw[:, :N]
    assert dA.stride(0) == K + pa and dB.stride(0) == K + pb and dC.stride(0) == N + pc
    capi.gemm_fp16(dA, dB, dC)
    torch.cuda.synchronize()
    full = host(Cw)
    assert O.count_poison(full[:, N:]) == full[:, N:].size, "padding columns written"
    _check(np.ascontiguousarray(full[:, :N]), O.gemm_f16(A, B), tag)


@pytest.mark.parametrize("case", LC.FP16_GATE_UP, ids=LC.case_id)
def test_fp16_gate_up_row(gpu, case):
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K = case
    route = capi.route(3, M, N, K)
    say("fp16 gate_up row", tag, "M", M, "N", N, "K", K, "route", route)
    assert route == tag
    A = O.randn_f16((M, K), 3 + M, 1.0)
    B = O.randn_f16((2 * N, K), 4 + N, 2 * K ** -0.5)
    C = capi.gemm_fp16_gate_up(dev(A, gpu), dev(B, gpu), C=poisoned((M, N), gpu))
    torch.cuda.synchronize()
    _check(host(C), O.gemm_gate_up_f16(A, B), tag)


@pytest.mark.parametrize("fmt,case", [(f, c) for f in (1, 2) for c in LC.W8[f]],
                         ids=lambda v: v if isinstance(v, int) else LC.case_id(v))
def test_w8a16_row(gpu, fmt, case):
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K = case
    route = capi.route(fmt, M, N, K)
    say("w8a16 fmt", fmt, "row", tag, "M", M, "N", N, "K", K, "route", route)
    assert route == tag
    A = O.randn_f16((M, K), 11 + M, K ** -0.5)
    q, s, z = _weights(N, K, fmt, 77 + N)
    C = poisoned((M, N), gpu)
    capi.gemm_w8a16(dev(A, gpu), dev(q, gpu), dev(s, gpu), dev(z, gpu) if z is not None else None,
                    fmt=fmt, group=128, C=C)
    torch.cuda.synchronize()
    _check(host(C), O.gemm_w8a16(A, q, s, z, 128, fmt), tag)


@pytest.mark.parametrize("fmt,case", [(f, c) for f in (1, 2) for c in LC.W8_GATE_UP[f]],
                         ids=lambda v: v if isinstance(v, int) else LC.case_id(v))
def test_w8a16_gate_up_row(gpu, fmt, case):
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K = case
    route = capi.route(3 + fmt, M, N, K)
    say("w8a16 gate_up fmt", fmt, "row", tag, "M", M, "N", N, "K", K, "route", route)
    assert route == tag
    A = O.randn_f16((M, K), 3 + M, 3 * K ** -0.5)
    q, s, z = _weights(2 * N, K, fmt, 9 + N)
    s = O.f2h(O.h2f(s) * 2)
    C = capi.gemm_w8a16_gate_up(dev(A, gpu), dev(q, gpu), dev(s, gpu),
                                dev(z, gpu) if z is not None else None, fmt=fmt, group=128,
                                C=poisoned((M, N), gpu))
    torch.cuda.synchronize()
    _check(host(C), O.gemm_gate_up_w8a16(A, q, s, z, 128, fmt), tag)


def _strided_w8(gpu, A, q, s, z, M, N, K, pa, pb, pc):
    """A, q as views into buffers pa / pb wider, C a view pc columns narrower than its buffer."""
    Aw = np.zeros((M, K + pa), np.float16)
    Aw[:, :K] = A
    qw = np.zeros((q.shape[0], K + pb), q.dtype)
    qw[:, :K] = q
    dA, dq = dev(Aw, gpu)[:, :K], dev(qw, gpu)[:, :K]
    Cw = poisoned((M, N + pc), gpu)
    dC = Cw[:, :N]
    assert dA.stride(0) == K + pa and dq.stride(0) == K + pb and dC.stride(0) == N + pc
    return dA, dq, dev(s, gpu), (dev(z, gpu) if z is not None else None), Cw, dC


@pytest.mark.parametrize("fmt,case", [(f, c) for f in (1, 2) for c in LC.W8_STRIDED[f]],
                         ids=lambda v: v if isinstance(v, int) else LC.case_id(v))
def test_w8a16_row_strided(gpu, fmt, case):
    """lda > K, ldw > K, ldc > N; the padding columns of C must stay untouched."""
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K, pa, pb, pc = case
    say("w8a16 fmt", fmt, "strided row", tag, "M", M, "N", N, "K", K, "pads", pa, pb, pc)
    assert capi.route(fmt, M, N, K) == tag
    A = O.randn_f16((M, K), 5 + M, K ** -0.5)
    q, s, z = _weights(N, K, fmt, 31 + N)
    dA, dq, ds, dz, Cw, dC = _strided_w8(gpu, A, q, s, z, M, N, K, pa, pb, pc)
    capi.gemm_w8a16(dA, dq, ds, dz, fmt=fmt, group=128, C=dC)
    torch.cuda.synchronize()
    full = host(Cw)
    assert O.count_poison(full[:, N:]) == full[:, N:].size, "padding columns written"
    _check(np.ascontiguousarray(full[:, :N]), O.gemm_w8a16(A, q, s, z, 128, fmt), tag)


@pytest.mark.parametrize("fmt,case", [(f, c) for f in (1, 2) for c in LC.W8_GATE_UP_STRIDED[f]],
                         ids=lambda v: v if isinstance(v, int) else LC.case_id(v))
def test_w8a16_gate_up_row_strided(gpu, fmt, case):
    """The fused gate/up on views into wider buffers (2N weight rows of ldw > K)."""
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K, pa, pb, pc = case
    say("w8a16 gate_up fmt", fmt, "strided row", tag, "M", M, "N", N, "K", K, "pads", pa, pb, pc)
    assert capi.route(3 + fmt, M, N, K) == tag
    A = O.randn_f16((M, K), 7 + M, 3 * K ** -0.5)
    q, s, z = _weights(2 * N, K, fmt, 13 + N)
    s = O.f2h(O.h2f(s) * 2)
    dA, dq, ds, dz, Cw, dC = _strided_w8(gpu, A, q, s, z, M, N, K, pa, pb, pc)
    capi.gemm_w8a16_gate_up(dA, dq, ds, dz, fmt=fmt, group=128, C=dC)
    torch.cuda.synchronize()
    full = host(Cw)
    assert O.count_poison(full[:, N:]) == full[:, N:].size, "padding columns written"
    _check(np.ascontiguousarray(full[:, :N]), O.gemm_gate_up_w8a16(A, q, s, z, 128, fmt), tag)


@pytest.mark.parametrize("case", LC.FP16_GATE_UP_STRIDED, ids=LC.case_id)
def test_fp16_gate_up_row_strided(gpu, case):
    import torch
    from cuda_tempiler_amd import capi

    tag, M, N, K, pa, pb, pc = case
    say("fp16 gate_up strided row", tag, "M", M, "N", N, "K", K, "pads", pa, pb, pc)
    assert capi.route(3, M, N, K) == tag
    A = O.randn_f16((M, K), 7 + M, 1.0)
    B = O.randn_f16((2 * N, K), 13 + N, 2 * K ** -0.5)
    dA, dB, _, _, Cw, dC = _strided_w8(gpu, A, B, A, None, M, N, K, pa, pb, pc)
    capi.gemm_fp16_gate_up(dA, dB, C=dC)
    torch.cuda.synchronize()
    full = host(Cw)
    assert O.count_poison(full[:, N:]) == full[:, N:].size, "padding columns written"
    _check(np.ascontiguousarray(full[:, :N]), O.gemm_gate_up_f16(A, B), tag)


@pytest.mark.parametrize("name,case", [(n, c) for n in sorted(LC.WITHOUT_PLAN)
                                       for c in LC.WITHOUT_PLAN[n]],
                         ids=lambda v: v if isinstance(v, str) else LC.case_id(v))
def test_row_without_its_plan(gpu, name, case):
    """The row's own kernel, where its plan's workspace is not there or lda is past the planned
    tiles' offsets: the workspace is that of the row's own splits."""
    import torch
    from cuda_tempiler_amd import capi
    from tests.test_ladder_coverage import LADDERS
    from tests.test_ladder_kernels import _own_bytes

    tag, M, N, K, pa = case
    op = ["fp16", "w8_fmt1", "w8_fmt2"].index(name)
    row = next(r for r in LADDERS[name][0] if r[2] == tag)
    ws = torch.empty(_own_bytes(row, case), dtype=torch.uint8, device=gpu)
    say(name, "row", tag, "M", M, "N", N, "K", K, "lda pad", pa, "workspace", ws.numel())
    assert capi.route(op, M, N, K) == tag
    A = O.randn_f16((M, K), 11 + M, K ** -0.5)
    dA = dev(A, gpu)
    if pa:
        wide = torch.zeros((M, K + pa), dtype=torch.float16, device=gpu)
        wide[:, :K] = dA
        dA = wide[:, :K]
    C = poisoned((M, N), gpu)
    if op == 0:
        B = O.randn_f16((N, K), 77 + N, K ** -0.5)
        capi.gemm_fp16(dA, dev(B, gpu), C, workspace=ws)
        ref = O.gemm_f16(A, B)
    else:
        q, s, z = _weights(N, K, op, 77 + N)
        capi.gemm_w8a16(dA, dev(q, gpu), dev(s, gpu), dev(z, gpu) if z is not None else None,
                        fmt=op, C=C, workspace=ws)
        ref = O.gemm_w8a16(A, q, s, z, 128, op)
    torch.cuda.synchronize()
    _check(host(C), ref, tag)


SPECIAL = [  # op, M, N, K: planned 64- and 128-row tiles with splits, sliced phase kernel, k slices
    (0, 9, 5120, 5120), (0, 200, 7168, 5120), (1, 15, 5120, 17408), (2, 15, 11264, 13312),
    (2, 50, 2560, 2560), (1, 300, 2560, 2560), (0, 5, 3840, 12288), (3, 100, 2048, 2048),
    (5, 300, 1280, 4096),
]


@pytest.mark.parametrize("case", SPECIAL, ids=lambda c: "op%d-m%d-n%d-k%d" % c)
def test_special_values_stay_in_their_row(gpu, case):
    """An infinity and a NaN in two rows of A, and the lowest and largest fp16 value in a third:
    their own rows of C are infinite or NaN where the exact product is (with the infinity's sign),
    and every other row has the bits it has without them -- the rows past M that a tile pads with
    included."""
    import torch
    from cuda_tempiler_amd import capi

    op, M, N, K = case
    fmt, gu = op % 3, op >= 3
    rows = 2 * N if gu else N
    A = dev(O.randn_f16((M, K), 5, K ** -0.5), gpu)
    if fmt == 0:
        B = dev(O.randn_f16((rows, K), 6, 1.0), gpu)
        W = B.double()
        run = lambda x: (capi.gemm_fp16_gate_up if gu else capi.gemm_fp16)(x, B)  # noqa: E731
    else:
        q, s, z = _weights(rows, K, fmt, 7)
        dq, ds, dz = dev(q, gpu), dev(s, gpu), dev(z, gpu) if z is not None else None
        f = capi.gemm_w8a16_gate_up if gu else capi.gemm_w8a16
        run = lambda x: f(x, dq, ds, dz, fmt=fmt)  # noqa: E731
        if fmt == 1:
            W = (dq.double() * ds.double()[:, None]).half().double()
        else:
            W = ((dq.view(rows, -1, 128).double() - dz.double()[:, :, None])
                 * ds.double()[:, :, None]).half().double().view(rows, K)
    say("special values", case)
    want = run(A).clone()
    x = A.clone()
    x[1, K // 2 + 3] = float("inf")
    x[3, K - 1] = float("nan")
    x[M - 1, 0], x[M - 1, K - 1] = -65504.0, 65504.0
    got = run(x)
    torch.cuda.synchronize()
    rest = [i for i in range(M) if i not in (1, 3, M - 1)]
    assert torch.equal(got[rest], want[rest])
    assert torch.isnan(got[3]).all()
    if gu:  # silu of an infinity is the epilogue's own affair
        assert not torch.isfinite(got[1]).any()
        return
    y = (x[[1, M - 1]].double() @ W.t()).half()
    assert torch.equal(torch.isnan(got[1]), torch.isnan(y[0]))
    inf = torch.isinf(y[0])
    assert torch.equal(torch.isinf(got[1]), inf) and torch.equal(got[1][inf], y[0][inf])
    # the last row: +-65504 times two weights beside a sum of order 1; fp32 sums of K terms
    big, ref = got[M - 1].double(), y[1].double()
    ok = torch.isfinite(ref) & (ref.abs() < 6e4)
    assert float((big - ref)[ok].norm()) <= 2e-3 * float(ref[ok].norm())
    assert not torch.isnan(big[ok]).any()
