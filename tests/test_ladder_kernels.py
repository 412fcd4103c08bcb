"""Every row of every shipped ladder has a GPU parity case that runs the row's own kernel.

A row's tag names the kernel it was written for, but a row may hand a shape to a planned tile or to
the sliced phase kernel, so the tag alone does not say what a case exercises.  Here the library
itself makes each case's call (tests/launch_recorder.py records the launches on the CPU), and the
kernel it launches is compared with the row's parameters.
"""
import pytest

from tests import ladder_cases as LC
from tests.launch_recorder import own_kernel, record
from tests.test_ladder_coverage import LADDERS
from tests.test_plan_rows import _own

OP = {"fp16": 0, "w8_fmt1": 1, "w8_fmt2": 2, "fp16_gate_up": 3, "w8_gate_up_fmt1": 4,
      "w8_gate_up_fmt2": 5}
# rows whose every shape runs by plan(): they have no kernel of their own
PLANNED = {"i256x256k64w4r8", "i8x192x256w1x4k64s3f", "i8x256w1x4k64s3t", "gi128x256k64s3",
           "gi256x256k64w4r8t", "gi8x128x256k128s2", "gi8x256w1x4k64s3t"}


def runs_own(row, fmt, gu, case, launches):
    name, args = own_kernel(row, fmt, gu)
    first = launches[0]
    if first["kernel"] != name or first["args"][:len(args)] != args:
        return False
    if row[3] in ("ilv", "ilv8") and not gu and not row[4].get("TAIL"):
        M, N, K = case[1:4]
        p = dict(row[4], kind=row[3])
        own = _own(p, M, N, K) or 1
        return first["grid"] == -(-M // p["BM"]) * (N // p["BN"]) * own
    if row[3] == "phase" and row[4].get("KS", 1) > 1:
        red = launches[1]["args"][0]
        return red == row[4]["KS"]
    return True


def _own_bytes(row, case):
    """The workspace of a row's own splits."""
    M, N, K = case[1:4]
    sp = _own(dict(row[4], kind=row[3]), M, N, K) or 1
    return sp * M * N * 4 if sp > 1 else 0


def _record(name, cases, **how):
    rows = {r[2]: r for r in LADDERS[name][0]}
    op = OP[name]
    calls = [dict(op=op, M=c[1], N=c[2], K=c[3], **how) for c in cases]
    if how.get("entry") == "ws":
        for call, c in zip(calls, cases):
            call["ws_bytes"] = _own_bytes(rows[c[0]], c)
            call["pads"] = (c[4], 0, 0)
    return [(c, rows[c[0]], g) for c, g in zip(cases, record(calls))]


@pytest.mark.parametrize("name", sorted(LADDERS))
def test_every_row_has_a_case_on_its_own_kernel(name):
    rows, _, cases = LADDERS[name]
    fmt, gu = OP[name] % 3, OP[name] >= 3
    done = _record(name, cases)
    done += _record(name, LC.WITHOUT_PLAN.get(name, []), entry="ws")
    ran = set()
    for c, r, g in done:
        assert g["rc"] == 0, c
        if runs_own(r, fmt, gu, c, g["launches"]):
            ran.add(c[0])
    missing = {r[2] for r in rows} - ran - PLANNED
    assert not missing, "%s: no case runs the own kernel of %s" % (name, sorted(missing))


@pytest.mark.parametrize("name", sorted(LC.WITHOUT_PLAN))
def test_cases_without_a_plan_run_their_rows(name):
    for c, r, g in _record(name, LC.WITHOUT_PLAN[name], entry="ws"):
        assert runs_own(r, OP[name] % 3, False, c, g["launches"]), (c, g)


def test_strided_w8_cases_route_as_named():
    """(test_ladder_coverage.py checks the fp16 ones.)"""
    for name, cases in (("w8_fmt1", LC.W8_STRIDED[1]), ("w8_fmt2", LC.W8_STRIDED[2]),
                        ("fp16_gate_up", LC.FP16_GATE_UP_STRIDED),
                        ("w8_gate_up_fmt1", LC.W8_GATE_UP_STRIDED[1]),
                        ("w8_gate_up_fmt2", LC.W8_GATE_UP_STRIDED[2])):
        route = LADDERS[name][1]
        for tag, M, N, K, pa, pb, pc in cases:
            assert route(M, N, K)["tag"] == tag, (name, M, N, K)
            assert pa % 8 == 0 and pb % (8 if name.startswith("fp16") else 16) == 0 and pc % 4 == 0


def test_counter_step_counts_every_dispatch():
    """A counter pass attributes dispatches to shapes in launch order: the count it expects of a
    call is the count of kernels the compiled dispatch launches."""
    from tempo.plugins.gfx950 import measure_shipped as ms

    for op in ("gemm_fp16", "gemm_w8a16"):
        shapes = list(ms.cases_of(op))
        for (M, N, K, fmt), got in zip(shapes, record([dict(op=fmt, M=M, N=N, K=K, entry="pool")
                                                       for M, N, K, fmt in shapes])):
            assert got["rc"] == 0 and len(got["launches"]) == ms.dispatches_per_launch(
                op, M, N, K, fmt), (op, M, N, K, fmt)
    for S, H, D, Hkv in ms.cases_of("fmha"):
        got, = record([dict(fmha=[1, S, S, H, Hkv, D, 1], entry="pool")])
        assert got["rc"] == 0 and len(got["launches"]) == ms.dispatches_per_launch(
            "fmha", S, H, D, Hkv), (S, H, D, Hkv)
