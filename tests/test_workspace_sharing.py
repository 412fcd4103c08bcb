"""Who may touch a split-K workspace, on the CPU: the library's launches are recorded
(tests/launch_recorder.py) instead of run.

A split-K call is a kernel that writes partial sums and a reduction that reads them.  Two threads
that call on one stream share the pool's buffer, so the pair of one call has to be enqueued without
the other's in between.
"""
import pytest

from tests.launch_recorder import record, record_threads

PAIRS = [  # one shape of each kind of row that takes the pool
    [dict(op=0, M=16, N=5120, K=5120), dict(op=0, M=512, N=4096, K=3840)],      # planned tiles
    [dict(op=1, M=16, N=10240, K=8192), dict(op=1, M=16, N=2048, K=8192)],      # sliced phase kernel
    [dict(op=2, M=200, N=5120, K=5120), dict(op=2, M=64, N=5120, K=17408)],     # planned, own split
    [dict(op=0, M=5, N=3840, K=12288), dict(op=0, M=64, N=3840, K=15360)],      # k slices, own split
    [dict(op=1, M=7, N=1024, K=5120), dict(op=1, M=128, N=5120, K=17408)],
    [dict(op=2, M=16, N=5120, K=17408), dict(op=2, M=128, N=34816, K=5120)],    # ..., a split tail
]


@pytest.mark.parametrize("calls", PAIRS, ids=lambda c: "-".join(
    "op%d_m%d_n%d_k%d" % (x["op"], x["M"], x["N"], x["K"]) for x in c))
def test_two_threads_on_one_stream_keep_their_pairs(calls):
    for pair in ([calls[0], calls[0]], [calls[1], calls[1]], calls):
        seq = record_threads(pair, repeat=4, delay_us=300)
        last, uses = {}, []  # uses: (position, thread) of every kernel that touches the workspace
        for i, l in enumerate(seq):
            if l["kernel"].startswith("k_splitk_reduce"):
                uses += [(last[l["thread"]], l["thread"]), (i, l["thread"])]
            last[l["thread"]] = i
        assert len(uses) == 16, [l["kernel"] for l in seq]
        order = [t for _, t in sorted(uses)]
        assert order[0::2] == order[1::2], order


@pytest.mark.gpu
@pytest.mark.parametrize("calls", PAIRS, ids=lambda c: "-".join(
    "op%d_m%d_n%d_k%d" % (x["op"], x["M"], x["N"], x["K"]) for x in c))
def test_two_threads_on_one_stream_get_their_own_sums(gpu, calls):
    """Both threads on the default stream and the pool: every result has the bits of the call made
    alone."""
    import threading

    import torch
    from cuda_tempiler_amd import capi
    from tests.gpu_util import say

    def make(c, seed):
        g = torch.Generator(device=gpu).manual_seed(seed)
        M, N, K, op = c["M"], c["N"], c["K"], c["op"]
        x = torch.randn((M, K), generator=g, device=gpu).half()
        if op == 0:
            w = torch.randn((N, K), generator=g, device=gpu).mul_(K ** -0.5).half()
            return lambda C: capi.gemm_fp16(x, w, C), (M, N)
        w = torch.randint(0, 127, (N, K), generator=g, device=gpu,
                          dtype=torch.int8 if op == 1 else torch.uint8)
        shape = (N,) if op == 1 else (N, K // 128)
        s = (torch.rand(shape, generator=g, device=gpu) * K ** -0.5 / 64).half()
        z = torch.full(shape, 64, dtype=torch.uint8, device=gpu) if op == 2 else None
        return lambda C: capi.gemm_w8a16(x, w, s, z, fmt=op, C=C), (M, N)

    runs = [make(c, 3 + i) for i, c in enumerate(calls)]
    want = [f(torch.empty(s, dtype=torch.float16, device=gpu)) for f, s in runs]
    outs = [[torch.zeros(s, dtype=torch.float16, device=gpu) for _ in range(50)] for _, s in runs]
    torch.cuda.synchronize()
    say("two threads", calls)
    ts = [threading.Thread(target=lambda f=f, o=o: [f(C) for C in o])
          for (f, _), o in zip(runs, outs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    for w, o in zip(want, outs):
        assert all(torch.equal(C, w) for C in o)


# Shapes of every kind of row that may take a workspace or do without: planned tiles, planned tiles
# beside a line or LDS-DMA row, the sliced phase kernel beside a line row without slices.
OPTIONAL = [dict(op=o, M=M, N=N, K=K) for o, M, N, K in (
    (0, 8, 5120, 5120), (0, 32, 5120, 5120), (0, 64, 7168, 5120), (0, 128, 7168, 5120),
    (0, 200, 7168, 5120), (0, 512, 4096, 3840), (0, 1024, 1024, 5120),
    (1, 16, 10240, 5120), (2, 16, 10240, 5120), (1, 32, 5120, 5120), (2, 32, 5120, 5120),
    (1, 64, 34816, 5120), (1, 200, 5120, 5120), (2, 256, 5120, 17408), (1, 500, 5120, 5120),
    (2, 1024, 2048, 5120))]
SWEEP = [dict(op=o, M=M, N=N, K=K) for o in (0, 1, 2) for M in (2, 16, 32, 48, 100, 200, 500, 1100)
         for N in (1024, 2048, 3840, 5120, 7168, 10240, 15360) for K in (1024, 5120, 12288)]


def _reduces(r):
    return [l for l in r["launches"] if l["kernel"].startswith("k_splitk_reduce")]


def _where(calls, **how):
    return [dict(c, **how) for c in calls]


def test_optional_splits_take_the_pool_and_the_callers_memory():
    """What the shapes of OPTIONAL are for: a pool or a workspace splits them, none does not."""
    some = [c for c, r, n in zip(OPTIONAL, record(OPTIONAL), record(_where(OPTIONAL, entry="none")))
            if _reduces(r) and n["rc"] == 0 and not _reduces(n)]
    assert len(some) >= 12 and {c["op"] for c in some} == {0, 1, 2}, some


@pytest.mark.parametrize("how", ["noalloc", "captured", "per thread"])
def test_what_can_do_without_shares_nothing(how):
    """Memory that work on another stream may be using -- the static array, the pool of a stream
    under capture (the graph may be replayed anywhere), the pool under the one handle of every
    thread's own stream -- is taken only by rows that refuse to run without a workspace."""
    calls = [c for c in OPTIONAL + SWEEP if how != "noalloc" or c["op"]]
    if how == "noalloc":
        got = record(_where(calls, entry="noalloc"))
    elif how == "captured":  # the stream's pool is warm: every call once before its capture
        both = [x for c in calls for x in (c, dict(c, capture=True))]
        got = record(both)[1::2]
    else:
        got = record(_where(calls, stream=2))  # hipStreamPerThread
    none = record(_where(calls, entry="none"))
    taken = 0
    for c, g, n in zip(calls, got, none):
        assert g["rc"] == 0, c
        if _reduces(g):
            assert n["rc"] != 0, c
            taken += 1
        elif n["rc"] == 0:  # one path without a workspace, whatever the reason
            assert [(l["kernel"], l["args"]) for l in g["launches"]] == [
                (l["kernel"], l["args"]) for l in n["launches"]], c
    assert taken > 10
