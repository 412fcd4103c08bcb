"""Who may touch a split-K workspace, on the CPU: the library's launches are recorded
(tests/launch_recorder.py) instead of run.

A split-K call is a kernel that writes partial sums and a reduction that reads them.  Two threads
that call on one stream share the pool's buffer, so the pair of one call has to be enqueued without
the other's in between.
"""
import pytest

from tests.launch_recorder import record_threads

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
