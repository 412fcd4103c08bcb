"""GPU parity of the attention forms that are chosen by the row and key counts: the few-rows
kernel, tiles of one and two key groups, and keys cut over several workgroups -- at the edges where
they change (31 / 32 / 33 packed rows, a last key block of one key, tiles whose key counts differ).

Tolerance: against the oracle's fp32 softmax the probabilities are rounded to fp16 before the
second product (relative error uniform in +-2^-11: 2.8e-4 rms if every term erred alike) and O is
rounded to fp16 (2.1e-4 rms in the 2-norm), 3.5e-4 in all; twice that is allowed.  LSE carries
fp32 sums only: 16 ulp at its magnitude of about 10 is 1.5e-5; 3e-5 allowed.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import dev, host, poisoned, say

pytestmark = pytest.mark.gpu

TOL = 7e-4
LSE_TOL = 3e-5

CASES = [
    # B, Sq, Sk, H, Hkv, D, causal
    (1, 1, 1, 2, 2, 128, True),         # one key
    (3, 1, 2049, 8, 2, 256, True),      # a last block of one key
    (2, 31, 640, 1, 1, 128, True),      # 31, 32, 33 packed rows
    (2, 8, 640, 8, 2, 256, False),
    (1, 11, 1100, 6, 2, 128, True),
    (1, 5, 3, 4, 2, 128, True),         # rows without keys
    (2, 33, 2000, 4, 4, 256, True),     # tiles, keys cut
    (1, 130, 1500, 6, 2, 128, True),    # tiles of two key groups, an odd block count, ragged rows
    (1, 300, 513, 4, 2, 128, False),
    (1, 1000, 520, 2, 1, 128, True),    # tiles without keys beside tiles of two key groups
    (70, 40, 77, 8, 8, 128, True),      # one key group: short tiles, more than two per CU
    (4, 38, 104, 8, 2, 256, True),      # a head's rows a tile: few blocks on an idle part
    (1, 16, 203, 32, 4, 256, True),
    (2, 127, 129, 6, 2, 128, False),
    (8, 120, 250, 32, 2, 256, True),    # (B x H at the CUs' count)
]


def _inputs(B, Sq, Sk, H, Hkv, D, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    return [O.f2h(g.standard_normal(s, dtype=np.float32))
            for s in ((B, Sq, H, D), (B, Sk, Hkv, D), (B, Sk, Hkv, D))]


def _check(got, lse, ref, lref):
    assert O.count_poison(got) == 0
    r = O.rel_l2(got, ref)
    inf = np.isneginf(lref)
    d = float(np.max(np.abs(lse[~inf] - lref[~inf]), initial=0.0))
    say("  relL2 %.3e, LSE %.1e" % (r, d))
    assert r <= TOL and np.array_equal(np.isneginf(lse), inf) and d <= LSE_TOL


@pytest.mark.parametrize("case", CASES, ids=lambda c: "b%d_q%d_k%d_h%d_kv%d_d%d_%d" % c)
def test_with_and_without_workspace(gpu, case):
    """capi.fmha_fwd (keys cut where the host finds it worth while) and the entry without a
    workspace (never cut) both meet the oracle."""
    import torch
    from cuda_tempiler_amd import capi

    B, Sq, Sk, H, Hkv, D, causal = case
    Q, K, V = _inputs(B, Sq, Sk, H, Hkv, D, seed=31 * Sq + Sk + D)
    scale = 1.0 / np.sqrt(D)
    ref, lref = O.fmha_fwd(Q, K, V, scale, causal)
    dQ, dK, dV = dev(Q, gpu), dev(K, gpu), dev(V, gpu)
    say("case", case)
    o, l = capi.fmha_fwd(dQ, dK, dV, scale, causal, O=poisoned(Q.shape, gpu))
    torch.cuda.synchronize()
    _check(host(o), host(l), ref, lref)
    o, l = poisoned(Q.shape, gpu), torch.empty((B, H, Sq), dtype=torch.float32, device=gpu)
    p = capi.fmha_params(dQ, dK, dV, o, l, scale, causal)
    capi._check(capi.lib().tempo_fmha_fwd_launch(p, capi._stream(None)), "tempo_fmha_fwd_launch")
    torch.cuda.synchronize()
    _check(host(o), host(l), ref, lref)


STRIDED = [  # case, the kernel and its key groups, whether keys are cut (given a workspace)
    ((2, 1, 4099, 16, 8, 256, True), "k_fmha_rows", None, True),
    ((3, 2, 200, 8, 2, 128, True), "k_fmha_rows", None, False),
    ((2, 31, 4000, 1, 1, 128, False), "k_fmha_rows", None, True),
    ((1, 600, 600, 8, 2, 128, True), "k_fmha_fwd", 2, False),   # first tile: one key block
    ((1, 130, 1500, 6, 2, 128, True), "k_fmha_fwd", 2, True),
    ((2, 33, 2000, 4, 4, 256, True), "k_fmha_fwd", 1, True),
    ((3, 300, 300, 4, 1, 256, True), "k_fmha_fwd", 1, False),
    ((70, 40, 77, 8, 8, 128, True), "k_fmha_fwd", 1, False),
    ((4, 38, 104, 8, 2, 256, True), "k_fmha_fwd", 1, False),    # a head's rows a tile
    ((2, 127, 129, 6, 2, 128, False), "k_fmha_fwd", 1, False),
]


def _layout(x, how, gpu, fill):
    """x [B, S, H, D] on the GPU in a wider buffer whose other elements hold `fill`."""
    import torch

    B, S, H, D = x.shape
    if how == "bhsd":
        buf = torch.full((B, H + 1, S + 5, D), fill, dtype=torch.float16, device=gpu)
        v = buf[:, :H, :S].permute(0, 2, 1, 3)
    else:  # a cache longer than S whose positions also hold other heads
        buf = torch.full((B, S + 37, H + 3, D + 16), fill, dtype=torch.float16, device=gpu)
        v = buf[:, :S, 1:H + 1, 8:8 + D]
    v.copy_(dev(x, gpu))
    return v, buf


@pytest.mark.parametrize("how", ["bhsd", "cache"])
@pytest.mark.parametrize("case", [s[0] for s in STRIDED],
                         ids=lambda c: "b%d_q%d_k%d_h%d_kv%d_d%d_%d" % c)
def test_strides_of_every_form(gpu, case, how):
    """Every operand a view into a wider buffer.  NaN around Q, K and V (the cache past Sk too) must
    not reach the result, and nothing around O may be written."""
    import torch
    from cuda_tempiler_amd import capi

    B, Sq, Sk, H, Hkv, D, causal = case
    Q, K, V = _inputs(B, Sq, Sk, H, Hkv, D, seed=17 * Sq + Sk)
    scale = 1.0 / np.sqrt(D)
    ref, lref = O.fmha_fwd(Q, K, V, scale, causal)
    nan = float("nan")
    (dQ, _), (dK, _), (dV, _) = (_layout(x, how, gpu, nan) for x in (Q, K, V))
    dO, buf = _layout(Q, how, gpu, 7.0)
    say("strided", how, case)
    for ws in (True, False):
        buf.fill_(7.0)
        l = torch.empty((B, H, Sq), dtype=torch.float32, device=gpu)
        if ws:
            capi.fmha_fwd(dQ, dK, dV, scale, causal, O=dO, LSE=l)
        else:
            p = capi.fmha_params(dQ, dK, dV, dO, l, scale, causal)
            capi._check(capi.lib().tempo_fmha_fwd_launch(p, capi._stream(None)), "launch")
        torch.cuda.synchronize()
        _check(host(dO.contiguous()), host(l), ref, lref)
        dO.fill_(7.0)
        assert torch.all(buf == 7.0)


@pytest.mark.parametrize("case", [s[0] for s in STRIDED if s[0][1] > 1],
                         ids=lambda c: "b%d_q%d_k%d_h%d_kv%d_d%d_%d" % c)
def test_special_values_stay_in_their_head(gpu, case):
    """An infinite key in KV head 0 of the first sequence, a NaN query row in its last head: the rows
    that score the key are NaN, as is the query's row.  Rows of another (batch, KV head) have the bits
    they have without them; rows that share a tile with them round against another reference."""
    import torch
    from cuda_tempiler_amd import capi

    B, Sq, Sk, H, Hkv, D, causal = case
    Q, K, V = (dev(x, gpu) for x in _inputs(B, Sq, Sk, H, Hkv, D, seed=3 * Sq + Sk))
    want, lwant = capi.fmha_fwd(Q, K, V, 0.1, causal)
    Q, K = Q.clone(), K.clone()
    G = H // Hkv
    j = Sk - 1 if not causal else Sk - Sq  # a key that every row sees
    j = max(j, 0)
    K[0, j, 0, 5] = float("inf")
    Q[B - 1, Sq // 2, H - 1, 2] = float("nan")
    got, lgot = capi.fmha_fwd(Q, K, V, 0.1, causal)
    torch.cuda.synchronize()
    say("special values", case)
    hit = torch.zeros((B, Sq, H), dtype=torch.bool, device=gpu)
    up = Q[0, :, :G, 5] > 0  # a score of +inf: the row's softmax is NaN (-inf: weight 0)
    hit[0, :, :G] = up
    hit[B - 1, Sq // 2, H - 1] = True
    assert torch.isnan(got[hit]).all()
    clean = torch.ones_like(hit)
    clean[0, :, :G] = False
    clean[B - 1, :, H - G:] = False
    assert torch.equal(got[clean], want[clean])
    if B > 1 or Hkv > 1:  # the query row's neighbours
        near = ~hit[B - 1, :, H - G:]
        a, b = got[B - 1, :, H - G:][near].double(), want[B - 1, :, H - G:][near].double()
        assert float((a - b).norm()) <= TOL * float(b.norm())
    c = clean.permute(0, 2, 1)
    assert torch.equal(lgot[c], lwant[c])
    assert torch.isfinite(got[0, :, :G][~up & ~hit[0, :, :G]]).all()


def test_captured_decode_step(gpu):
    """A decode step whose keys are cut, recorded in a graph: the workspace belongs to the graph's
    pool, and every replay, between eager calls on other data, equals the eager result."""
    import torch
    from cuda_tempiler_amd import capi

    Q, K, V = (dev(x, gpu) for x in _inputs(2, 1, 4000, 8, 2, 128, seed=5))
    want, lwant = capi.fmha_fwd(Q, K, V, 0.1)
    o, l = torch.empty_like(Q), torch.empty_like(lwant)
    p = capi.fmha_params(Q, K, V, o, l, 0.1)
    assert capi.lib().tempo_fmha_fwd_workspace_bytes(p) > 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        capi.fmha_fwd(Q, K, V, 0.1, O=o, LSE=l)
    for _ in range(3):
        o.zero_()
        l.zero_()
        g.replay()
        capi.fmha_fwd(Q, V, K, 0.1)
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(l, lwant)
