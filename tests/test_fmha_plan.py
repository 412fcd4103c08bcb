"""Host side of the attention workspace (CPU only): which calls ask for one, and how much."""
import pytest

from cuda_tempiler_amd import capi


def _need(B, Sq, Sk, H, Hkv, D, causal=1):
    f = capi._p(0x1000)
    p = capi.TempoFmhaParams(f, f, f, f, None, B, H, Hkv, Sq, Sk, D, 0.1, causal,
                             Sq * H * D, H * D, D, Sk * Hkv * D, Hkv * D, D,
                             Sk * Hkv * D, Hkv * D, D, Sq * H * D, H * D, D)
    return capi.lib().tempo_fmha_fwd_workspace_bytes(p)


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,D", [
    (1, 4096, 4096, 16, 8, 256),   # 512 tiles: the part is full
    (64, 1, 2048, 32, 8, 128),     # 512 workgroups of the few-rows kernel
    (1, 1, 96, 16, 8, 128),        # three key blocks: nothing to cut
    (1, 1, 4096, 16, 8, 64),       # not covered
])
def test_calls_without_a_workspace(B, Sq, Sk, H, Hkv, D):
    assert _need(B, Sq, Sk, H, Hkv, D) == 0


def test_strided_gpu_cases_reach_every_form():
    """The GPU cases on strided operands run the kernel they are listed with, cut where they say."""
    from tests.launch_recorder import record
    from tests.test_gpu_fmha_ranges import STRIDED

    met = set()
    for (case, kernel, groups, cut), g in zip(STRIDED, record([dict(fmha=s[0]) for s in STRIDED])):
        first = g["launches"][0]
        assert g["rc"] == 0 and first["kernel"] == kernel and len(g["launches"]) == 1 + cut, case
        assert groups is None or first["args"][2] == groups, case
        met.add((kernel, case[5], groups, cut))
    assert len(met) == 8


@pytest.mark.parametrize("case,tiles", [
    ((4, 38, 104, 8, 2, 256, True), 4 * 8),        # a head's rows a tile
    ((2, 127, 129, 6, 2, 128, False), 2 * 6),
    ((8, 32, 250, 32, 2, 256, True), 8 * 32),      # ... B x H at the CUs' count
    ((9, 40, 60, 32, 2, 256, True), 9 * 2 * 5),    # past it: 16 heads' rows packed, 5 tiles of 128
    ((4, 128, 104, 8, 2, 256, True), 4 * 2 * 4),   # whole tiles either way: packed
    ((1, 187, 187, 8, 4, 256, True), 8 * 2),       # a short last tile, the longest one
    ((1, 187, 187, 8, 4, 256, False), 4 * 3),      # every tile as long: packed
    ((1, 8, 96, 4, 1, 256, True), 4),              # few rows, few blocks: not the few-rows kernel
    ((1, 8, 160, 4, 1, 256, True), 1),             # its five blocks: that kernel
    ((4, 38, 104, 8, 8, 256, True), 4 * 8),        # nothing to pack
    ((32, 107, 107, 8, 1, 256, True), 32 * 7),     # a full part: packed tiles bring in fewer keys
    ((2, 101, 101, 16, 2, 128, True), 2 * 2 * 7),  # packed causal tiles are shorter
    ((2, 40, 101, 16, 2, 128, True), 2 * 16),
])
def test_which_tiles_pack_heads(case, tiles):
    """Without a workspace: one workgroup per (batch, head group, tile)."""
    from tests.launch_recorder import record

    g = record([dict(fmha=case, entry="none")])[0]
    assert [l["grid"] for l in g["launches"]] == [tiles] and g["rc"] == 0


@pytest.mark.parametrize("causal", [0, 1])
def test_workspace_holds_whole_ranges_and_is_bounded(causal):
    """splits x rows x (D + 2) floats, 2..64 splits, and splits x tiles within one round of the
    256 CUs: at most 256 x 128 rows' partial results (33.8 MB at D = 256)."""
    cut = 0
    for D in (128, 256):
        for B in (1, 2, 7):
            for H, Hkv in ((8, 8), (16, 2), (32, 8)):
                for Sq in (1, 4, 33, 500):
                    for Sk in (64, 511, 4096, 30000):
                        need = _need(B, Sq, Sk, H, Hkv, D, causal)
                        unit = B * H * Sq * (D + 2) * 4
                        assert need % unit == 0 and need // unit <= 64
                        assert need // unit != 1 and need <= 256 * 128 * (D + 2) * 4
                        cut += need > 0
    assert cut > 0
