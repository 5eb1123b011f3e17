"""Host-side rules that choose a launch form, swept without a GPU: workspaces stay within what the entry points without a
caller's workspace hold, and every call that was accepted has a plan."""
import ctypes
import itertools

import pytest

from cottention_transformer_amd import _loader

BF16, F16 = _loader.BF16, _loader.F16


@pytest.fixture(params=[(256, 8), (64, 2), (38, 1), (304, 8)], ids=lambda g: f"{g[0]}cus-{g[1]}xcds")
def lib(request):
    L = _loader.lib()
    assert L.cott_plan_geometry(*request.param) == _loader.OK
    yield L, request.param
    assert L.cott_plan_geometry(0, 0) == _loader.OK


def test_wide_head_workspace_fits_the_builtin_scratch(lib):
    L, (cus, _) = lib
    for h, n, dk, dv in itertools.product((1, 2, 3, 8, 16, 40, 300), (1, 735, 737, 1024, 5000, 65536), (48, 144, 192, 256), (16, 144, 256, 400)):
        if dk <= 128 and 32 <= dv <= 128:
            continue
        for dt in (BF16, F16):
            fwd = L.cott_causal_workspace_bytes(1, h, n, dk, dv, dt)
            # at most one workgroup per CU, each of whose groups but the last leaves one slot of at most 64 KiB
            assert fwd <= cus * 65536 and fwd <= 48 << 20
            if n <= 736:
                assert fwd == 0


def test_short_sequences_take_no_workspace(lib):
    L, _ = lib
    for h, d in itertools.product((1, 2, 7, 12, 16, 32, 64), (32, 48, 64, 80, 128)):
        for n in (1, 63, 64, 128, 256):
            assert L.cott_causal_workspace_bytes(1, h, n, d, d, BF16) == 0
            assert L.cott_causal_bwd_workspace_bytes(1, h, n, d, d, BF16) == 0
            assert L.cott_noncausal_workspace_bytes(1, h, n, d, d, BF16) == 0
            # no workspace: one group, which is also what the forward with the preparation inside needs
            assert L.cott_noncausal_fwd_prep_supported(1, h, n, d, d, BF16) == 1
            assert L.cott_causal_fwd_f32in_supported(1, h, n, d, d) == (1 if d <= 64 else 0)


def test_preparation_inside_the_forward_keeps_its_shapes(lib):
    """128-wide q / k rows need value tiles of 64 columns: short sequences are not cut into narrower halves."""
    L, _ = lib
    for h, n, dv in itertools.product((1, 2, 8, 16, 32), (1, 64, 256, 500, 768), (64, 80, 128)):
        if n <= 256:
            assert L.cott_causal_fwd_prep_supported(1, h, n, 128, dv, BF16, 64) == 1


def test_narrow_values_beside_wide_rows(lib):
    """128-wide rows with 64 value columns: few heads run as one group of whole problems only as long as that is the faster
    form, and more heads, whose sequences are whole anyway, keep their column halves."""
    L, (cus, _) = lib
    sets, nsets = (ctypes.c_int * 64)(), ctypes.c_int(0)

    def plan(which, h, n):
        assert L.cott_plan_describe(which, 0, 1, h, n, 128, 64, BF16, sets, ctypes.byref(nsets)) == _loader.OK
        return sets[1], sets[2]  # column halves, groups

    for which, h, chunks in ((0, 2, 4), (0, 8, 8), (0, 16, 8), (2, 2, 4), (2, 8, 6), (2, 16, 6)):
        if h * 4 > cus:
            continue
        assert plan(which, h, 64 * chunks) == (1, 1)
        if h * 8 <= cus:  # (room for groups)
            assert plan(which, h, 64 * chunks + 1)[1] > 1
    if cus > 200:
        assert plan(0, cus // 2 - 10, 500) == (2, 1)


def test_where_the_preparation_inside_the_forward_is_preferred(lib):
    """Few heads: up to the measured lengths; many heads: as before, whatever the length; never where it is not supported."""
    L, (cus, _) = lib
    for causal, d, h, chunks in ((1, 32, 8, 8), (1, 64, 8, 4), (1, 64, 16, 6), (1, 128, 8, 1), (0, 32, 8, 6), (0, 64, 8, 4), (0, 64, 16, 6),
                                 (0, 128, 8, 2)):
        if h * 4 > cus:
            continue
        ask = L.cott_causal_fwd_prep_preferred if causal else L.cott_noncausal_fwd_prep_preferred
        for n in (1, 64 * chunks, 64 * chunks + 1):
            assert ask(1, h, n, d, d, BF16, *((0,) if causal else ())) == (n <= 64 * chunks), (causal, d, h, n)
    for h, n, d in itertools.product((1, 8, 100, 130, 512), (1, 64, 300, 512, 1023, 4096), (32, 64, 128)):
        sup = L.cott_noncausal_fwd_prep_supported(1, h, n, d, d, BF16)
        assert L.cott_noncausal_fwd_prep_preferred(1, h, n, d, d, BF16) <= sup
        if h == 512:
            assert L.cott_noncausal_fwd_prep_preferred(1, h, n, d, d, BF16) == sup
            assert L.cott_causal_fwd_prep_preferred(1, h, n, d, d, BF16, 0) == 1
