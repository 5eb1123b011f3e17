"""in_bnhd of the preparation entry points is a flag whatever its value; strides go to entry points of their own."""
import pytest
import torch

DEV = "cuda:0"
FLAGS = (1, -1, 2, 255, 12345, 12352, 1 << 30)


@pytest.mark.skipif(torch.cuda.is_available(), reason="hands over pointers that no kernel may follow")
def test_every_flag_passes_the_checks_without_a_gpu():
    """Where no device answers, a call that passes all checks ends at the launch; a value taken for a stride would be refused or
    be read with."""
    from cottention_transformer_amd import _loader
    L = _loader.lib()
    p = [0x1000 * (i + 1) for i in range(9)]
    for flag in (0, *FLAGS):
        assert L.cott_prep_ex_fwd(*p[:6], *(None,) * 5, 0, 0, flag, 1, 2, 8, 32, 32, _loader.BF16, _loader.BF16, None) == _loader.ERR_HIP
        assert L.cott_prep_ex_bwd(*p, *(None,) * 6, 0, 0, flag, 1, 2, 8, 32, 32, _loader.BF16, _loader.BF16, None) == _loader.ERR_HIP


def test_strides_are_checked():
    from cottention_transformer_amd import _loader
    L = _loader.lib()
    bf = _loader.BF16
    for stride in (0, 1, 56, 63, 65, 100, -64, 12345):  # H * D = 64
        assert L.cott_prep_strided_fwd(*(None,) * 11, 0, 0, stride, 1, 2, 8, 32, 32, bf, bf, None) == _loader.ERR_INVALID
        assert L.cott_prep_strided_bwd(*(None,) * 15, 0, 0, stride, 1, 2, 8, 32, 32, bf, bf, None) == _loader.ERR_INVALID
        assert L.cott_causal_fwd_prep_strided(*(None,) * 12, 0, 0, 0, stride, 0, None, 0, 0, 1, 2, 8, 32, 32, bf, None, 0, None) == _loader.ERR_INVALID
        assert L.cott_noncausal_fwd_prep_strided(*(None,) * 10, stride, 0, 1, 2, 8, 32, 32, bf, None) == _loader.ERR_INVALID
        assert "between positions" in _loader.last_error()
    wide = 1 << 28
    assert L.cott_causal_fwd_prep_strided(*(None,) * 12, 0, 0, 0, wide, 0, None, 0, 0, 1, 2, 8, 32, 32, bf, None, 0, None) == _loader.ERR_UNSUPPORTED
    assert L.cott_noncausal_fwd_prep_strided(*(None,) * 10, wide, 0, 1, 2, 8, 32, 32, bf, None) == _loader.ERR_UNSUPPORTED
    # no positions, no tensors
    assert L.cott_prep_strided_fwd(*(None,) * 11, 0, 0, 64, 1, 2, 0, 32, 32, bf, bf, None) == _loader.OK


@pytest.mark.gpu
def test_every_flag_means_positions_first():
    """Each entry point on (B,N,H,D) tensors: the same results for every nonzero flag."""
    from cottention_transformer_amd import _loader
    L = _loader.lib()
    b, h, n, d, bf = 2, 3, 70, 64, _loader.BF16
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(b, n, h, d, generator=g).to(DEV, torch.bfloat16) for _ in range(3))
    gq, gk, gv = (torch.randn(b, h, n, d, generator=g).to(DEV, torch.bfloat16) for _ in range(3))
    stream = torch.cuda.current_stream().cuda_stream
    ptr = lambda ts: [t.data_ptr() for t in ts]
    ws = torch.empty(max(16, L.cott_causal_workspace_bytes(b, h, n, d, d, bf)), dtype=torch.uint8, device=DEV)
    first = None
    for flag in FLAGS:
        outs = [torch.zeros(b, h, n, d, device=DEV, dtype=torch.bfloat16) for _ in range(3 + 3 + 4 + 4)]
        prep, grads, causal, non = outs[:3], outs[3:6], outs[6:10], outs[10:]
        rcs = [L.cott_prep_ex_fwd(*ptr((q, k, v, *prep)), *(None,) * 5, 0, 0, flag, b, h, n, d, d, bf, bf, stream),
               L.cott_prep_ex_bwd(*ptr((q, k, v, gq, gk, gv, *grads)), *(None,) * 6, 0, 0, flag, b, h, n, d, d, bf, bf, stream),
               L.cott_causal_fwd_prep(*ptr((q, k, v, *causal)), *(None,) * 5, 0, 0, 0, flag, 0, b, h, n, d, d, bf, ws.data_ptr(), ws.numel(), stream),
               L.cott_noncausal_fwd_prep(*ptr((q, k, v, *non)), *(None,) * 3, flag, 0, b, h, n, d, d, bf, stream)]
        assert rcs == [0] * 4, flag
        first = first or outs
        assert all(torch.equal(a, c) for a, c in zip(outs, first)) and all(t.abs().sum() > 0 for t in outs), flag
