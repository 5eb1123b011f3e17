"""Autocast steps on fp32 tensors: the forward rounds them inside the kernel, the backward reads the bf16 gradient; both bit for
bit what the ops give on converted tensors."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF = torch.float32, torch.bfloat16


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


# widths below their padding, ragged lengths, one chunk, column halves, more workgroups than CUs (two output wavefronts)
@pytest.mark.parametrize("case", [(1, 2, 128, 64, 64), (1, 1, 1, 32, 32), (1, 5, 63, 48, 32), (2, 20, 300, 64, 96), (20, 16, 100, 64, 64),
                                  (20, 16, 65, 48, 128), (8, 16, 1023, 64, 64), (3, 50, 130, 32, 64)],
                         ids=lambda c: "x".join(map(str, c)))
def test_equals_converted_tensors(ct, case):
    from cottention_transformer_amd import _loader, ops
    b, h, n, dk, dv = case
    assert _loader.lib().cott_causal_fwd_f32in_supported(*case) == 1
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(b, h, n, d, generator=g).to(DEV) for d in (dk, dk, dv))
    got, want = ops.causal_dot_product_as(q, k, v, BF), ops.causal_dot_product(q.to(BF), k.to(BF), v.to(BF))
    assert got.dtype == BF and torch.equal(got, want)


def test_other_calls_convert(ct):
    """Sequence groups, wide rows, unaligned and mixed tensors take the conversion; CustomAttention's result is the same."""
    from cottention_transformer_amd import _loader, ops
    assert _loader.lib().cott_causal_fwd_f32in_supported(1, 2, 4096, 64, 64) == 0
    assert _loader.lib().cott_causal_fwd_f32in_supported(8, 16, 256, 128, 128) == 0
    q, k, v = (torch.randn(1, 2, 129 * 64, device=DEV)[..., 64:].contiguous().view(1, 2, 128, 64) for _ in range(3))
    odd = torch.randn(2 * 128 * 64 + 1, device=DEV)[1:].view(1, 2, 128, 64)  # 4 bytes past an aligned address
    for x in (q, odd, q.half().float(), q.double().float().to(BF)):
        got = ops.causal_dot_product_as(x, k, v, BF)
        assert torch.equal(got, ops.causal_dot_product(x.to(BF).clone(), k.to(BF), v.to(BF)))
    with torch.autocast("cuda", dtype=BF):
        out = ct.CustomAttention.apply(q.requires_grad_(True), k, v)
    assert torch.equal(out, ops.causal_dot_product(q.detach().to(BF), k.to(BF), v.to(BF)))
    assert torch.autograd.grad(out.float().sum(), q)[0].dtype == F32


# one group and several (the group-state pass reads d_o too), ragged, widths below their padding
@pytest.mark.parametrize("case", [(1, 2, 128, 64, 64), (1, 1, 1, 48, 64), (1, 2, 700, 64, 48), (2, 20, 100, 48, 48), (1, 3, 4097, 64, 64)],
                         ids=lambda c: "x".join(map(str, c)))
def test_backward_of_a_bf16_gradient(ct, case):
    from cottention_transformer_amd import _loader, ops
    b, h, n, dk, dv = case
    assert _loader.lib().cott_causal_bwd_g16_supported(*case) == 1
    g = torch.Generator().manual_seed(n)
    q, k, v, do = (torch.randn(b, h, n, d, generator=g).to(DEV) for d in (dk, dk, dv, dv))
    do = do.to(BF)
    for layout in (do, do.transpose(1, 2).contiguous().transpose(1, 2)):
        for got, want in zip(ops.causal_backward_from(q, k, v, layout), ops.causal_backward(q, k, v, do.float())):
            assert got.dtype == F32 and torch.equal(got, want)


def test_backward_of_other_gradients_converts(ct):
    from cottention_transformer_amd import _loader, ops
    assert _loader.lib().cott_causal_bwd_g16_supported(1, 2, 128, 64, 128) == 0
    q, k, v = (torch.randn(1, 2, 70, d, device=DEV) for d in (32, 32, 64))
    do = torch.randn(1, 2, 70, 64, device=DEV)
    for g in (do, do.to(BF), do.half()):
        for got, want in zip(ops.causal_backward_from(q, k, v, g), ops.causal_backward(q, k, v, g.float())):
            assert torch.equal(got, want)
    with pytest.raises(RuntimeError, match="prev_grad must have shape"):
        ops.causal_backward_from(q, k, v, do[:, :, :5].to(BF))


def test_strided_inputs_of_other_shapes_are_converted_before_they_are_copied(ct):
    """Transposed fp32 heads of a width the converting forward is not built for: the 16-bit copies and the output are all
    that is allocated (three tensors converted with their strides, three made contiguous, one output)."""
    from cottention_transformer_amd import ops
    q, k, v = (torch.randn(4, 128, 75, 128, device=DEV).transpose(1, 2) for _ in range(3))
    want = ct.causal_dot_product(*(t.bfloat16() for t in (q, k, v)))
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    got = ops.causal_dot_product_as(q, k, v, torch.bfloat16)
    assert torch.equal(got, want)
    assert torch.cuda.max_memory_allocated() - held <= 7.5 * 2 * q.numel()
