"""Which projections are converted into one matrix: ordinary tensors of fitting shapes on one device; others are multiplied one by
one, as nn.functional.linear takes them."""
import pytest
import torch

DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32


class Sub(torch.Tensor):
    pass


def test_joint_form():
    from cottention_transformer_amd.autograd import _joint_form
    x = torch.randn(4, 8)
    w = [torch.nn.Parameter(torch.randn(n, 8)) for n in (8, 4)]
    b = [torch.nn.Parameter(torch.randn(n)) for n in (8, 4)]
    none = [None, None]
    assert _joint_form(x, w, b, BF) and _joint_form(x, w, none, BF) and _joint_form(x.to(BF), w, none, BF)
    for bad_w in (w[:1], [w[0], w[1].to(BF)], [w[0], w[1].to("meta")], [w[0], torch.randn(4, 9)], [w[0], torch.randn(8)],
                  [w[0], w[1].detach().as_subclass(Sub)]):
        assert not _joint_form(x, bad_w, none[:len(bad_w)], BF)
    for bad_b in ([b[0], None], [None, b[1]], [b[0], torch.randn(1)], [b[0], torch.randn(1, 4)], [b[0], b[1].to("meta")],
                  [b[0].detach().as_subclass(Sub), b[1]]):
        assert not _joint_form(x, w, bad_b, BF)
    assert not _joint_form(x.as_subclass(Sub), w, b, BF)


@pytest.mark.gpu
def test_a_bias_for_all_outputs():
    """A bias of one element, which linear spreads over the outputs: outputs and gradients as from the layers themselves."""
    from cottention_transformer_amd.autograd import project
    torch.manual_seed(0)
    lins = [torch.nn.Linear(64, 64, device=DEV) for _ in range(3)]
    lins[1].bias = torch.nn.Parameter(torch.full((1,), 3.0, device=DEV))
    x = torch.randn(100, 64, device=DEV)
    with torch.autocast("cuda", dtype=BF):
        got, want = project(x, *lins), [lin(x) for lin in lins]
    g = [torch.randn_like(y) for y in got]
    params = [p for lin in lins for p in lin.parameters()]
    for a, c in zip((*got, *torch.autograd.grad(got, params, g)), (*want, *torch.autograd.grad(want, params, g))):
        assert a.shape == c.shape and float((a.float() - c.float()).norm().detach() / c.float().norm().detach()) <= 1e-2


@pytest.mark.gpu
def test_kernels_take_ordinary_tensors_only():
    """Subclasses and sources of another shape go through torch's own operations."""
    from cottention_transformer_amd import ops
    src, one = torch.randn(64, device=DEV), torch.full((1,), 2.0, device=DEV)
    for x in (src.as_subclass(Sub), one):
        dst = torch.full((64,), -1.0, dtype=BF, device=DEV)
        ops.convert_into([(src, torch.empty(64, dtype=BF, device=DEV)), (x, dst)], BF)
        assert torch.equal(dst, x.as_subclass(torch.Tensor).to(BF).expand(64))
    mask = torch.zeros(2, 8, device=DEV)
    assert ops.keep_and_counts(mask, 2, 8, True) is not None and ops.keep_and_counts(mask.as_subclass(Sub), 2, 8, True) is None
    rows = torch.randn(300, 64, device=DEV).to(BF)
    assert type(ops.column_sums(rows.as_subclass(Sub))) is Sub and type(ops.column_sums(rows)) is torch.Tensor
    parts = torch.randn(2, 8, 4, device=DEV)
    assert type(ops.add_pieces(parts.as_subclass(Sub), [8])[0]) is Sub
