"""The three projections of a block as one GEMM: q, k, v as column slices of one tensor through every preparation entry point, bit
for bit as contiguous tensors; the operator's outputs and gradients against nn.Linear."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from cottention_transformer_amd import ops as ops_
    return ops_


def slices(b, n, h, dk, dv, dtype, seed, order=(0, 1, 2)):
    """q, k, v (B,N,H,D) as slices of one (B,N,H*(2 Dk + Dv)) tensor, and contiguous copies."""
    g = torch.Generator().manual_seed(seed)
    whole = torch.randn(b, n, h * (2 * dk + dv), generator=g).to(DEV, dtype)
    views = [t.view(b, n, h, d) for t, d in zip(whole.split((h * dk, h * dk, h * dv), dim=-1), (dk, dk, dv))]
    views = [views[i] for i in order]
    return views, [t.contiguous() for t in views]


def side(b, n, h, dk):
    g = torch.Generator().manual_seed(1)
    keep = torch.rand(b, n, generator=g) < 0.8
    table = torch.randn(n + 3, 16, generator=g)
    return keep.to(DEV), keep.float().cumsum(-1).to(DEV), torch.rand(h, generator=g).to(DEV), table.to(DEV), torch.arange(n, device=DEV)[None]


# one group, column halves, sequence groups, 128-wide rows (colscan_kernel), widths below their padding, odd lengths
CASES = [(2, 100, 3, 64, 64), (8, 2048, 16, 64, 64), (1, 1500, 4, 64, 64), (2, 130, 4, 128, 128), (1, 4100, 2, 128, 128), (3, 77, 2, 48, 32),
         (1, 1, 1, 32, 32), (2, 65, 5, 96, 64)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype", [BF, torch.float16])
def test_slices_of_one_tensor_equal_contiguous_ones(ops, case, dtype):
    b, n, h, dk, dv = case
    strided, packed = slices(*case, dtype, seed=n)
    assert ops._token_stride(*strided, b, h, n, dk, dv) == h * (2 * dk + dv)
    keep, cnt, sig, table, pos = side(b, n, h, dk)
    for x in (strided, packed):
        grads = None
        out = [ops.prepare_inputs(*x, keep, cnt, sig, rotary=(table, pos), bnhd=True, check_positions=False)]
        g = [torch.randn(t.shape, generator=torch.Generator().manual_seed(2)).to(DEV, dtype) for t in out[0]]
        grads = ops.prepare_inputs_backward(*x, *g, keep, cnt, sig, want_dsig=True, rotary=(table, pos), bnhd=True, check_positions=False)
        out.append(grads)
        if ops.fused_preparation_supported(dtype, b, h, n, dk, dv, 16):
            o, prepared, states = ops.causal_dot_product_prepared(*x, keep, cnt, sig, rotary=(table, pos), bnhd=True, merged_heads=True,
                                                                  save_states=True)
            out.append((o, *prepared, *(() if states is None else (states,))))
        if ops.noncausal_fused_preparation_supported(dtype, b, h, n, dk, dv):
            o, prepared = ops.noncausal_dot_product_prepared(*x, keep, cnt, sig, bnhd=True, merged_heads=True)
            out.append((o, *prepared))
        if x is strided:
            first = out
    assert len(first) == len(out) >= 2
    for got, want in zip(first, out):
        assert all(torch.equal(a, c) for a, c in zip(got, want))
    dq, dk_, dv_, _ = first[1]  # ... slices of one tensor again
    assert ops._token_stride(dq, dk_, dv_, b, h, n, dk, dv) == h * (2 * dk + dv) or n * b * h == 1


def test_other_strided_inputs_are_copied(ops):
    """Slices in another order, with a gap, of a transposed tensor, off the alignment: results of contiguous copies."""
    b, n, h, d = 2, 70, 3, 64
    cases = [slices(b, n, h, d, d, BF, 3, order)[0] for order in ((1, 0, 2), (0, 2, 1), (2, 1, 0))]
    wide = torch.randn(b, n, 3 * h * d + 8, device=DEV).to(BF)
    cases.append([t.view(b, n, h, d) for t in wide[..., 8:].split(h * d, dim=-1)])
    cases.append([torch.randn(b, h, n, d, device=DEV).to(BF).transpose(1, 2) for _ in range(3)])
    flat = torch.randn(b * n * 3 * h * d + 1, device=DEV).to(BF)[1:].view(b, n, 3 * h * d)
    cases.append([t.view(b, n, h, d) for t in flat.split(h * d, dim=-1)])
    for x in cases:
        assert ops._token_stride(*x, b, h, n, d, d) == 0
        for got, want in zip(ops.prepare_inputs(*x, bnhd=True), ops.prepare_inputs(*(t.contiguous() for t in x), bnhd=True)):
            assert torch.equal(got, want)


@pytest.mark.parametrize("rows,e,bias", [((3, 70), 96, True), ((2, 2048), 256, False), ((8, 1024), 768, True), ((1, 1), 64, True)])
def test_joint_projections_against_linear(rows, e, bias):
    """Outputs and gradients of project() under autocast against fp64 on the rounded operands; frozen weights; grad of x in fp32
    without a rounding in between."""
    from cottention_transformer_amd.autograd import project
    torch.manual_seed(0)
    lins = [torch.nn.Linear(e, e, bias=bias).to(DEV) for _ in range(3)]
    lins[1].weight.requires_grad_(False)
    x = torch.randn(*rows, e, device=DEV, requires_grad=True)
    with torch.autocast("cuda", dtype=BF):
        ys = project(x, *lins)
    gs = [torch.randn_like(y) for y in ys]
    params = [p for lin in lins for p in lin.parameters() if p.requires_grad]
    got = torch.autograd.grad(ys, [x, *params], gs)
    x64 = x.detach().to(BF).double().requires_grad_(True)
    refs = [torch.nn.Linear(e, e, bias=bias, device=DEV, dtype=torch.float64) for _ in lins]
    for r, lin in zip(refs, lins):
        r.weight.data.copy_(lin.weight.to(BF))
        r.weight.requires_grad_(lin.weight.requires_grad)
        if bias:
            r.bias.data.copy_(lin.bias.to(BF))
    want_y = [r(x64) for r in refs]
    want = torch.autograd.grad(want_y, [x64, *(p for r in refs for p in r.parameters() if p.requires_grad)], [g.double() for g in gs])
    rel = lambda a, c: float((a.detach().double() - c.detach()).norm() / c.detach().norm())
    for y, w in zip(ys, want_y):
        assert y.dtype == BF and y.shape == (*rows, e) and rel(y, w) <= 4e-3  # one rounding to bf16: 2^-9 at most
    assert got[0].dtype == torch.float32 and rel(got[0], want[0]) <= 1e-5     # fp32 sums of exact products
    for a, c in zip(got[1:], want[1:]):
        assert a.dtype == torch.float32 and rel(a, c) <= 4e-3                 # bf16 pieces or result
