"""Weight gradients of the projections: which are cut into row pieces, and that cutting keeps the sums of the single GEMM."""
import pytest
import torch

DEV = "cuda:0"
BF, HF = torch.bfloat16, torch.float16


def test_row_pieces():
    """Small weights as far as 2048 rows a piece go; larger ones only where a piece has more rows than its fp32 sum is worth."""
    from cottention_transformer_amd.autograd import _row_pieces
    assert [_row_pieces(r, 1024, 1024) for r in (4095, 4096, 8192, 16384, 1 << 16, 6144)] == [1, 2, 4, 8, 16, 2]
    assert [_row_pieces(r, 3072, 1024) for r in (4096, 8192, 16384, 16383)] == [2, 4, 4, 1]
    assert [_row_pieces(16384, out, n) for out, n in ((2304, 768), (1536, 1536), (6144, 2048))] == [8, 4, 1]
    assert [_row_pieces(r, 2048, 2048) for r in (4096, 8192, 16384)] == [1, 2, 2]
    assert [_row_pieces(r, 4608, 1536) for r in (4096, 8192, 16384)] == [1, 2, 2]


# single weights of either side of 1 M elements, several pieces; operands as slices of a wider matrix
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF, HF])
@pytest.mark.parametrize("rows,out,inner,wide", [(4096, 64, 128, 64), (8192, 1024, 1024, 1024), (16384, 2048, 2048, 2048), (16384, 3072, 1024, 3072),
                                                 (8192, 72, 256, 216)])
def test_pieces_keep_fp32_sums(rows, out, inner, wide, dtype):
    """Every second piece nearly takes back what the one before it added: a piece rounded to 16 bits would lose the difference
    (fp16: is infinite).  Sums of R products in fp32 err by at most a few units of 2^-24 sqrt(R) of their magnitude."""
    from cottention_transformer_amd.autograd import _row_pieces, _weight_gradient
    pieces = _row_pieces(rows, out, inner)
    assert pieces > 1
    g = torch.Generator(device=DEV).manual_seed(rows + out)
    x = torch.randn(rows, inner, generator=g, device=DEV).abs().to(dtype) * 4
    gy = torch.randn(rows, wide, generator=g, device=DEV).abs().to(dtype) * 16
    half = rows // pieces
    for p in range(1, pieces, 2):
        x[p * half:(p + 1) * half] = x[(p - 1) * half:p * half]
        gy[p * half:(p + 1) * half] = -gy[(p - 1) * half:p * half]
    gy[-1] += 1
    gy = gy[:, wide - out:]
    with torch.no_grad():
        got = _weight_gradient(gy, x)
    want = gy.double().t() @ x.double()
    magnitude = gy.double().abs().t() @ x.double().abs()
    assert got.dtype == torch.float32 and want.abs().max() > 0
    assert ((got.double() - want).abs() / magnitude).max() <= 4 * 2.0 ** -24 * rows ** 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("e", [256, 2048])
def test_gradients_of_16_bit_parameters_are_rounded_once(e):
    """Parameters in bf16, 8192 and 16384 rows (cut): every gradient is the bf16 number nearest to the sum, but where the sum's own
    error decides; and with a second derivative to record, products that have one."""
    from cottention_transformer_amd.autograd import project
    torch.manual_seed(e)
    rows = 8192 if e == 256 else 16384
    lin = torch.nn.Linear(e, e, bias=False, device=DEV, dtype=BF)
    x = torch.randn(rows, e, device=DEV, dtype=BF, requires_grad=True)
    y, = project(x, lin)
    g = torch.randn_like(y)
    got, = torch.autograd.grad(y, lin.weight, g, retain_graph=True)
    want = g.double().t() @ x.detach().double()
    # the share of numbers within the sum's error (about 1e-6 of its magnitude sqrt(R)) of the middle between two bf16 ones
    assert got.dtype == BF and float((got != want.to(BF)).double().mean()) <= 2e-3
    again, = torch.autograd.grad(y, lin.weight, g, create_graph=True)
    assert again.requires_grad and float((again.detach().double() - want).norm() / want.norm()) <= 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("trained", [(0,), (1,), (2,), (0, 2), (0, 1, 2), ()])
def test_frozen_projections_cost_no_gradient(trained, monkeypatch):
    """Weights and biases of the joint form that need no gradient: no product and no sum of their columns, the others' unchanged."""
    from cottention_transformer_amd import autograd, ops
    torch.manual_seed(0)
    rows, e, sizes = 4096, 128, (128, 64, 192)
    lins = [torch.nn.Linear(e, n, device=DEV) for n in sizes]
    x = torch.randn(rows, e, device=DEV)
    gs = [torch.randn(rows, n, device=DEV, dtype=BF) for n in sizes]

    def gradients():
        params = [p for lin in lins for p in lin.parameters() if p.requires_grad]
        with torch.autocast("cuda", dtype=BF):
            ys = autograd.project(x, *lins)
        return torch.autograd.grad(ys, params, gs) if params else ()
    everything = gradients()
    for i, lin in enumerate(lins):
        lin.requires_grad_(i in trained)
    columns = {"w": [], "b": []}
    product, total = autograd._weight_gradient, ops.column_sums
    monkeypatch.setattr(autograd, "_weight_gradient", lambda g, x, *a: (columns["w"].append(g.shape[1]), product(g, x, *a))[1])
    monkeypatch.setattr(ops, "column_sums", lambda g, *a: (columns["b"].append(g.shape[1]), total(g, *a))[1])
    got = gradients()
    assert sum(columns["w"]) == sum(columns["b"]) == sum(sizes[i] for i in trained)
    for a, c in zip(got, [everything[2 * i + j] for i in trained for j in (0, 1)]):
        assert a.shape == c.shape and float((a - c).norm() / c.norm()) <= 1e-5  # the same fp32 sums in another order


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [100, 4096])  # one GEMM; row pieces, whose sum is in the parameters' type already
def test_parameter_gradients_own_their_memory(rows):
    """.grad of each weight and bias of the joint form holds its own numbers and nothing else."""
    from cottention_transformer_amd.autograd import project
    torch.manual_seed(0)
    lins = [torch.nn.Linear(64, n, device=DEV) for n in (64, 32, 64)]
    with torch.autocast("cuda", dtype=BF):
        ys = project(torch.randn(rows, 64, device=DEV), *lins)
    torch.autograd.backward(ys, [torch.randn_like(y) for y in ys])
    params = [p for lin in lins for p in lin.parameters()]
    assert all(p.grad.untyped_storage().nbytes() == 4 * p.numel() and p.grad.is_contiguous() for p in params)
    assert len({p.grad.untyped_storage().data_ptr() for p in params}) == len(params)


@pytest.mark.gpu
@pytest.mark.parametrize("pieces,sizes,width", [(1, [1], 4), (2, [3, 5, 1], 12), (3, [64, 0, 7], 1028), (16, [100], 36), (8, [1024, 1024, 1024], 1024),
                                                (2, [1, 2, 3, 4, 5, 6, 7, 8], 4), (2, [1] * 9, 4), (2, [5], 6)])
def test_add_pieces(pieces, sizes, width):
    """Each block's sum in memory of its own; edges of a thread's four elements and a workgroup's 1024, empty blocks, more blocks or
    odder widths than the kernel takes."""
    from cottention_transformer_amd import ops
    parts = torch.randn(pieces, sum(sizes), width, generator=torch.Generator().manual_seed(pieces)).to(DEV)
    got = ops.add_pieces(parts, sizes)
    assert [tuple(t.shape) for t in got] == [(n, width) for n in sizes]
    for t, block in zip(got, parts.split(sizes, dim=1)):
        # at most 15 additions in fp32
        assert t.untyped_storage().nbytes() == 4 * t.numel()
        assert (t.double() - block.double().sum(0)).abs().le(block.double().abs().sum(0) * 2.0 ** -24 * pieces).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,sizes,ld", [(2, [8], 8), (100, [8, 16, 264], 288), (129, [768, 768, 768], 2304), (5000, [48, 0, 8], 64), (300, [12, 4], 16),
                                           (300, [8] * 9, 72)])
def test_column_sums_in_blocks(rows, sizes, ld):
    """The sums of one array, block by block in memory of their own: few rows (one launch a block), parts, what torch adds."""
    from cottention_transformer_amd import ops
    x = torch.randn(rows, ld, generator=torch.Generator().manual_seed(rows)).to(DEV, BF)[:, :sum(sizes)]
    got, whole = ops.column_sums(x, sizes), ops.column_sums(x)
    assert all(t.untyped_storage().nbytes() == 4 * t.numel() and t.shape == (n,) for t, n in zip(got, sizes))
    bound = x.double().abs().sum(0) * 2.0 ** -24 * 8 + 1e-30  # (as for the whole)
    for t, block, b in zip(got, x.double().sum(0).split(sizes), bound.split(sizes)):
        assert (t.double() - block).abs().le(b).all()
    if rows >= 128 and sum(sizes) % 8 == 0 and len(sizes) <= 8 and all(n % 8 == 0 for n in sizes):
        assert torch.equal(torch.cat(got), whole)


def test_refused_blocks():
    import ctypes
    from cottention_transformer_amd import _loader
    L = _loader.lib()

    def call(f, sizes, *tail, out=0x1000):
        n = len(sizes)
        return f((ctypes.c_void_p * n)(*[out] * n), (ctypes.c_long * n)(*sizes), n, *tail)
    pieces = lambda sizes, p=2, **kw: call(lambda *a: L.cott_add_pieces(0x1000, *a), sizes, p, None, **kw)
    columns = lambda sizes, ld=64, **kw: call(lambda *a: L.cott_column_sums_blocks(0x1000, *a), sizes, 1000, ld, _loader.BF16, None, 0, None, **kw)
    for bad in ([6], [-4], [4] * 9, [4, 2]):
        assert pieces(bad) == _loader.ERR_INVALID
    assert pieces([4], 0) == _loader.ERR_INVALID and pieces([4], out=0x1004) == _loader.ERR_INVALID and pieces([4], out=None) == _loader.ERR_INVALID
    for bad in ([12], [-8], [8] * 9, [72]):
        assert columns(bad) == _loader.ERR_INVALID
    assert columns([8], 12) == _loader.ERR_INVALID and columns([8, 8]) == _loader.ERR_WORKSPACE
    assert pieces([]) == pieces([0]) == columns([]) == _loader.OK


@pytest.mark.parametrize("recording", [False, True])
def test_batched_products_get_no_transposed_right_operand(recording, monkeypatch):
    """Column-major hidden states (one sequence, transposed), and products whose own backward would multiply by such: on the CPU,
    with the batched product replaced."""
    from cottention_transformer_amd import autograd

    class OnGpu(torch.Tensor):
        is_cuda = True
    seen = []

    def bmm(a, b, out_dtype=None):
        seen.append(b.is_contiguous())
        return torch.matmul(a.as_subclass(torch.Tensor).float(), b.as_subclass(torch.Tensor).float())
    monkeypatch.setattr(autograd.torch, "bmm", bmm)
    gy = torch.randn(4096, 8)
    x = torch.randn(16, 4096).t()
    with torch.set_grad_enabled(recording):
        got = autograd._weight_gradient(gy.to(BF).requires_grad_(recording), x.to(BF).as_subclass(OnGpu)).detach()
    want = gy.to(BF).float().t() @ x.to(BF).float()
    assert seen == ([] if recording else [True])
    assert float((got.float() - want).norm() / want.norm()) <= 4e-3
