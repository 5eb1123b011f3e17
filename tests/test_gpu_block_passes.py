"""The small passes of an attention block (cott_block.hip) against torch: edges of tiles, pieces and shares."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def ops():
    from cottention_transformer_amd import ops as ops_
    return ops_


@pytest.mark.parametrize("dtype", [BF, HF])
@pytest.mark.parametrize("sizes", [(1,), (7, 8, 9), (0, 2048, 1, 100003), (8,) * 8, (16,) * 9])
def test_convert(ops, dtype, sizes):
    """Bit for bit what copy_ gives, subnormal, halfway, largest and infinite numbers among them; more arrays than one launch takes."""
    special = torch.tensor([0.0, -0.0, 1 + 2.0 ** -8, 1 + 3 * 2.0 ** -8, 1 + 2.0 ** -11, 3.4e38, -3.4e38, float("inf"), 1e-40, 6e-8, 65519.0, 65520.0])
    srcs = []
    for i, n in enumerate(sizes):
        x = torch.randn(n, generator=torch.Generator().manual_seed(i)) * 100
        x[:min(n, 12)] = special[:min(n, 12)]
        srcs.append(x.to(DEV))
    pairs = [(x, torch.empty(x.shape, dtype=dtype, device=DEV)) for x in srcs]
    ops.convert_into(pairs, dtype)
    for x, y in pairs:
        assert torch.equal(y, x.to(dtype))


def test_convert_of_other_arrays(ops):
    """Strided, unaligned, 64-bit and already converted sources are copied one by one."""
    base = torch.randn(64, 65, device=DEV)
    for src in (base.t(), base.flatten()[1:9], base.double(), base.to(BF)):
        dst = torch.empty(src.shape, dtype=BF, device=DEV)
        ops.convert_into([(base, torch.empty(64, 65, dtype=BF, device=DEV)), (src, dst)], BF)
        assert torch.equal(dst, src.to(BF))


@pytest.mark.parametrize("running", [True, False])
@pytest.mark.parametrize("shape", [(1, 1), (3, 63), (2, 512), (5, 8191), (2, 8193), (1, 40001)])
@pytest.mark.parametrize("dtype", [F32, BF, HF])
def test_keep_and_counts(ops, shape, running, dtype):
    g = torch.Generator().manual_seed(shape[1])
    mask = torch.where(torch.rand(*shape, generator=g) < 0.7, 0.0, torch.finfo(dtype).min)
    mask = torch.where(torch.rand(*shape, generator=g) < 0.1, -0.0, mask).to(DEV, dtype)
    mask[..., -1] = float("nan")
    if dtype is F32 and shape[1] > 2:
        mask[..., 1] = 1e-42  # not zero
    keep, cnt = ops.keep_and_counts(mask[:, None, None, :], *shape, running)
    want = mask == 0
    assert keep.dtype == torch.bool and torch.equal(keep, want)
    total = want.float().cumsum(-1) if running else want.sum(-1, keepdim=True).float().expand(shape)
    assert torch.equal(cnt, total)


def test_masks_of_another_kind(ops):
    mask = torch.zeros(2, 1, 1, 8, device=DEV)
    assert ops.keep_and_counts(mask.double(), 2, 8, True) is None and ops.keep_and_counts(mask.bool(), 2, 8, True) is None
    assert ops.keep_and_counts(mask.expand(2, 1, 8, 8), 2, 8, True) is None and ops.keep_and_counts(mask.cpu(), 2, 8, True) is None
    assert ops.keep_and_counts(torch.zeros(8, 2, device=DEV).t(), 2, 8, True) is None


@pytest.mark.parametrize("rows,cols,ld", [(2, 8, 8), (63, 264, 264), (64, 256, 512), (129, 2304, 2304), (16384, 768, 2304), (5000, 48, 48)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_column_sums(ops, rows, cols, ld, dtype):
    x = torch.randn(rows, ld, generator=torch.Generator().manual_seed(rows)).to(DEV, dtype)[:, :cols]
    got, want = ops.column_sums(x), x.double().sum(0)
    # fp32 sums of n terms in chains of at most a few hundred: well inside 2^-24 sqrt(n) of the terms' magnitude times 8
    bound = x.double().abs().sum(0) * 2.0 ** -24 * 8
    assert got.dtype == F32 and (got.double() - want).abs().le(bound + 1e-30).all()


@pytest.mark.parametrize("b,h,n", [(1, 1, 1), (3, 5, 1000), (8, 16, 2048), (1, 2, 70001)])
def test_head_sums(b, h, n):
    from cottention_transformer_amd import _loader
    x = torch.randn(b, h, n, generator=torch.Generator().manual_seed(n)).to(DEV)
    out = torch.empty(h, device=DEV)
    assert _loader.lib().cott_head_sums(x.data_ptr(), out.data_ptr(), b, h, n, torch.cuda.current_stream().cuda_stream) == 0
    want = x.double().sum((0, 2))
    assert (out.double() - want).abs().le(x.double().abs().sum((0, 2)) * 2.0 ** -24 * 8).all()
