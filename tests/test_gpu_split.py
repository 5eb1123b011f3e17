"""Causal fp32 ops on split operands (cott_split.h): widths below their padding, ragged lengths on either side of a chunk of 32 and
of the one-group limits, infinite entries."""
import pytest
import torch

from util import inputs, rel_l2, worst_block

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32 = torch.float32


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


# With three terms a product misses at most 1.5 2^-23 of it, of either sign (2^-26 rms), and the fp32 sums round.  A result passes at most N / 32 additions to its
# state and about 50 sums within a chunk and between groups; with independent roundings of 2^-25 rms that is
# 2^-25 sqrt(4200 / 32 + 50) = 4e-7, taken twice over for the worst block.
CASES = [(1, 1, 1, 80, 96), (1, 2, 31, 128, 64), (1, 2, 33, 64, 128), (2, 3, 65, 112, 128), (1, 2, 128, 128, 128), (1, 2, 129, 128, 128),
         (1, 16, 256, 128, 96), (1, 16, 257, 96, 96), (2, 20, 100, 80, 48), (1, 3, 4100, 128, 128), (1, 2, 700, 48, 80)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_three_terms_keep_fp32_precision(ct, oracle, case):
    q, k, v, do = inputs(*case, F32, seed=case[2])
    dev = [t.to(DEV) for t in (q, k, v, do)]
    for rev in (False, True):
        got, ref = ct.causal_dot_product(*dev[:3], rev), oracle.causal(q, k, v, rev)
        assert rel_l2(got, ref) <= 4e-7 and worst_block(got, ref) <= 8e-7, rev
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.causal_backward(*dev), oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= 4e-7 and worst_block(got, ref) <= 8e-7, name


# dV starts from the sums of dK's groups, transposed: widths that differ below the same padding, a group or two, many, last ones
# short.  Two terms: a product misses lo lo and the rounding of both lo, 3 x 2^-18 of it, and the masked scores are split again.
# A last block of one position holds gradients of one score: what its products miss is relative to their magnitudes, not their sum.
@pytest.mark.parametrize("case", [(1, 2, 2100, 80, 112), (1, 16, 300, 112, 80), (1, 3, 2100, 48, 64), (2, 4, 1030, 64, 48),
                                  (1, 24, 640, 64, 64), (1, 24, 641, 64, 64), (1, 2, 192, 128, 128), (1, 2, 193, 128, 128)],
                         ids=lambda c: "x".join(map(str, c)))
def test_gradients_of_grouped_sequences(ct, oracle, case):
    q, k, v, do = inputs(*case, F32, seed=case[2])
    bar = 4e-7 if max(case[3:]) > 64 else 6 * 2.0**-18
    own = [(x[:, :, -1] * y[:, :, -1]).double() for x, y in ((k, q), (v, do))]
    block = max(float((p.abs().sum(-1) / p.sum(-1).abs()).max()) for p in own) if case[2] % 64 == 1 else 2
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.causal_backward(*(t.to(DEV) for t in (q, k, v, do))),
                              oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= bar and worst_block(got, ref) <= block * bar, name


@pytest.mark.parametrize("n,at", [(70, 40), (300, 100)])  # one group; groups, so that sums and prefixes carry the infinity
@pytest.mark.parametrize("which", ["q", "k", "v"])
def test_infinite_entries_of_three_term_ops(ct, which, n, at):
    """One infinite entry: its own row (q) or everything after it is infinite or no number exactly where 64-bit arithmetic has
    it, with the same sign, and the rest is as precise as ever.  Whole numbers, whose lower terms are zero, among the others.
    Left out: positions before an infinite value in its block of 16, where a masked score, zero, is multiplied with it."""
    g = torch.Generator().manual_seed(n)
    q, k = (torch.rand(1, 2, n, 128, generator=g) + 0.25 for _ in range(2))
    v = torch.randint(1, 4, (1, 2, n, 128), generator=g).float() * torch.where(torch.rand(1, 2, 1, 128, generator=g) < 0.5, -1.0, 1.0)
    x = {"q": q, "k": k, "v": v}[which]
    x[0, 1, at, 5] = float("inf")
    got = ct.causal_dot_product(q.to(DEV), k.to(DEV), v.to(DEV)).cpu().double()
    q, k, v = q.double(), k.double(), v.double()
    S = torch.zeros(1, 2, 128, 128, dtype=torch.float64)
    want = torch.empty(1, 2, n, 128, dtype=torch.float64)
    for t in range(n):
        S = S + k[:, :, t, :, None] * v[:, :, t, None, :]
        want[:, :, t] = (q[:, :, t, :, None] * S).sum(-2)
    if which == "v":
        before = slice(at // 16 * 16, at)
        got[:, 1, before, 5] = want[:, 1, before, 5]
    finite = torch.isfinite(want)
    assert not finite.all() and torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    assert float((got[finite] - want[finite]).norm() / want[finite].norm()) <= 4e-7


# Operands are rounded to their terms and the state and the scores cut: what the six products leave out is below 2^-24 of a
# product of two operands and 1.5 2^-23 of one with a state or score, 2^-22 over a score and its product with C, of either sign.
# (All terms cut: 2^-21 each, always of the product's sign; 1.0078124, just below 1 + 2^-7, is the worst of that, 1.0039 of this.)
@pytest.mark.parametrize("n", [1, 31, 128])
@pytest.mark.parametrize("x", [1.0078124, 1.00392904, 1.0117187, 1.9921874])
def test_products_at_the_worst_of_their_split(ct, n, x):
    """Every entry the same number: no averaging over different products, and sums of equal numbers err little."""
    t = torch.full((1, 2, n, 128), x, device=DEV)
    want = t[0, 0, 0, 0].double() ** 3 * 128
    s = torch.arange(1, n + 1, device=DEV, dtype=torch.float64)
    for got, count in ((ct.causal_dot_product(t, t, t), s), (ct.causal_dot_product(t, t, t, True), s.flip(0))):
        assert float((got.double() / (want * count)[:, None] - 1).abs().max()) <= 2.0**-22
    for got, count in zip(ct.causal_backward(t, t, t, t), (s, s.flip(0), s.flip(0))):
        assert float((got.double() / (want * count)[:, None] - 1).abs().max()) <= 2.0**-22


def test_products_have_no_bias(ct):
    """Random positive numbers: the mean of the relative errors is far below that of a single rounding (2^-25), where products that
    leave out parts of their own sign are all too small (by 2^-23.6)."""
    g = torch.Generator().manual_seed(0)
    q, k, v = ((torch.rand(1, 4, 128, 128, generator=g) + 1).to(DEV) for _ in range(3))
    want = torch.tril(q.double() @ k.double().transpose(-1, -2).contiguous()) @ v.double()
    assert abs(float((ct.causal_dot_product(q, k, v).double() / want - 1).mean())) <= 2.0**-27


@pytest.mark.parametrize("n,at", [(70, 40), (300, 100)])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_largest_numbers_of_three_term_ops(ct, which, n, at):
    """A finite number whose nearest bf16 number is infinite, in one operand, with others that keep the results finite."""
    g = torch.Generator().manual_seed(n)
    x = [(torch.rand(1, 2, n, 128, generator=g) + 0.5) * 2.0**-40 for _ in range(3)]
    x[which][0, 1, at, 5] = 3.4e38
    x[which][0, 1, at, 6] = -3.395e38
    q, k, v = (t.to(DEV) for t in x)
    for rev in (False, True):
        scores = q.double() @ k.double().transpose(-1, -2).contiguous()
        want = (torch.triu(scores) if rev else torch.tril(scores)) @ v.double()
        got = ct.causal_dot_product(q, k, v, rev).double()
        assert torch.isfinite(got).all()
        # entries of very different size: against the magnitudes that were added
        scale = (torch.triu(scores.abs()) if rev else torch.tril(scores.abs())) @ v.double().abs()
        terms = q.double().abs() @ k.double().abs().transpose(-1, -2).contiguous()
        scale = torch.maximum(scale, (torch.triu(terms) if rev else torch.tril(terms)) @ v.double().abs())
        assert float(((got - want).abs() / scale).max()) <= 4e-7
