"""Sequences on either side of the lengths up to which a call runs as one group per head (few heads, one launch) against
the oracle: the last length of the one-group form, one position more, and ragged ones."""
import pytest
import torch

from util import TOL, inputs, rel_l2, worst_block

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


def assert_blocks(got, ref, dt, op=None):
    """Every block of 64 rows, a last partial one among them, within the type's tolerance.  Of fp32 products from split
    operands the tolerance is no bound relative to a row of ONE term (the last row of a sum over the future) whose score
    happens to be small.  There op = (A, B, C) of G(A, B, C, reversed) bounds every row of the partial block absolutely, by
    |A_s| sum |B_s'| |C_s'| times 3 * 2^-17 (two products, each 2^-18 for either split and for the term left out) and
    2^-17 for fp32 sums of 64 + 64 terms."""
    n = ref.shape[2]
    whole = n // 64 * 64
    if op is None or dt is not F32 or whole == n:
        assert worst_block(got, ref) <= TOL[dt]
        return
    if whole:
        assert worst_block(got[:, :, :whole], ref[:, :, :whole]) <= TOL[dt]
    a, b, c = (t[:, :, whole:].double().norm(dim=-1) for t in op)
    bound = a * (b * c).flip(-1).cumsum(-1).flip(-1) * 2.0 ** -15
    err = (got[:, :, whole:].double().cpu() - torch.from_numpy(ref[:, :, whole:])).norm(dim=-1)
    assert (err <= bound).all()


CASES = [(1, 2, 768, 64, 64, BF), (1, 2, 769, 64, 64, HF), (2, 6, 1023, 64, 64, HF), (2, 6, 1025, 64, 64, BF),
         (1, 3, 511, 32, 32, BF), (1, 9, 768, 32, 32, HF), (1, 2, 256, 128, 128, BF), (1, 2, 257, 128, 128, BF),
         (4, 4, 768, 128, 128, HF), (1, 9, 500, 128, 64, BF), (1, 9, 500, 64, 128, BF), (2, 20, 300, 80, 96, HF),
         (1, 2, 256, 64, 64, F32), (1, 16, 512, 64, 64, F32), (1, 17, 513, 48, 64, F32), (2, 2, 127, 32, 64, F32)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + "-" + str(c[5]).split(".")[-1])
def test_all_forms(ct, oracle, case):
    b, h, n, dk, dv, dt = case
    q, k, v, do = inputs(b, h, n, dk, dv, dt, seed=n)
    dev = [t.to(DEV) for t in (q, k, v, do)]
    for rev in (False, True):
        got, ref = ct.causal_dot_product(*dev[:3], rev), oracle.causal(q, k, v, rev)
        assert rel_l2(got, ref) <= TOL[dt], rev
        assert_blocks(got, ref, dt, (q, k, v) if rev else None)
    future = (None, (v, do, q), (k, q, do))  # dK and dV sum over the future
    for name, got, ref, op in zip(("dQ", "dK", "dV"), ct.causal_backward(*dev), oracle.causal_bwd(q, k, v, do), future):
        assert rel_l2(got, ref) <= TOL[dt], name
        assert_blocks(got, ref, dt, op)
    assert rel_l2(ct.noncausal_dot_product(*dev[:3]), oracle.noncausal(q, k, v)) <= TOL[dt]
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.noncausal_backward(*dev), oracle.noncausal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= TOL[dt], "non-causal " + name
    leaves = [t.clone().requires_grad_(True) for t in dev[:3]]  # forward and backward as the autograd function pairs them
    out = ct.CustomAttention.apply(*leaves)
    out.backward(dev[3])
    for name, got, ref in zip(("dQ", "dK", "dV"), leaves, oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got.grad, ref) <= TOL[dt], name
