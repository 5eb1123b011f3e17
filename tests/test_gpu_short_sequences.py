"""Sequences on either side of the lengths up to which a call runs as one group per head (few heads, one launch) against
the oracle: the last length of the one-group form, one position more, and ragged ones."""
import pytest
import torch

from util import TOL, inputs, rel_l2, worst_block as worst_block_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


def worst_block(got, ref):
    """Over whole blocks of 64 rows: of fp32 products from split operands, err <= 3 * 2^-17 |q_s| |k_s'| |v_s'|, which is no
    bound relative to a row of ONE term (the last row, in the reversed direction) whose q . k happens to be small."""
    n = max(got.shape[2] // 64 * 64, 1)
    return worst_block_of(got[:, :, :n], ref[:, :, :n])


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
        assert rel_l2(got, ref) <= TOL[dt] and worst_block(got, ref) <= TOL[dt], rev
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.causal_backward(*dev), oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= TOL[dt] and worst_block(got, ref) <= TOL[dt], name
    assert rel_l2(ct.noncausal_dot_product(*dev[:3]), oracle.noncausal(q, k, v)) <= TOL[dt]
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.noncausal_backward(*dev), oracle.noncausal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= TOL[dt], "non-causal " + name
    leaves = [t.clone().requires_grad_(True) for t in dev[:3]]  # forward and backward as the autograd function pairs them
    out = ct.CustomAttention.apply(*leaves)
    out.backward(dev[3])
    for name, got, ref in zip(("dQ", "dK", "dV"), leaves, oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got.grad, ref) <= TOL[dt], name
