"""Causal ops of 16-bit heads outside the 32..128 column range (wide_scan_kernel) against the oracle.

Tolerance: inputs are exact, products and sums are fp32, state and scores enter the products with all their bits, so what is
left is the rounding of the output: at most half a unit in the last place of every element, 2^-9 (bf16) and 2^-12 (fp16,
away from its subnormals) of it, plus 2^-13 for the fp32 sums of outputs that cancel."""
import pytest
import torch

from util import inputs, rel_l2, worst_block

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF = torch.bfloat16, torch.float16
BOUND = {BF: 2.0 ** -9 + 2.0 ** -13, HF: 2.0 ** -12 + 2.0 ** -13}


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


CASES = [
    (1, 1, 1, 256, 256, BF),      # one position
    (1, 2, 31, 256, 256, BF),     # less than a chunk
    (1, 2, 32, 160, 160, HF),     # exactly one chunk; last slice half empty
    (2, 3, 33, 192, 192, BF),     # one chunk and one position
    (1, 9, 64, 256, 256, HF),     # two chunks, more heads than XCDs
    (1, 2, 203, 224, 224, BF),    # odd number of chunks, padded contracted dim
    (1, 2, 1000, 256, 256, BF),
    (1, 2, 130, 256, 64, HF),     # the ops of a gradient call differ in padded width
    (1, 2, 130, 64, 256, BF),
    (1, 2, 96, 48, 144, BF),      # contracted dim far below its padding
    (1, 2, 737, 256, 256, BF),    # 24 chunks: the shortest sequence cut into groups
    (1, 2, 736, 256, 256, HF),    # ... and the longest that is not
    (1, 3, 2050, 64, 192, HF),    # groups of unequal length
    (1, 1, 4100, 160, 160, BF),   # sixteen groups forward
    (1, 1, 70, 144, 400, HF),     # seven slices; the gradients contract 400 columns (plain-FMA kernel)
]
IDS = lambda c: "x".join(map(str, c[:5])) + "-" + str(c[5]).split(".")[-1]


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_forward_and_gradients(ct, oracle, case):
    b, h, n, dk, dv, dt = case
    q, k, v, do = inputs(b, h, n, dk, dv, dt, seed=n)
    dev = [t.to(DEV) for t in (q, k, v, do)]
    for rev in (False, True):
        got, ref = ct.causal_dot_product(*dev[:3], rev), oracle.causal(q, k, v, rev)
        assert rel_l2(got, ref) <= BOUND[dt], rev
        assert worst_block(got, ref, 32) <= 2 * BOUND[dt], rev
    for name, got, ref in zip(("dQ", "dK", "dV"), ct.causal_backward(*dev), oracle.causal_bwd(q, k, v, do)):
        assert rel_l2(got, ref) <= BOUND[dt], name


@pytest.mark.parametrize("dk", [144, 192, 256])
@pytest.mark.parametrize("dt", [BF, HF], ids=["bf16", "fp16"])
def test_states_and_scores_take_part_with_all_their_bits(ct, oracle, dt, dk):
    """Two fp32 numbers that differ in the last of their 24 bits cancel to that bit: state entries 1 + 2^-12 + 2^-23 and
    1 + 2^-12 read at position 40 (the next chunk), scores of the same values at position 20 (their own chunk), against
    values that use all the bits of their type.  Every product and partial sum is an fp32 number, so is the output: exact."""
    q, k, v = (torch.zeros(1, 1, 64, d, dtype=dt) for d in (dk, dk, 160))
    last = dk - 1
    c = 1 + 2.0 ** (-7 if dt is BF else -10)
    # columns 0..63: the state; row `last` holds all three terms, row 3 two of them
    for t, (row, x, y) in enumerate(((last, 1, 1), (last, 2.0 ** -12, 1), (last, 2.0 ** -12, 2.0 ** -11), (3, 1, 1), (3, 2.0 ** -12, 1))):
        k[0, 0, t, row] = x
        v[0, 0, t, :64] = y
    q[0, 0, 40, last], q[0, 0, 40, 3] = 4096, -4096
    # columns 64..: the scores of positions 16 and 17 at position 20
    q[0, 0, 20, 8:11] = torch.tensor([1, 1, 2.0 ** -11], dtype=dt)
    k[0, 0, 16, 8:11] = torch.tensor([1, 2.0 ** -12, 2.0 ** -12], dtype=dt)
    k[0, 0, 17, 8:10] = torch.tensor([1, 2.0 ** -12], dtype=dt)
    v[0, 0, 16, 64:], v[0, 0, 17, 64:] = 4096 * c, -4096 * c
    got = ct.causal_dot_product(*(t.to(DEV) for t in (q, k, v))).double().cpu()
    assert (got[0, 0, 40, :64] == 2.0 ** -11).all()
    assert (got[0, 0, 20, 64:] == 2.0 ** -11 * c).all()
    assert torch.equal(got, torch.from_numpy(oracle.causal(q, k, v)))
    # ... and summed over the future
    rev = ct.causal_dot_product(*(t.flip(2).contiguous().to(DEV) for t in (q, k, v)), True).double().cpu()
    assert torch.equal(rev.flip(2), got)


@pytest.mark.parametrize("dt", [BF, HF], ids=["bf16", "fp16"])
def test_states_in_and_out(ct, oracle, dt):
    """A sequence in two calls, the state handed over, equals the sequence in one; the state is held in fp32."""
    q, k, v, _ = inputs(1, 2, 150, 256, 160, dt, seed=7)
    qd, kd, vd = (t.to(DEV) for t in (q, k, v))
    o1, s1 = ct.causal_prefill(qd[:, :, :70], kd[:, :, :70], vd[:, :, :70])
    o2, s2 = ct.causal_prefill(qd[:, :, 70:], kd[:, :, 70:], vd[:, :, 70:], state=s1)
    assert rel_l2(torch.cat((o1, o2), 2), oracle.causal(q, k, v)) <= BOUND[dt]
    # sums of 150 products in fp32: 150 * 2^-24 at the very most
    assert rel_l2(s2, (k.double().transpose(2, 3) @ v.double()).numpy()) <= 150 * 2.0 ** -24


@pytest.mark.parametrize("scale", [2.0 ** -12, 1.0, 2.0 ** 9], ids=["small", "unit", "large"])
def test_fp16_state_range(ct, oracle, scale):
    """Scores, state and their 16-bit halves leave fp16's range on both sides; the outputs (brought back by q) do not:
    values of `scale`, keys of 1 / 16 .. 16 times `scale`."""
    q, k, v, _ = inputs(1, 1, 300, 256, 256, HF, seed=3)
    k, v, q = (k.float() * 16 * scale).half(), (v.float() * scale).half(), (q.float() * min(1.0, scale ** -2 * 2.0 ** 6)).half()
    got, ref = ct.causal_dot_product(q.to(DEV), k.to(DEV), v.to(DEV)).double().cpu(), torch.from_numpy(oracle.causal(q, k, v))
    assert torch.isfinite(got).all()
    # half a unit of 2^-24, the spacing of fp16's subnormals, where the output is one
    assert ((got - ref).abs() <= 2.0 ** -11 * ref.abs() + 2.0 ** -25 + 2.0 ** -13 * ref.pow(2).mean().sqrt()).all()


@pytest.mark.parametrize("dt", [BF, HF], ids=["bf16", "fp16"])
def test_an_infinite_value_stays_in_its_column(ct, dt):
    """v[40, 5] infinite: from position 64 (the next chunk) on column 5 is no number a finite sum could give, every other
    column what it is without it."""
    q, k, v, _ = (t.to(DEV) for t in inputs(1, 1, 128, 256, 256, dt, seed=4))
    want = ct.causal_dot_product(q, k, v)
    v[0, 0, 40, 5] = float("inf")
    got = ct.causal_dot_product(q, k, v)
    other = [j for j in range(256) if j != 5]
    assert torch.equal(got[..., other], want[..., other])
    assert torch.isfinite(got[0, 0, :32, 5]).all()
    assert not torch.isfinite(got[0, 0, 64:, 5]).any()


@pytest.mark.parametrize("x", [float("inf"), -float("inf")])
@pytest.mark.parametrize("dt", [BF, HF], ids=["bf16", "fp16"])
def test_an_infinite_value_within_its_chunk(ct, dt, x):
    """v[40, 5] infinite: from there to the end of the chunk column 5 is infinite with the sign of the score times that of x
    (no score of these inputs is zero), in both directions: reversed, the positions of the chunk up to 40."""
    q, k, v, _ = (t.to(DEV) for t in inputs(1, 1, 96, 256, 256, dt, seed=4))
    v[0, 0, 40, 5] = x
    want = torch.sign(q[0, 0].float() @ k[0, 0, 40].float()) * x
    for rev, rows in ((False, slice(40, 64)), (True, slice(32, 41))):
        assert torch.equal(ct.causal_dot_product(q, k, v, rev)[0, 0, rows, 5].float(), want[rows])


@pytest.mark.parametrize("dt", [BF, HF], ids=["bf16", "fp16"])
def test_the_largest_start_states(ct, dt):
    """Start states of 2^126, of either sign and 2^125 apart: the sums are fp32's, and infinite in fp16 only as outputs."""
    q, k, v, _ = (t.to(DEV) for t in inputs(1, 1, 40, 160, 160, dt, seed=2))
    q[0, 0, :, :2] = torch.tensor([1.0, -1.0], device=DEV).to(dt)
    q[0, 0, :, 2:] = 0
    state = torch.zeros(1, 1, 160, 160, device=DEV)
    state[0, 0, 0, :80], state[0, 0, 1, :80] = 2.0 ** 126, 2.0 ** 125
    state[0, 0, 0, 80:], state[0, 0, 1, 80:] = -(2.0 ** 126), -(2.0 ** 126)
    o, _ = ct.causal_prefill(q, k, v, state=state)
    want = torch.tensor(2.0 ** 125, device=DEV).to(dt)  # (fp16: infinite)
    assert (o[..., :80] == want).all()
    # equal entries cancel: what is left of the first chunk is the sequence's own part
    assert torch.equal(o[..., :32, 80:], ct.causal_prefill(q, k, v)[0][..., :32, 80:])


def test_groups_need_no_workspace(ct):
    """Called without the workspace it asks for, the library walks the sequence whole."""
    from cottention_transformer_amd import _loader
    q, k, v, _ = (t.to(DEV) for t in inputs(1, 2, 2000, 192, 192, BF, seed=6))
    want, out, L = ct.causal_dot_product(q, k, v), torch.empty_like(v), _loader.lib()
    assert L.cott_causal_workspace_bytes(1, 2, 2000, 192, 192, _loader.BF16) > 0
    rc = L.cott_causal_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 1, 2, 2000, 192, 192, _loader.BF16, 0, None, 0,
                           torch.cuda.current_stream().cuda_stream)
    assert rc == _loader.OK
    # both within half a unit of the same number
    assert rel_l2(out, want.double().cpu().numpy()) <= 2 * BOUND[BF]


def test_states_in_and_out_of_groups(ct, oracle):
    q, k, v, _ = inputs(1, 1, 4000, 256, 144, HF, seed=8)
    qd, kd, vd = (t.to(DEV) for t in (q, k, v))
    o1, s1 = ct.causal_prefill(qd[:, :, :1900], kd[:, :, :1900], vd[:, :, :1900])
    o2, s2 = ct.causal_prefill(qd[:, :, 1900:], kd[:, :, 1900:], vd[:, :, 1900:], state=s1)
    assert rel_l2(torch.cat((o1, o2), 2), oracle.causal(q, k, v)) <= BOUND[HF]
    # 4000 products summed in fp32, errors of either sign: sqrt(4000) * 2^-24 in the mean
    assert rel_l2(s2, (k.double().transpose(2, 3) @ v.double()).numpy()) <= 64 * 2.0 ** -24


def test_more_heads_than_one_launch_holds(ct):
    """2^19 heads of one position: twelve workgroups of 768 threads a head for the gradients, over 2^32 threads in all.  The
    plain-FMA kernel took 3 * 2^19 * 8 * 256."""
    h, d = 1 << 19, 256
    q, k, v, do = (torch.randn(1, h, 1, d, device=DEV).to(BF) for _ in range(4))
    dq, dk, dv = ct.causal_backward(q, k, v, do)
    dot = lambda a, b: (a.float() * b.float()).sum(-1, keepdim=True)
    for got, ref in ((dq, dot(do, v) * k.float()), (dk, dot(do, v) * q.float()), (dv, dot(q, k) * do.float())):
        # half a unit of the output, and the fp32 sum of 256 products that cancel: 256 * 2^-24 of their absolute sum
        assert float((got.float() - ref).norm() / ref.norm()) <= BOUND[BF]
        assert float((got[0, -1].float() - ref[0, -1]).norm() / ref[0, -1].norm()) <= 2 * BOUND[BF]
