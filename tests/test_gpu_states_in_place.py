"""cott_causal_fwd_state with state_in and state_out the same memory: the results of distinct buffers, bit for bit, also
where a head's sequence is cut into groups whose workgroups run in any order (the start state is in their slots before
the launch that writes state_out begins)."""
import pytest
import torch

from util import TOL, inputs, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64

# (heads, positions, Dk, Dv, type, cut into groups): every kernel that starts from a state; odd widths and lengths
CASES = [(2, 4000, 64, 64, BF, True), (16, 8192, 64, 64, HF, True), (5, 3001, 48, 80, BF, True), (4, 4100, 128, 128, BF, True),
         (16, 9000, 128, 128, HF, True), (3, 2100, 112, 64, BF, True), (2, 2500, 32, 128, HF, True), (2, 3000, 64, 64, F32, True),
         (3, 2051, 48, 64, F32, True), (2, 2500, 128, 96, F32, True), (2, 1500, 32, 64, F32, True), (2, 2000, 256, 256, BF, True),
         (1, 4100, 160, 144, HF, True), (3, 900, 64, 192, BF, True), (300, 200, 64, 64, BF, False), (2, 300, 256, 160, BF, False),
         (2, 100, 64, 64, F64, False)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:4])) + "-" + str(c[4]).split(".")[-1])
def test_same_memory_equals_distinct(case):
    from cottention_transformer_amd import _loader, ops
    h, n, dk, dv, dt, groups = case
    L, code = _loader.lib(), ops._DTYPES[dt]
    q, k, v, _ = inputs(1, h, n, dk, dv, dt, seed=n)
    acc = F64 if dt is F64 else F32
    start = torch.randn(1, h, dk, dv, generator=torch.Generator().manual_seed(h)).to(acc)
    dev = [t.to(DEV) for t in (q, k, v)]
    need = L.cott_causal_workspace_bytes(1, h, n, dk, dv, code)
    assert (need > 0) == groups
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)

    def run(sin, sout):
        o = torch.empty(1, h, n, dv, dtype=dt, device=DEV)
        rc = L.cott_causal_fwd_state(*(t.data_ptr() for t in dev), o.data_ptr(), sin.data_ptr(), sout.data_ptr(), 1, h, n, dk, dv,
                                     code, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
        assert rc == _loader.OK, _loader.last_error()
        return o

    sin, sout = start.to(DEV), torch.empty(1, h, dk, dv, dtype=acc, device=DEV)
    want = run(sin, sout)
    assert torch.equal(sin.cpu(), start)
    both = start.to(DEV)
    got = run(both, both)
    assert torch.equal(got, want) and torch.equal(both, sout)
    # and the values themselves: the states, and the outputs of the last positions, which every earlier group adds to
    s_ref = start.double() + k.double().transpose(2, 3) @ v.double()
    assert rel_l2(sout, s_ref.numpy()) <= TOL[F64 if dt is F64 else F32]
    m = min(n, 70)
    before = s_ref - k.double()[:, :, n - m:].transpose(2, 3) @ v.double()[:, :, n - m:]
    scores = torch.tril(q.double()[:, :, n - m:] @ k.double()[:, :, n - m:].transpose(2, 3))
    o_ref = q.double()[:, :, n - m:] @ before + scores @ v.double()[:, :, n - m:]
    assert rel_l2(want[:, :, n - m:], o_ref.numpy()) <= TOL[dt]
