"""One new token through a whole block (cott_decode_block) and the decode step in column strips."""
import pytest
import torch

from util import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF = torch.bfloat16, torch.float16


@pytest.fixture(scope="module")
def ct():
    import cottention_transformer_amd as ct_
    return ct_


def block_reference(x, wq, wk, wv, wo, state, sig, cnt, table, pos):
    """The same steps in fp64 on the CPU, rounded to x's type where the block leaves 16-bit numbers."""
    b, h, d = state.shape[:3]
    dt = x.dtype
    q, k, v = ((x.double() @ w.double().t()).to(dt).double().reshape(b, h, d) for w in (wq, wk, wv))
    r = table.shape[1]
    sn, cs = table[pos, :r // 2].double(), table[pos, r // 2:].double()
    out = []
    for t in (q, k):
        t = t.clone()
        e, o = t[..., 0:r:2].clone(), t[..., 1:r:2].clone()
        t[..., 0:r:2], t[..., 1:r:2] = e * cs - o * sn, o * cs + e * sn
        out.append(torch.nn.functional.normalize(t, dim=-1, eps=1e-12))
    q, k = out
    v = v / (cnt ** sig.double()).clamp(min=1.0)[None, :, None]
    s = state.double() + k[..., None] * v[..., None, :]
    o = (q[..., None, :] @ s)[..., 0, :].to(dt).double().reshape(b, h * d)
    return (o @ wo.double().t()).to(dt), s


# rows from one to all sixteen; contractions of one to 64 steps of 32 (fewer and more than the eight wavefronts)
@pytest.mark.parametrize("case", [(1, 1, 32, BF), (3, 3, 32, HF), (1, 12, 64, BF), (16, 5, 64, HF), (2, 16, 128, BF),
                                  (7, 3, 256, HF), (1, 9, 256, BF)], ids=lambda c: "x".join(map(str, c[:3])))
def test_block_against_fp64(ct, case):
    from cottention_transformer_amd import ops
    from cottention_transformer_amd.modules import rotary_table
    b, h, d, dt = case
    e = h * d
    g = torch.Generator().manual_seed(e + b)
    x = torch.randn(b, e, generator=g).to(dt)
    ws = [(torch.randn(e, e, generator=g) / e ** 0.5).to(dt) for _ in range(4)]
    state = 0.1 * torch.randn(b, h, d, d, generator=g)
    sig, table = torch.sigmoid(torch.randn(h, generator=g)), rotary_table(40, 32)
    y_ref, s_ref = block_reference(x, *ws, state, sig, 9.0, table, 17)
    s = state.to(DEV)
    y = ops.decode_block(x.to(DEV), *(w.to(DEV) for w in ws), s, sig.to(DEV), 9.0, (table.to(DEV), 17))
    # a projection's sum in another order may round to the neighbouring 16-bit number: one unit of q, k, v, o and y each
    unit = 2.0 ** (-8 if dt is BF else -11)
    assert y.shape == (b, e) and rel_l2(y, y_ref.double().numpy()) <= 3 * unit
    assert rel_l2(s, s_ref.numpy()) <= 3 * unit


def test_block_is_refused_where_not_built(ct):
    from cottention_transformer_amd import ops
    w = torch.zeros(64, 64, device=DEV, dtype=BF)
    for b, dt, msg in ((17, BF, "at most 16"), (1, torch.float32, "bf16 / fp16")):
        x, wt = torch.zeros(b, 64, device=DEV, dtype=dt), w.to(dt)
        with pytest.raises(RuntimeError, match=msg):
            ops.decode_block(x, wt, wt, wt, wt, torch.zeros(b, 1, 64, 64, device=DEV))


@pytest.mark.parametrize("b", [1, 16, 17])
def test_module_tokens_equal_the_separate_calls(ct, b, monkeypatch):
    """GPTCosAttention's recurrent inference: the same tokens with the one-call form switched off."""
    from types import SimpleNamespace
    from cottention_transformer_amd import ops
    from cottention_transformer_amd.modules import GPTCosAttention
    cfg = SimpleNamespace(hidden_size=256, num_attention_heads=4, max_position_embeddings=64, rotary_dim=32, attn_pdrop=0.0,
                          resid_pdrop=0.0, fast_inference=True)
    torch.manual_seed(3)
    m = GPTCosAttention(cfg).to(DEV, BF).eval()
    tokens = torch.randn(4, b, 1, 256, device=DEV).to(BF)
    calls = []
    inner = ops.decode_block
    monkeypatch.setattr(ops, "decode_block", lambda *a, **k: calls.append(1) or inner(*a, **k))

    def generate():
        m.reset_state()
        return torch.cat([m(t)[0] for t in tokens], 1), m.state

    with torch.no_grad():
        got, state = generate()
    assert len(calls) == (4 if b <= 16 else 0)
    want, state_want = generate()  # with gradients enabled: the projections are called separately
    assert len(calls) == (4 if b <= 16 else 0) and want.requires_grad and not got.requires_grad
    assert rel_l2(got, want.detach().double().cpu().numpy()) <= 3 * 2.0 ** -8
    assert rel_l2(state, state_want.double().cpu().numpy()) <= 3 * 2.0 ** -8


# heads on either side of where strips start, and of a workgroup of its own for every wavefront
@pytest.mark.parametrize("case", [(1, 3, 128, 128), (1, 300, 32, 64), (1, 513, 96, 128), (1, 63, 200, 256), (1, 1025, 32, 64)],
                         ids=lambda c: "x".join(map(str, c)))
def test_decode_in_column_strips(ct, oracle, case):
    b, h, dk, dv = case
    g = torch.Generator().manual_seed(h)
    q, k, v = (torch.randn(b, h, x, generator=g).to(BF) for x in (dk, dk, dv))
    state = torch.randn(b, h, dk, dv, generator=g)
    ref_state = state.double().numpy().copy()
    ref = oracle.decode_step(ref_state, q, k, v)
    s = state.to(DEV)
    o = ct.decode_step(s, q.to(DEV), k.to(DEV), v.to(DEV))
    assert rel_l2(o, ref) <= 2.0 ** -9 + 2.0 ** -16   # the output's rounding
    assert rel_l2(s, ref_state) <= 2.0 ** -23         # one fp32 multiply-add per entry


# fewer heads than strips are made of, more, and the workgroup-per-head kernel (16 columns)
@pytest.mark.parametrize("case", [(1, 3, 128), (2, 150, 64), (1, 1025, 64), (1, 5, 256), (1, 3, 16)], ids=lambda c: "x".join(map(str, c)))
def test_output_in_the_memory_of_an_input(ct, oracle, case):
    """decode_step(..., out=): q, k or v themselves, or a tensor that overlaps all three of them by half a head."""
    b, h, d = case
    g = torch.Generator().manual_seed(h)
    q, k, v = (torch.randn(b, h, d, generator=g).to(BF) for _ in range(3))
    state = torch.randn(b, h, d, d, generator=g)
    ref_state = state.double().numpy().copy()
    ref = oracle.decode_step(ref_state, q, k, v)
    for which in ("q", "k", "v", "part"):
        flat = torch.empty(4, b * h * d, dtype=BF, device=DEV)
        x = dict(zip("qkv", (row.view(b, h, d) for row in flat)))
        for name, t in zip("qkv", (q, k, v)):
            x[name].copy_(t)
        out = x[which] if which != "part" else flat.view(-1)[b * h * d - d // 2:][:b * h * d].view(b, h, d)
        s = state.to(DEV)
        got = ct.decode_step(s, x["q"], x["k"], x["v"], out=out)
        assert got is out and rel_l2(out, ref) <= 2.0 ** -9 + 2.0 ** -16, which   # the output's rounding
        assert rel_l2(s, ref_state) <= 2.0 ** -23, which                          # one fp32 multiply-add per entry


def test_prepared_output_in_the_memory_of_an_input(ct):
    from cottention_transformer_amd import ops
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(2, 9, 128, generator=g).to(DEV, BF) for _ in range(3))
    state = torch.randn(2, 9, 128, 128, generator=g).to(DEV)
    want_state = state.clone()
    want = ops.decode_step_prepared(want_state, q, k, v)
    for i in range(3):
        x = [t.clone() for t in (q, k, v)]
        s = state.clone()
        got = ops.decode_step_prepared(s, *x, out=x[i])
        # the same sum in one wavefront's order or in strips: half a unit each
        assert got is x[i] and rel_l2(got, want.double().cpu().numpy()) <= 2.0 ** -8 and torch.equal(s, want_state)


@pytest.mark.parametrize("dt", [torch.float32, torch.float64, HF, BF], ids=["fp32", "fp64", "fp16", "bf16"])
def test_norm_const_in_place_of_its_sigmoid(ct, dt):
    """The sigmoid formed in the kernel is torch's, bit for bit: same states and outputs from norm_const and from sig."""
    from cottention_transformer_amd import ops
    g = torch.Generator().manual_seed(5)
    b, h, d = 3, 40, 64
    norm = torch.linspace(-8, 8, h, device=DEV).to(dt).reshape(1, h, 1, 1)
    sig = norm.sigmoid().reshape(h).float()
    x = torch.float64 if dt is torch.float64 else BF
    q, k, v = (torch.randn(b, h, d, generator=g).to(DEV, x) for _ in range(3))
    s1 = torch.randn(b, h, d, d, generator=g).to(DEV, torch.float64 if x is torch.float64 else torch.float32)
    s2 = s1.clone()
    o1 = ops.decode_step_prepared(s1, q, k, v, sig=sig, cnt=37.0)
    o2 = ops.decode_step_prepared(s2, q, k, v, norm_const=norm, cnt=37.0)
    assert torch.equal(o1, o2) and torch.equal(s1, s2)
    with pytest.raises(RuntimeError, match="norm_const"):
        ops.decode_step_prepared(s2, q, k, v, norm_const=norm[:, :3], cnt=37.0)


@pytest.mark.parametrize("grad", [False, True], ids=["one call", "separate calls"])
def test_module_tokens_follow_norm_const(ct, grad):
    """norm_const written through .data between two tokens counts from the next one on."""
    from types import SimpleNamespace
    from cottention_transformer_amd.modules import GPTCosAttention
    cfg = SimpleNamespace(hidden_size=128, num_attention_heads=2, max_position_embeddings=64, rotary_dim=32, attn_pdrop=0.0,
                          resid_pdrop=0.0, fast_inference=True)
    torch.manual_seed(3)
    m, fresh = GPTCosAttention(cfg).to(DEV, BF).eval(), GPTCosAttention(cfg).to(DEV, BF).eval()
    fresh.load_state_dict(m.state_dict())
    fresh.norm_const.data.fill_(-3.0)
    tokens = torch.randn(3, 1, 1, 128, device=DEV).to(BF)
    with torch.set_grad_enabled(grad):
        for t in tokens[:2]:
            m(t)
        fresh.state, fresh.cur_s = m.state.clone(), m.cur_s
        m.norm_const.data.fill_(-3.0)
        got, want = m(tokens[2])[0], fresh(tokens[2])[0]
    assert torch.equal(got, want) and torch.equal(m.state, fresh.state)


def test_module_token_calls_a_projection_whose_forward_was_replaced(ct):
    from types import SimpleNamespace
    from cottention_transformer_amd.modules import GPTCosAttention
    cfg = SimpleNamespace(hidden_size=128, num_attention_heads=2, max_position_embeddings=64, rotary_dim=32, attn_pdrop=0.0,
                          resid_pdrop=0.0, fast_inference=True)
    m = GPTCosAttention(cfg).to(DEV, BF).eval()
    m.out_proj.forward = lambda x: torch.full_like(x, 3.0)
    with torch.no_grad():
        assert (m(torch.randn(1, 1, 128, device=DEV).to(BF))[0] == 3.0).all()


def test_every_launch_of_a_token_and_of_wide_heads_is_counted(ct):
    from cottention_transformer_amd import _loader, ops
    x, w, s = torch.randn(1, 64, device=DEV).to(BF), torch.randn(64, 64, device=DEV).to(BF), torch.zeros(1, 1, 64, 64, device=DEV)
    wide = torch.randn(1, 2, 1000, 256, device=DEV).to(BF)
    _loader.profile_enable(True)
    try:
        for name in _loader.KERNEL_IDS:
            _loader.profile_read(name)
        ops.decode_block(x, w, w, w, w, s)
        ct.causal_dot_product(wide, wide, wide)
        counts = {name: _loader.profile_read(name)[1] for name in _loader.KERNEL_IDS}
    finally:
        _loader.profile_enable(False)
    assert {k: n for k, n in counts.items() if n} == {"token_linear": 2, "decode": 1, "wide_sums": 1, "wide_scan": 1}
    names = [_loader.lib().cott_kernel_name(i).decode() for i in _loader.KERNEL_IDS.values()]
    assert all(names) and len(set(names)) == len(names)
