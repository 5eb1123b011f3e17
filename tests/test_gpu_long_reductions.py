"""Reductions around a block for batches that one workgroup per head or sequence does not carry."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# up to one step's rows, one more; sequences in pieces; second steps of their own; lengths that are left to torch
@pytest.mark.parametrize("b,h,n", [(1, 1, 32768), (16, 3, 2049), (64, 4, 2048), (1, 2, 131072), (3, 5, 98304), (600, 2, 512), (70, 3, 500), (1, 2, 70001),
                                   (0, 3, 5), (2, 3, 0)])
def test_head_sums(b, h, n):
    from cottention_transformer_amd import ops
    x = torch.randn(b, h, n, generator=torch.Generator().manual_seed(n)).to(DEV)
    got, want = ops.head_sums(x), x.double().sum((0, 2))
    assert got.shape == (h,) and got.dtype == torch.float32
    # chains of at most a few hundred additions, as in the sums of one step
    assert (got.double() - want).abs().le(x.double().abs().sum((0, 2)) * 2.0 ** -24 * 8).all()


def _workgroup_rows(monkeypatch, call):
    """The most rows that one workgroup of cott_head_sums adds, and the longest mask row cott_keep_counts walks, during call()."""
    from cottention_transformer_amd import _loader
    real, seen = _loader.lib(), {"head": 0, "mask": 0}

    class Watched:
        def __getattr__(self, name):
            f = getattr(real, name)

            def wrapped(*a):
                if name == "cott_head_sums":
                    seen["head"] = max(seen["head"], a[2] * a[4])
                if name == "cott_keep_counts":
                    seen["mask"] = max(seen["mask"], a[5])
                return f(*a)
            return wrapped
    watched = Watched()
    monkeypatch.setattr(_loader, "lib", lambda: watched)
    call()
    return dict(seen)


def test_norm_const_gradient_of_a_long_batch(monkeypatch):
    """The derivative of norm_const over 64 x 2048 positions: no workgroup adds more than 32768 rows."""
    from cottention_transformer_amd import ops
    b, n, h, d = 64, 2048, 2, 32
    g = torch.Generator().manual_seed(0)
    q, k, v, gq, gk, gv = (torch.randn(b, h, n, d, generator=g).to(DEV) for _ in range(6))
    cnt = torch.arange(1, n + 1.0).expand(b, n).contiguous().to(DEV)
    sig = torch.tensor([0.3, 0.7], device=DEV)
    out = []
    seen = _workgroup_rows(monkeypatch, lambda: out.append(ops.prepare_inputs_backward(q, k, v, gq, gk, gv, None, cnt, sig, want_dsig=True)[3]))
    s64, c64 = sig.double().requires_grad_(True), cnt.double()[:, None, :, None]
    ((v.double() / torch.clamp(c64 ** s64[None, :, None, None], min=1)) * gv.double()).sum().backward()
    assert 0 < seen["head"] <= 1 << 15
    assert float((out[0].double() - s64.grad).norm() / s64.grad.norm()) <= 1e-5


@pytest.mark.parametrize("kind", ["gpt", "bert"])
def test_mask_of_one_long_sequence(monkeypatch, kind):
    """A single masked sequence of 40000 positions: its mask is not walked by one workgroup; the result is that of the kernel."""
    from types import SimpleNamespace
    from cottention_transformer_amd import ops
    from cottention_transformer_amd.modules import BertCosAttention, GPTCosAttention
    torch.manual_seed(0)
    s, e = 40000, 64
    cfg = SimpleNamespace(hidden_size=e, num_attention_heads=2, max_position_embeddings=64, rotary_dim=16, attn_pdrop=0.0,
                          resid_pdrop=0.0, attention_probs_dropout_prob=0.0)
    m = (GPTCosAttention if kind == "gpt" else BertCosAttention)(cfg).to(DEV)
    x = torch.randn(1, s, e, device=DEV)
    mask = torch.where(torch.rand(1, 1, 1, s, device=DEV) < 0.8, 0.0, -1e30)
    kw = {"position_ids": torch.zeros(1, s, dtype=torch.int64, device=DEV)} if kind == "gpt" else {}
    outs = []
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        seen = _workgroup_rows(monkeypatch, lambda: outs.append(m(x, attention_mask=mask, **kw)[0]))
        monkeypatch.setattr(ops, "keep_and_counts_preferred", lambda *a: True)
        outs.append(m(x, attention_mask=mask, **kw)[0])
    assert seen["mask"] <= 1 << 15 and torch.equal(*outs)
