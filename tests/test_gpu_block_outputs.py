"""What a block hands out beside its output: keys and values for a cache, in memory of their own."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("b,s", [(2, 70), (1, 1)])
@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kind", ["gpt", "bert"])
def test_cached_keys_and_values_hold_nothing_else(kind, b, s, grad):
    """Under autocast the projections are one GEMM; what is cached of them is not a view of all three.  Values are those of the
    layers, gradients pass through."""
    from cottention_transformer_amd.modules import BertCosAttention, GPTCosAttention
    torch.manual_seed(0)
    e, h = 128, 4
    cfg = SimpleNamespace(hidden_size=e, num_attention_heads=h, max_position_embeddings=128, rotary_dim=16, attn_pdrop=0.0,
                          resid_pdrop=0.0, attention_probs_dropout_prob=0.0, is_decoder=True)
    m = (GPTCosAttention if kind == "gpt" else BertCosAttention)(cfg).to(DEV)
    x = torch.randn(b, s, e, device=DEV, requires_grad=grad)
    with torch.autocast("cuda", dtype=torch.bfloat16), torch.set_grad_enabled(grad):
        key, value = m(x, use_cache=True)[1] if kind == "gpt" else m(x)[-1]
        want_k, want_v = (lin(x).view(b, s, h, e // h).permute(0, 2, 1, 3)
                          for lin in ((m.k_proj, m.v_proj) if kind == "gpt" else (m.key, m.value)))
    for t in (key, value):
        assert t.shape == (b, h, s, e // h) and t.untyped_storage().nbytes() == t.numel() * t.element_size()
    assert value.stride() == want_v.stride() and float((value - want_v).norm() / want_v.norm()) <= 1e-2
    if kind == "bert":
        assert key.stride() == want_k.stride() and float((key - want_k).norm() / want_k.norm()) <= 1e-2
    if grad:
        got, = torch.autograd.grad(value.float().sum(), x)
        want, = torch.autograd.grad(want_v.float().sum(), x)
        assert float((got - want).norm() / want.norm()) <= 1e-2
