"""The native host module: which calls it takes, and that they equal the Python path's."""
import pytest
import torch
from torch.overrides import TorchFunctionMode

DEV = "cuda:0"
F32, F64, BF, HF = torch.float32, torch.float64, torch.bfloat16, torch.float16
THREE, FOUR = ("causal_saving", "causal_f32in", "noncausal"), ("noncausal_backward",)


class Seen(TorchFunctionMode):
    """Any function mode: the native module leaves the calls to Python, whose operations the mode sees."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.fixture(scope="module")
def native():
    from cottention_transformer_amd import _loader
    return _loader.native()


def all_none(native, q, k, v, g):
    out = [getattr(native, f)(q, k, v) for f in THREE] + [native.causal(q, k, v, False), native.noncausal_backward(q, k, v, g),
                                                          native.causal_backward(q, k, v, g, None)]
    return all(x is None for x in out)


def test_calls_left_to_python_without_a_gpu(native):
    q = torch.randn(1, 2, 8, 32)
    assert all_none(native, q, q, q, q) and all_none(native, None, 3, "x", [])
    assert native.decode_block(*(q,) * 7, 1.0, q, 0) is None
    for name, n in (("causal", 4), ("causal_saving", 3), ("causal_backward", 5), ("decode_block", 10)):
        with pytest.raises(TypeError):
            getattr(native, name)(*(q,) * (n - 1))


def make(b, h, n, dk, dv, dt, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(b, h, n, d, generator=g).to(DEV, dt) for d in (dk, dk, dv, dv)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(1, 2, 70, 64, 64, F32), (2, 3, 700, 64, 128, BF), (1, 2, 3000, 128, 128, HF), (1, 2, 40, 288, 288, F32),
                                  (1, 1, 50, 256, 256, BF), (1, 2, 33, 32, 32, F64), (8, 16, 300, 64, 64, BF)],
                         ids=lambda c: "x".join(map(str, c[:5])) + "-" + str(c[5]).split(".")[-1])
def test_equals_the_python_path(native, case):
    from cottention_transformer_amd import ops
    q, k, v, g = make(*case)
    calls = [lambda: ops.causal_dot_product(q, k, v), lambda: ops.causal_dot_product(q, k, v, True), lambda: ops.causal_dot_product_saving(q, k, v),
             lambda: ops.causal_dot_product_as(q, k, v, BF), lambda: ops.causal_backward(q, k, v, g),
             lambda: ops.causal_backward_from(q, k, v, g.to(BF)), lambda: ops.noncausal_dot_product(q, k, v),
             lambda: ops.noncausal_backward(q, k, v, g)]
    _, states = ops.causal_dot_product_saving(q, k, v)
    if states is not None:
        calls.append(lambda: ops.causal_backward(q, k, v, g, saved=states))
    assert native.causal(q, k, v, False) is not None and native.noncausal(q, k, v) is not None
    for call in calls:
        got = call()
        with Seen():
            assert all_none(native, q, k, v, g)
            want = call()
        flat = lambda x: [t for t in (x if isinstance(x, tuple) else (x,)) if t is not None]
        assert len(flat(got)) == len(flat(want))
        for a, c in zip(flat(got), flat(want)):
            assert a.dtype == c.dtype and a.shape == c.shape and torch.equal(a, c)


@pytest.mark.gpu
def test_other_tensors_are_left_to_python(native):
    q, k, v, g = make(1, 2, 64, 64, 64, BF)
    strided = q.transpose(1, 2).contiguous().transpose(1, 2)
    sub = torch.nn.Parameter(q.clone()).data.as_subclass(type("Sub", (torch.Tensor,), {}))
    for x in (strided, sub, q.float(), q[0], q[..., :32].contiguous(), q.cpu(), q[:, :, :0], q.to(torch.int16)):
        assert native.causal(x, k, v, False) is None and native.noncausal(x, k, v) is None
        assert native.causal_backward(x, k, v, g, None) is None
    assert native.causal_backward(q, k, v, g[:, :, :5].contiguous(), None) is None
    assert native.causal_backward(q, k, v, g, torch.zeros(3, device=DEV)) is None
    from cottention_transformer_amd import ops
    with pytest.raises(RuntimeError, match="prev_grad must have shape"):
        ops.causal_backward(q, k, v, g[:, :, :5].contiguous())
    with pytest.raises(RuntimeError, match="divisible by 16"):  # the library's own refusal
        ops.causal_dot_product(*(t[..., :40].contiguous() for t in (q, k)), v)
    with pytest.raises(RuntimeError):  # a batched tensor of a transform has no memory to hand over
        torch.vmap(lambda x: ops.causal_dot_product(x, x, x))(torch.stack([q, q]))


@pytest.mark.gpu
def test_current_stream_is_taken(native):
    from cottention_transformer_amd import ops
    q, k, v, _ = make(8, 16, 512, 64, 64, BF)
    want = ops.causal_dot_product(q, k, v)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        x = v * 2            # on the side stream: the op has to run behind it there
        got = ops.causal_dot_product(q, k, x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, ops.causal_dot_product(q, k, v * 2)) and not torch.equal(got, want)
