"""GPU: the C++ eager route (csrc/kd_torch.cpp) against the custom ops.

Both launch the same kernels on the same operands, so every output is equal bit
for bit; what autograd, hooks, checkpointing and modes see has to be what the
custom ops show them."""
import pytest
import torch

from kerneldev_amd import _lib, flash_attention
from kerneldev_amd.attention import build_plan_from_tokens
from kerneldev_amd.span_head import span_scores
from kerneldev_amd.synth import CONFIG3_LAYOUT, cocktail_batch, qkvdo

pytestmark = pytest.mark.gpu


def _both(monkeypatch, fn):
    got = fn()
    with monkeypatch.context() as m:
        m.setattr(_lib, "eager", lambda *t: False)
        return got, fn()


CASES = [
    (2, 3, 333, 64, torch.bfloat16, {}),
    (1, 2, 1200, 128, torch.float16, dict(hadamard=True, out_layout="bthd")),
    (2, 2, 512, 128, torch.bfloat16, dict(qk_dtype="fp8_e4m3", hadamard=True)),
    (2, 2, 400, 256, torch.bfloat16, dict(qk_dtype="fp8_e4m3", precision="bf16")),
    (2, 2, 200, 64, torch.bfloat16, dict(precision="ieee", causal=False)),
    (1, 2, 129, 32, torch.float32, dict(precision="ieee")),
    (2, 4, 256, 16, torch.float16, {}),
    (2, 2, 300, 32, torch.float32, {}),
    (1, 1, 1100, 16, torch.float32, dict(out_layout="bthd")),
]


@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("how", ["causal", "metadata", "tokens", "strided"])
def test_same_bits_as_the_ops(dev, monkeypatch, case, how):
    B, H, T, D, dtype, kw = case
    q, k, v, do = (x.to(dev) for x in qkvdo(B, H, T, D, seed=T, dtype=dtype))
    tokens, *meta = (x.to(dev)[:, :T] for x in cocktail_batch(B, 2048, CONFIG3_LAYOUT, seed=3))
    if how == "strided":  # layouts the kernels take as they are, and one they do not (odd row strides)
        q = q.transpose(1, 2).contiguous().transpose(1, 2)
        k = torch.empty(*k.shape[:3], D + 3, dtype=dtype, device=dev)[..., 3:].copy_(k)
        do = do.transpose(2, 3).contiguous().transpose(2, 3)

    def run():
        xs = [x.detach().requires_grad_(True) for x in (q, k, v)]
        opts = dict(kw)
        if how == "metadata":
            opts.update(zip(("in_span", "span_id", "is_prefix"), meta))
            opts["lens"] = torch.full((B,), T - 9, dtype=torch.int32, device=dev)
        elif how == "tokens":
            opts["plan"] = build_plan_from_tokens(tokens, D)
        (o, lse), mask = flash_attention(*xs, return_lse=True, return_attention_mask=True, **opts)
        return (o, lse, mask, *torch.autograd.grad(o, xs, do))

    got, want = _both(monkeypatch, run)
    for x, y in zip(got, want):
        assert torch.equal(x, y) and x.stride() == y.stride() and x.requires_grad == y.requires_grad


def test_span_head_same_bits(dev, monkeypatch):
    tokens = cocktail_batch(2, 1024, CONFIG3_LAYOUT, seed=4)[0].to(dev)
    h = torch.randn(2, 1024, 96, device=dev).bfloat16()

    def run():
        x = h.clone().requires_grad_(True)
        s = span_scores(tokens, x)
        return s, torch.autograd.grad(s.sum(), x)[0]

    got, want = _both(monkeypatch, run)
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_what_autograd_sees(dev):
    q, k, v, do = (x.to(dev) for x in qkvdo(1, 2, 200, 64, seed=5))
    xs = [x.requires_grad_(True) for x in (q, k, v)]
    o, lse = flash_attention(*xs, return_lse=True)
    assert lse.requires_grad
    assert torch.autograd.grad(lse.sum(), q, allow_unused=True)[0] is None  # LSE's gradient is ignored
    # a second derivative is refused where it is used
    g = torch.autograd.grad(flash_attention(*xs), xs, do, create_graph=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(g[0].float().sum(), q)
    # saved tensors pass through the hooks, and an operand changed in place is found out
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
        o = flash_attention(*xs)
    o.backward(do)
    assert len(seen) == 7
    x = q * 1
    o = flash_attention(x, k, v)
    x.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        o.backward(do)


def test_calls_that_are_not_plain_take_the_op(dev):
    q, k, v, _ = (x.to(dev) for x in qkvdo(1, 2, 200, 64, seed=6))
    want = flash_attention(q, k, v)
    ops = []

    class Seen(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            ops.append(str(func))
            return func(*args, **(kwargs or {}))

    with Seen():
        assert torch.equal(flash_attention(q, k, v), want)
    assert "kdattn.fwd.default" in ops
    z = torch.randn(1, 2, 200, 64, device=dev, dtype=torch.complex64)
    n, r = z.conj().imag, -z.imag  # a lazily negated view
    assert n.is_neg() and torch.equal(flash_attention(n, n, n, precision="ieee"), flash_attention(r, r, r, precision="ieee"))
    with torch._subclasses.fake_tensor.FakeTensorMode():
        f = torch.empty(1, 2, 200, 64, device=dev, dtype=torch.bfloat16)
        assert flash_attention(f, f, f).shape == f.shape
    with torch.device("cpu"):  # a function mode
        assert torch.equal(flash_attention(q, k, v), want)
