"""Operands whose types differ.

The kernels read q, k and v as one type.  CPU: what the bf16x3 packing hands
over; GPU: the calls themselves, against the same calls on converted operands."""
import pytest
import torch

from kerneldev_amd import attention as A
from kerneldev_amd import flash_attention


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float64])
def test_packing_reads_fp32_only(monkeypatch, dtype):
    """kd_x3_pack reads its sources as fp32: every tensor handed to it is one, with the operand's values."""
    seen = []
    monkeypatch.setattr(A, "_x3_call", lambda pack, tensors, *shape: seen.extend(t[0] for t in tensors))
    q, k = torch.randn(1, 2, 5, 16), torch.randn(1, 2, 5, 16).to(dtype)
    A._x3_packed((q, k, k), ("hhl", "hlh", "hlh"), 1, 2, 5, 16, 64)
    assert [t.dtype for t in seen] == [torch.float32] * 3
    assert torch.equal(seen[0], q) and torch.equal(seen[1], k.float())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 64, 130])
@pytest.mark.parametrize("d", [16, 32])
def test_bf16x3_with_narrower_keys_and_values(dev, d, T):
    g = torch.Generator().manual_seed(d + T)
    q, k, v, do = (torch.randn(1, 3, T, d, generator=g).to(dev) for _ in range(4))
    k, v = k.to(torch.bfloat16), v.to(torch.float16)
    xs, ys = [x.clone().requires_grad_(True) for x in (q, k, v)], [x.float().requires_grad_(True) for x in (q, k, v)]
    o, want = flash_attention(*xs), flash_attention(*ys)
    assert torch.equal(o, want)
    for x, a, b in zip(xs, torch.autograd.grad(o, xs, do), torch.autograd.grad(want, ys, do)):
        assert a.dtype == x.dtype and torch.equal(a, b.to(x.dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("q_type,k_type,v_type", [(torch.bfloat16, torch.float16, torch.bfloat16),
                                                  (torch.float16, torch.float32, torch.float32),
                                                  (torch.float32, torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("d,kw", [(64, {}), (128, dict(hadamard=True)), (32, dict(precision="ieee"))])
def test_keys_and_values_are_taken_in_the_type_of_q(dev, q_type, k_type, v_type, d, kw):
    g = torch.Generator().manual_seed(d)
    q, k, v, do = (torch.randn(1, 2, 130, d, generator=g).to(t).to(dev) for t in (q_type, k_type, v_type, q_type))
    xs, ys = [x.clone().requires_grad_(True) for x in (q, k, v)], [x.to(q_type).requires_grad_(True) for x in (q, k, v)]
    o, want = flash_attention(*xs, **kw), flash_attention(*ys, **kw)
    assert o.dtype == q_type and torch.equal(o, want)
    for x, a, b in zip(xs, torch.autograd.grad(o, xs, do), torch.autograd.grad(want, ys, do)):
        assert a.dtype == x.dtype and torch.equal(a, b.to(x.dtype))
