"""GPU: kd_x3_pack and kd_x3_unpack against their torch form (x3_reference.py), bit for bit.

Every head dim, both row patterns, both summed blocks, wider rows than three parts, row
counts that are no multiple of a workgroup, strided fp32 sides, one to four tensors a call."""
import ctypes

import pytest
import torch

from kerneldev_amd import _lib
from kerneldev_amd.attention import _strides3, _stream
from x3_reference import hi_lo, x3

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 3, 37), (1, 5, 129), (3, 2, 256)]


def _strided(x, how):
    if how == "bthd":
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if how == "wide":  # rows of d + 8 in a larger tensor
        return torch.zeros(*x.shape[:3], x.shape[3] + 8, device=x.device)[..., 8:].copy_(x)
    return x


def _args(B, H, T, d, Dp, n):
    a = _lib.X3Args()
    a.n, a.B, a.H, a.T, a.d, a.Dp = n, B, H, T, d, Dp
    return a


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("how", ["plain", "bthd", "wide"])
@pytest.mark.parametrize("d,Dp", [(16, 64), (16, 48), (32, 128), (32, 96), (64, 256), (64, 192)])
def test_pack(dev, d, Dp, how, shape):
    B, H, T = shape
    g = torch.Generator().manual_seed(d + T)
    xs = [torch.randn(B, H, T, d, generator=g) * 10.0 ** k for k in (-3, 0, 3, 0)]
    xs[0].view(-1)[:4] = torch.tensor([0.0, -0.0, 1e-40, 3e38])
    xs = [_strided(x.to(dev), how) for x in xs]
    for n in (1, 4):
        a, out = _args(B, H, T, d, Dp, n), [torch.full((B, H, T, Dp), 7.0, device=dev).bfloat16() for _ in range(n)]
        for i in range(n):
            a.src[i], a.src_strides[i], a.dst[i], a.sel[i] = xs[i].data_ptr(), _strides3(xs[i]), out[i].data_ptr(), i % 2
        _lib.check(_lib.load().kd_x3_pack(ctypes.byref(a), _stream(dev)), "kd_x3_pack")
        for i in range(n):
            assert torch.equal(out[i].view(torch.int16), x3(xs[i], "hlh" if i % 2 else "hhl", Dp).view(torch.int16))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("how", ["plain", "bthd", "wide"])
@pytest.mark.parametrize("d,Dp", [(16, 64), (16, 48), (32, 128), (64, 256), (64, 192)])
def test_unpack(dev, d, Dp, how, shape):
    B, H, T = shape
    g = torch.Generator().manual_seed(d + T)
    x = [torch.randn(B, H, T, Dp, generator=g).to(dev) for _ in range(3)]
    hi = [t.bfloat16() for t in x]
    lo = [(t - h.float()).bfloat16() for t, h in zip(x, hi)]
    out = [_strided(torch.full((B, H, T, d), 7.0, device=dev), how) for _ in x]
    for n in (1, 3):
        a = _args(B, H, T, d, Dp, n)
        for i in range(n):
            a.src[i], a.lo[i], a.dst[i], a.dst_strides[i] = hi[i].data_ptr(), lo[i].data_ptr(), out[i].data_ptr(), _strides3(out[i])
            a.sel[i] = 1 + i % 2
        _lib.check(_lib.load().kd_x3_unpack(ctypes.byref(a), _stream(dev)), "kd_x3_unpack")
        for i in range(n):
            assert torch.equal(out[i], hi_lo(hi[i], lo[i], d, 1 + i % 2))
