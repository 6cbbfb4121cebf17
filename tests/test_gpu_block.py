"""GPU: RMSNorm and the SwiGLU gate of gpt.py on their kernels (kd_block.hip).

Against the same formulas in fp64 on the same 16-bit inputs.  The kernels work
in fp32 and round once, so an output is within half an ulp of the exact value
plus the fp32 arithmetic's error: 2^-8 |ref| (bf16, half of 2^-7) or 2^-11
|ref| (fp16), and 2^-19 of the largest term that enters it (fp32 sums of up to
2048 terms, exp2 and one division).
"""
import pytest
import torch
import torch.nn.functional as F

from kerneldev_amd import _lib
from kerneldev_amd.gpt import RMSNorm, SwiGLU

pytestmark = pytest.mark.gpu


def _close(got, ref, dtype, scale):
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    tiny = 0.0 if dtype == torch.bfloat16 else 2.0 ** -25  # fp16's subnormal spacing
    err = (got.double() - ref).abs()
    assert bool((err <= ulp * 1.01 * ref.abs() + 2.0 ** -19 * scale + tiny).all()), (err / (ref.abs() + 1e-30)).max().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 8), (3, 5, 504), (2, 7, 512), (9, 520), (1, 4, 1024), (5, 1032), (2, 3, 2048)])
def test_rms_norm(dev, shape, dtype):
    g = torch.Generator("cpu").manual_seed(sum(shape))
    x = (torch.randn(shape, generator=g) * 3).to(dtype).to(dev).requires_grad_(True)
    dy = torch.randn(shape, generator=g).to(dtype).to(dev)
    y = RMSNorm()(x)
    assert "CppFunction" in type(y.grad_fn).__name__
    dx, = torch.autograd.grad(y, x, dy)
    x64 = x.detach().double().requires_grad_(True)
    r = torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-6)
    y64 = x64 * r
    want, = torch.autograd.grad(y64, x64, dy.double())
    _close(y.detach(), y64.detach(), dtype, y64.detach().abs())
    d = dy.double()
    terms = (r * (d.abs() + y64.abs() * (d * y64).abs().mean(-1, keepdim=True))).detach()
    _close(dx, want, dtype, terms)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 7, 8, 2048, 2055, 40000])
def test_gate(dev, n, dtype):
    g = torch.Generator("cpu").manual_seed(n)
    a, b, dy = ((torch.randn(n, generator=g) * s).to(dtype).to(dev) for s in (6, 2, 1))
    a[0] = -80.0  # exp(80) is finite in fp32; the gate is about -80 e^-80
    a.requires_grad_(True), b.requires_grad_(True)
    y = _lib.native().swiglu(a, b)
    da, db = torch.autograd.grad(y, (a, b), dy)
    a64, b64 = a.detach().double().requires_grad_(True), b.detach().double().requires_grad_(True)
    y64 = F.silu(a64) * b64
    wa, wb = torch.autograd.grad(y64, (a64, b64), dy.double())
    _close(y.detach(), y64.detach(), dtype, y64.detach().abs())
    # silu' = s + a s (1 - s): its two terms may cancel
    s = torch.sigmoid(a64.detach())
    _close(da, wa, dtype, (dy.double() * b64.detach()).abs() * (s + a64.detach().abs() * s * (1 - s)))
    _close(db, wb, dtype, wb.abs())


def test_the_eager_forms_where_the_kernels_do_not_apply(dev):
    x = torch.randn(4, 36, device=dev)
    for y in (x, x.bfloat16(), x.bfloat16()[:, :24], torch.randn(2, 4096, device=dev).bfloat16(), x.cpu().half()):
        assert RMSNorm()(y).shape == y.shape  # fp32, a width of 36, strided rows, wide rows, the CPU
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert RMSNorm()(x.bfloat16()[:, :32].contiguous()).dtype == torch.float32  # pow runs in fp32 there
    # second derivatives exist as for the eager forms
    m = SwiGLU(64, 128).to(dev).bfloat16()
    z = torch.randn(3, 64, device=dev).bfloat16().requires_grad_(True)
    out = m(RMSNorm()(z)).float().pow(2).sum()
    gz, = torch.autograd.grad(out, z, create_graph=True)
    gg, = torch.autograd.grad(gz.float().pow(2).sum(), z)
    z64 = z.detach().double().requires_grad_(True)
    w1, w2, w3 = (w.weight.detach().double() for w in (m.w1, m.w2, m.w3))
    n = z64 * torch.rsqrt(z64.pow(2).mean(-1, keepdim=True) + 1e-6)
    o64 = ((F.silu(n @ w1.T) * (n @ w3.T)) @ w2.T).pow(2).sum()
    g64, = torch.autograd.grad(o64, z64, create_graph=True)
    gg64, = torch.autograd.grad(g64.pow(2).sum(), z64)
    # bf16 activations and gradients between the layers: a few per cent of a second derivative
    assert (gg.double() - gg64).norm() <= 0.1 * gg64.norm()
    compiled = torch.compile(RMSNorm(), fullgraph=True)
    w = torch.randn(8, 64, device=dev).bfloat16()
    assert torch.allclose(compiled(w).float(), RMSNorm()(w).float(), rtol=2 ** -6)
    # forward-mode AD and vmap through the eager forms
    import torch.autograd.forward_ad as fw
    with fw.dual_level():
        t = fw.unpack_dual(RMSNorm()(fw.make_dual(w, torch.ones_like(w)))).tangent
        assert t is not None and t.shape == w.shape
    assert torch.vmap(RMSNorm())(w[None]).shape == (1, 8, 64)


def test_gradient_layout_follows_the_operand(dev):
    from kerneldev_amd import flash_attention

    x = torch.randn(2, 100, 3, 64, device=dev).bfloat16()
    q = x.transpose(1, 2).requires_grad_(True)  # [B, H, T, d] in [B, T, H, d] memory
    c = x.transpose(1, 2).contiguous().requires_grad_(True)
    do = torch.randn_like(c)
    gq, = torch.autograd.grad(flash_attention(q, q, q), q, do)
    gc, = torch.autograd.grad(flash_attention(c, c, c), c, do)
    assert torch.equal(gq, gc) and gq.stride() == q.stride() and gc.is_contiguous()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 128, 136), (64, 120, 128), (65, 256, 8), (200, 264, 520),
                                   (1000, 128, 128), (4097, 72, 200), (16384, 256, 256), (5000, 2048, 1024)])
def test_weight_gradient(dev, M, N, K, dtype):
    """Edges of the 64-token steps, the 128 x 128 tiles and the pieces of the tokens.  fp32 sums of M products
    (each exact): 2^-24 sqrt(M) of the root of the sum of squares, four times that and one rounding allowed."""
    from kerneldev_amd.gpt import Projection

    g = torch.Generator("cpu").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dtype).to(dev)
    dy = torch.randn(M, N, generator=g).to(dtype).to(dev)
    p = Projection(K, N).to(dev).to(dtype)
    x.requires_grad_(True)
    y = p(x)
    assert "CppFunction" in type(y.grad_fn).__name__
    dx, dw = torch.autograd.grad(y, (x, p.weight), dy)
    ref = dy.double().t() @ x.detach().double()
    size = (dy.double().square().t() @ x.detach().double().square()).sqrt()
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (dw.double() - ref).abs()
    assert bool((err <= 1.01 * ulp * ref.abs() + 2.0 ** -22 * M ** 0.5 * size + 2.0 ** -25).all())
    want = dy.double() @ p.weight.detach().double()
    assert (dx.double() - want).norm() <= 2 * ulp * want.norm()


def test_projection_forms(dev):
    """The library's linear where the kernel does not apply, hooks, frozen weights and second derivatives."""
    from kerneldev_amd.gpt import Projection

    p = Projection(64, 72).to(dev).bfloat16()
    x = torch.randn(2, 5, 64, device=dev).bfloat16()
    seen = []
    p.register_forward_hook(lambda *a: seen.append(1))
    assert torch.equal(p(x), F.linear(x, p.weight)) and seen == [1]
    with torch.no_grad():
        assert p(x).grad_fn is None
    y = p(x.transpose(0, 1))
    assert y.shape == (5, 2, 72) and y.requires_grad
    with torch.autocast("cuda", dtype=torch.float16):
        assert p(x).dtype == torch.float16
    p.weight.requires_grad_(False)
    z = x.clone().requires_grad_(True)
    assert torch.autograd.grad(p(z).sum(), z)[0].shape == z.shape
    p.weight.requires_grad_(True)
    gz, = torch.autograd.grad(p(z).float().pow(2).sum(), z, create_graph=True)
    gw, = torch.autograd.grad(gz.float().sum(), p.weight)
    w64 = p.weight.detach().double().requires_grad_(True)
    g64, = torch.autograd.grad((2 * (z.detach().double() @ w64.T) @ w64).sum(), w64)
    assert (gw.double() - g64).norm() <= 0.05 * g64.norm()
    assert set(p.state_dict()) == {"weight"}


@pytest.mark.parametrize("D,own", [(8, False), (24, False), (32, True)])
def test_many_narrow_rows(dev, D, own):
    """Both sides of the rule on narrow rows: torch's expressions past 2^17 of them, unless they are 32 wide."""
    for rows, want in ((1 << 17, True), ((1 << 17) + 1, own)):
        x = torch.randn(rows, D, device=dev).bfloat16().requires_grad_(True)
        y = RMSNorm()(x)
        assert ("CppFunction" in type(y.grad_fn).__name__) == want
        ref = x.detach().double()
        ref = ref * torch.rsqrt(ref.pow(2).mean(-1, keepdim=True) + 1e-6)
        # torch's form rounds the square, the mean, the factor and the product to bf16 (2^-9 each)
        assert (y.detach().double() - ref).norm() <= 2.0 ** -7 * ref.norm()


def test_more_rows_than_a_launch_holds(dev):
    """2^26 rows of a wave each are 2^32 threads: the rows at every launch's ends, forward and backward."""
    rows, D = (1 << 26) + 5, 32
    x = torch.randn(rows, D, device=dev, dtype=torch.bfloat16, generator=torch.Generator(dev).manual_seed(1))
    dy = torch.randn(rows, D, device=dev, dtype=torch.bfloat16, generator=torch.Generator(dev).manual_seed(2))
    x.requires_grad_(True)
    y = RMSNorm()(x)
    assert "CppFunction" in type(y.grad_fn).__name__
    dx, = torch.autograd.grad(y, x, dy)
    at = torch.cat([torch.arange(max(0, i - 64), min(rows, i + 64)) for i in (0, 1 << 25, 1 << 26, rows)]).to(dev)
    x64 = x.detach()[at].double().requires_grad_(True)
    y64 = x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-6)
    want, = torch.autograd.grad(y64, x64, dy[at].double())
    # one rounding of fp32 results: 2^-9
    assert (y.detach()[at].double() - y64.detach()).norm() <= 2.0 ** -8 * y64.detach().norm()
    assert (dx[at].double() - want).norm() <= 2.0 ** -8 * want.norm()
