"""GPU: work lists cut into pieces (kd_attn_fwd_ws / kd_attn_bwd_ws, kd_combine.hip).

Small shapes whose lists are cut, against the fp64 oracle at the repository's
bars, at the places where pieces can go wrong: lists shorter than the piece
count (empty pieces), ragged ends, fully masked rows, narrow heads, the
rotation and residuals of the combining kernel, fp8 scores, fp32.  And against
the uncut entry points: O + O_lo, the only output with a residual here,
carries P to 16 bits whichever row maximum a piece took, so the two sums
differ by at most 2^-15 relative (rel-RMS).
"""
import ctypes

import pytest
import torch

from kerneldev_amd import _lib
from kerneldev_amd.attention import _attn_args, _fwd_op, _strides3
from kerneldev_amd.synth import CocktailLayout, cocktail_batch, qkvdo
from test_gpu_attention import _case

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _args(B, H, T, D, dtype):
    a = _lib.AttnArgs()
    a.B, a.H, a.T, a.D, a.sm_scale = B, H, T, D, D ** -0.5
    a.dtype = {BF: _lib.KD_BF16, HF: _lib.KD_F16, F32: _lib.KD_F32}[dtype]
    return a


def _cocktail(B, T, seed):
    lay = CocktailLayout((9, 40), (T // 4, T // 2), (3, 6), (5, T // 20))
    return cocktail_batch(B, T, lay, seed)[1:]


CASES = [
    # B, H, T, D, dtype, mask, options
    (1, 2, 1000, 64, BF, "causal", {}),
    (1, 3, 1537, 64, BF, "cocktail", dict(hadamard=True, hadamard_seed=2)),
    (1, 2, 1025, 128, HF, "cocktail", dict(hadamard=True)),
    (2, 1, 1111, 128, BF, "cocktail", dict(precision="ieee")),
    (1, 2, 1100, 128, BF, "causal", dict(qk_dtype="fp8_e4m3")),
    (1, 1, 2047, 32, HF, "cocktail", dict(precision="bf16")),
    (1, 1, 2000, 16, BF, "causal", {}),
    (1, 2, 900, 256, BF, "cocktail", {}),
    (1, 1, 700, 256, BF, "causal", dict(qk_dtype="fp8_e4m3")),
    (1, 2, 300, 64, F32, "causal", dict(precision="ieee")),
    (2, 1, 450, 128, F32, "cocktail", {}),
    (1, 1, 333, 256, F32, "cocktail", dict(precision="ieee")),
    (1, 4, 513, 32, F32, "causal", dict(precision="ieee")),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}H{c[1]}T{c[2]}d{c[3]}-{c[4]}-{c[5]}-{c[6]}")
@pytest.mark.parametrize("ragged", [False, True])
def test_pieces_against_the_oracle(dev, case, ragged):
    B, H, T, D, dtype, mask, kw = case
    lib, a = _lib.load(), _args(B, H, T, D, dtype)
    assert lib.kd_attn_fwd_ws_bytes(ctypes.byref(a)) > 0 and lib.kd_attn_bwd_ws_bytes(ctypes.byref(a)) > 0
    q, k, v, do = qkvdo(B, H, T, D, seed=31 + T, dtype=dtype)
    inp = dict(name=f"pieces {case}", q=q, k=k, v=v, do=do, causal=True)
    if mask == "cocktail":
        inp["in_span"], inp["span_id"], inp["is_prefix"] = _cocktail(B, T, seed=T)
    # ragged: most of the last tiles are empty, and their rows fully masked
    lens = torch.tensor([T * 2 // 5 + 7 * b for b in range(B)], dtype=torch.int32) if ragged else None
    _case(inp, dev, lens=lens, **kw)


def test_pieces_against_the_uncut_kernels(dev):
    B, H, T, D = 1, 2, 1500, 64
    q, k, v, do = (x.to(dev) for x in qkvdo(B, H, T, D, seed=5))
    meta = [x.to(dev) for x in _cocktail(B, T, seed=6)]
    sc, lib = D ** -0.5, _lib.load()
    o, lse, plan, o_lo, *_ = _fwd_op(q, k, v, None, *meta, sc, 0, True)
    a = _attn_args(q, k, v, sc)
    o2, lo2, lse2 = torch.empty_like(o), torch.empty_like(o_lo), torch.empty_like(lse)
    a.o, a.o_strides, a.o_lo, a.lse = o2.data_ptr(), _strides3(o2), lo2.data_ptr(), lse2.data_ptr()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.kd_attn_fwd(ctypes.byref(a), *_lib.plan_ref(plan), st), "kd_attn_fwd")
    torch.cuda.synchronize()
    x, y = o.double() + o_lo.double(), o2.double() + lo2.double()
    assert (x - y).norm() <= 2 ** -15 * y.norm()
    # |LSE| <= 2^5 here, formed from fp32 sums: a few units of 2^-18
    assert (lse - lse2).abs().max() <= 2 ** -16
    # a workspace that is too small is refused, and nothing runs
    need = lib.kd_attn_fwd_ws_bytes(ctypes.byref(a))
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    r = lib.kd_attn_fwd_ws(ctypes.byref(a), *_lib.plan_ref(plan), ctypes.c_void_p(ws.data_ptr()), need - 1, st)
    assert r == _lib.KD_ERR_INVALID


def test_pieces_capture(dev):
    """Forward and backward with pieces in one HIP graph, every replay equal to the eager result."""
    from kerneldev_amd import flash_attention

    q, k, v, do = (x.to(dev) for x in qkvdo(1, 2, 1200, 64, seed=8))
    xs = [x.clone().requires_grad_(True) for x in (q, k, v)]

    def step():
        return torch.autograd.grad(flash_attention(*xs), xs, do)

    want = [g.clone() for g in step()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = step()
    for _ in range(3):
        other = flash_attention(q.flip(2).contiguous(), k, v)
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want)) and torch.isfinite(other).all()


@pytest.mark.parametrize("B,H,T,D,dtype", [(1, 2, 1000, 64, BF), (1, 12, 700, 128, HF), (1, 2, 300, 32, F32)])
def test_full_lists_against_the_oracle(dev, B, H, T, D, dtype):
    """No mask: the lists are marked full, in the forward and the backward, which choose their own piece counts."""
    a = _args(B, H, T, D, dtype)
    a.lists = _lib.KD_LISTS_FULL
    lib = _lib.load()
    assert lib.kd_attn_fwd_ws_bytes(ctypes.byref(a)) > 0 or lib.kd_attn_bwd_ws_bytes(ctypes.byref(a)) > 0
    q, k, v, do = qkvdo(B, H, T, D, seed=T, dtype=dtype)
    _case(dict(name=f"full {B} {H} {T} {D}", q=q, k=k, v=v, do=do, causal=False), dev)
