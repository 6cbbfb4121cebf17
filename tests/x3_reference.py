"""The packing of the bf16x3 path in torch operations: what kd_x3_pack and kd_x3_unpack
(csrc/kd_x3.hip) compute, for the tests of the layout and of the kernels."""
import torch


def x3(x, pattern, Dp):
    """[B, H, T, d] fp32 -> contiguous bf16 [B, H, T, Dp]: the parts named by pattern ('h', 'l'), then zeros."""
    xh = x.to(torch.bfloat16)
    xl = (x - xh.to(torch.float32)).to(torch.bfloat16)
    parts = [xh if c == "h" else xl for c in pattern]
    pad = Dp - len(pattern) * x.shape[-1]
    if pad:
        parts.append(xh.new_zeros(x.shape[:-1] + (pad,)))
    return torch.cat(parts, dim=-1)


def hi_lo(hi, lo, d, second):
    """fp32 (hi + lo)[..., 0:d] + (hi + lo)[..., second * d:(second + 1) * d]."""
    x = hi.to(torch.float32).add_(lo.to(torch.float32))
    return x[..., :d] + x[..., second * d:(second + 1) * d]
