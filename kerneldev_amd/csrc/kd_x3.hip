// The operands of the bf16x3 route: fp32 rows of d values as bf16 rows of Dp >=
// 3 d, and back.  x = h + l with h = bf16(x), l = bf16(x - h); a packed row is
// [h, h, l] (Q, dO) or [h, l, h] (K, V), zeros behind, so that one product of
// packed rows is the three products of the parts (attention.py).  Unpacking adds
// a result's rounding residual and its two blocks that hold h, in fp32.
//
// One launch packs all operands of a pass and one unpacks all its results
// (blockIdx.y: which), 16 bytes of bf16 a lane; formed with torch operations
// the same took about 25 launches a forward and backward, the whole of a small
// step's time (fp32 B2 H62 T90 d32: 750 us).
#include "kd_internal.h"

namespace kd {
namespace {

KD_DEV const float* row_of(const kd_x3_args& a, const void* base, const int64_t* st, int64_t row) {
  const int t = int(row % a.T), bh = int(row / a.T), b = bh / a.H, h = bh - b * a.H;
  return static_cast<const float*>(base) + b * st[0] + h * st[1] + t * st[2];
}

__global__ __launch_bounds__(256) void k_x3_pack(kd_x3_args a, int wpr) {  // wpr: 8-column words of a packed row
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x, row = i / wpr;
  if (row >= int64_t(a.B) * a.H * a.T) return;
  const int which = blockIdx.y, col = int(i - row * wpr) * 8, part = col / a.d;
  u32x4 out{};
  if (part < 3) {
    const float* p = row_of(a, a.src[which], a.src_strides[which], row) + (col - part * a.d);
    const f32x4 u = *reinterpret_cast<const f32x4*>(p), v = *reinterpret_cast<const f32x4*>(p + 4);
    const float f[8] = {u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]};
    out = pack8<BF16>(f);
    if (part == (a.sel[which] == 0 ? 2 : 1)) out = pack8_residual<BF16>(f, out);
  }
  *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(a.dst[which]) + row * a.Dp + col) = out;
}

__global__ __launch_bounds__(256) void k_x3_unpack(kd_x3_args a, int wpr) {  // wpr: 8-column words of an fp32 row
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x, row = i / wpr;
  if (row >= int64_t(a.B) * a.H * a.T) return;
  const int which = blockIdx.y, col = int(i - row * wpr) * 8;
  float f[8];
  auto sum = [&](int c, float (&x)[8]) {
    const u32x4 h = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.src[which]) + row * a.Dp + c);
    const u32x4 l = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.lo[which]) + row * a.Dp + c);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      x[2 * w] = to_f32<BF16>(uint16_t(h[w] & 0xFFFFu)) + to_f32<BF16>(uint16_t(l[w] & 0xFFFFu));
      x[2 * w + 1] = to_f32<BF16>(uint16_t(h[w] >> 16)) + to_f32<BF16>(uint16_t(l[w] >> 16));
    }
  };
  float g[8];
  sum(col, f);
  sum(a.sel[which] * a.d + col, g);
  float* out = const_cast<float*>(row_of(a, a.dst[which], a.dst_strides[which], row)) + col;
  *reinterpret_cast<f32x4*>(out) = f32x4{f[0] + g[0], f[1] + g[1], f[2] + g[2], f[3] + g[3]};
  *reinterpret_cast<f32x4*>(out + 4) = f32x4{f[4] + g[4], f[5] + g[5], f[6] + g[6], f[7] + g[7]};
}

}  // namespace

int launch_x3(const kd_x3_args& a, bool pack, hipStream_t st) {
  const int wpr = (pack ? a.Dp : a.d) / 8;
  const int64_t words = int64_t(a.B) * a.H * a.T * wpr;
  const dim3 grid(unsigned((words + 255) / 256), unsigned(a.n));
  if (pack) hipLaunchKernelGGL(k_x3_pack, grid, dim3(256), 0, st, a, wpr);
  else hipLaunchKernelGGL(k_x3_unpack, grid, dim3(256), 0, st, a, wpr);
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

}  // namespace kd
