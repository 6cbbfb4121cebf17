// Pieces of one row's work list, put together.
//
// Where a shape has fewer row (or key) blocks than the chip has slots for
// them, the attention kernels cut every block's list into SplitArgs::ns
// pieces, one workgroup each, and leave fp32 partial results here:
//   forward     O of the piece, not normalised, with its row maximum (in log2
//               units) and its row sum:  O = sum_s w_s O_s / sum_s w_s l_s,
//               w_s = exp2(m_s - max m),  LSE2 = max m + log2(sum_s w_s l_s)
//   dQ, dK, dV  the piece's sum of products; the pieces add up
// The pieces are added in ascending order, so a result does not depend on the
// order in which workgroups finish.
//
// Bound by memory: ns (D + 2) floats a row are read once and a row of the
// output written.  One lane takes four columns, so a row's lanes read whole
// 16-byte words side by side.
#include <type_traits>

#include "kd_internal.h"

namespace kd {
namespace {

struct OutRow {
  void* p;            // output, element strides below
  int64_t st[3];      // b, h, t
  void* lo;           // contiguous rounding residuals [B, H, T, D], or NULL
  float scale;
  const float* signs;  // rotate back by R^T (R = diag(s) H_D / sqrt(D)), or NULL
};

struct CombineArgs {
  const float* part;   // [ns][rows][D] of output 0, then of output 1
  const float* ml;     // forward: [ns][rows][2]
  float* lse;          // forward
  OutRow out[2];
  int64_t rows;
  int H, T, D, ns;
  int lanes_log2;      // lanes a row, log2(D / 4)
  bool lo32;           // residuals in fp32 (precision KD_PREC_SPLIT3)
};

template <class E>
KD_DEV void store4(const OutRow& o, const CombineArgs& c, int64_t row, int col, const float (&f)[4]) {
  const int t = int(row % c.T), bh = int(row / c.T), b = bh / c.H, h = bh - b * c.H;
  const int64_t at = b * o.st[0] + h * o.st[1] + t * o.st[2] + col;
  if constexpr (std::is_same<E, F32>::value) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(o.p) + at) = f32x4{f[0], f[1], f[2], f[3]};
  } else {
    const u32x2 w = {pack2<E>(f[0], f[1]), pack2<E>(f[2], f[3])};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(o.p) + at) = w;
    if (o.lo == nullptr) return;
    if (c.lo32)
      *reinterpret_cast<f32x4*>(static_cast<float*>(o.lo) + row * c.D + col) =
          f32x4{f[0] - to_f32<E>(uint16_t(w[0] & 0xFFFFu)), f[1] - to_f32<E>(uint16_t(w[0] >> 16)),
                f[2] - to_f32<E>(uint16_t(w[1] & 0xFFFFu)), f[3] - to_f32<E>(uint16_t(w[1] >> 16))};
    else
      *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(o.lo) + row * c.D + col) =
          u32x2{pack2_residual<E>(f[0], f[1], w[0]), pack2_residual<E>(f[2], f[3], w[1])};
  }
}

template <class E>
__global__ __launch_bounds__(256) void k_combine_fwd(CombineArgs c) {
  const int lane = int(threadIdx.x) & ((1 << c.lanes_log2) - 1);
  const int64_t row = int64_t(blockIdx.x) * (256 >> c.lanes_log2) + (threadIdx.x >> c.lanes_log2);
  if (row >= c.rows) return;
  const float NEG_INF = -__builtin_inff();
  float m = NEG_INF;
  for (int s = 0; s < c.ns; ++s) m = fmaxf(m, c.ml[2 * (s * c.rows + row)]);
  float l = 0.f, o[4] = {};
  for (int s = 0; s < c.ns; ++s) {
    const f32x2 ml = *reinterpret_cast<const f32x2*>(c.ml + 2 * (s * c.rows + row));
    const f32x4 x = *reinterpret_cast<const f32x4*>(c.part + (s * c.rows + row) * c.D + 4 * lane);
    const float w = ml[0] == NEG_INF ? 0.f : fast_exp2(ml[0] - m);
    l = __builtin_fmaf(w, ml[1], l);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(w, x[i], o[i]);
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] *= inv;
  store4<E>(c.out[0], c, row, 4 * lane, o);
  if (c.lse != nullptr && lane == 0) c.lse[row] = l > 0.f ? m + fast_log2(l) : NEG_INF;
}

// blockIdx.y: which of the outputs (dQ; or dV, dK)
template <class E>
__global__ __launch_bounds__(256) void k_combine_grad(CombineArgs c) {
  const OutRow& out = c.out[blockIdx.y];
  const int lane = int(threadIdx.x) & ((1 << c.lanes_log2) - 1);
  const int64_t row = int64_t(blockIdx.x) * (256 >> c.lanes_log2) + (threadIdx.x >> c.lanes_log2);
  const int64_t at = row < c.rows ? row : c.rows - 1;  // (lanes past the end still join the exchanges below)
  const float* p = c.part + (int64_t(blockIdx.y) * c.ns * c.rows + at) * c.D + 4 * lane;
  float g[4] = {};
  for (int s = 0; s < c.ns; ++s) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(p + s * c.rows * c.D);
#pragma unroll
    for (int i = 0; i < 4; ++i) g[i] += x[i];
  }
  float scale = out.scale;
  if (out.signs != nullptr) {  // Walsh-Hadamard butterflies: strides 1, 2 in the lane, 4 .. D / 2 across lanes
#pragma unroll
    for (int hs = 1; hs < 4; hs <<= 1)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j & hs) continue;
        const float u = g[j], v = g[j + hs];
        g[j] = u + v;
        g[j + hs] = u - v;
      }
    for (int m = 1; m < (1 << c.lanes_log2); m <<= 1)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float other = __shfl_xor(g[j], m, 64);
        g[j] = (lane & m) ? other - g[j] : g[j] + other;
      }
    scale *= c.D == 128 ? 0.088388347648318440f : 0.125f;  // / sqrt(D); built at D = 64 and 128
#pragma unroll
    for (int j = 0; j < 4; ++j) g[j] *= out.signs[4 * lane + j] * scale;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) g[j] *= scale;
  }
  if (row < c.rows) store4<E>(out, c, row, 4 * lane, g);
}

OutRow out_row(void* p, const int64_t* st, void* lo, float scale, const float* signs) {
  return OutRow{p, {st[0], st[1], st[2]}, lo, scale, signs};
}

CombineArgs combine_args(const AttnArgs& a, const SplitArgs& sp) {
  CombineArgs c{};
  c.part = sp.part;
  c.rows = int64_t(a.B) * a.H * a.T;
  c.H = a.H;
  c.T = a.T;
  c.D = a.D;
  c.ns = sp.ns;
  c.lanes_log2 = __builtin_ctz(unsigned(a.D / 4));
  c.lo32 = a.precision == KD_PREC_SPLIT3;
  return c;
}

int launch(const AttnArgs& a, const CombineArgs& c, bool fwd, int outputs, hipStream_t st) {
  const int64_t rpb = 256 >> c.lanes_log2;
  const dim3 grid(unsigned((c.rows + rpb - 1) / rpb), unsigned(outputs)), block(256);
  auto go = [&](auto e) {
    using E = decltype(e);
    if (fwd) hipLaunchKernelGGL(k_combine_fwd<E>, grid, block, 0, st, c);
    else hipLaunchKernelGGL(k_combine_grad<E>, grid, block, 0, st, c);
  };
  if (a.dtype == KD_BF16) go(BF16{});
  else if (a.dtype == KD_F16) go(F16{});
  else go(F32{});
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

}  // namespace

// How many pieces.  A block's list is a serial chain of up to T / 64 tile
// steps, so with fewer workgroups than the chip holds the longest list is the
// kernel's time.  Pieces shorten it, and cost the partial results' way through
// memory (ns rows D floats written and read, at ~5.9 TB/s), a second launch and
// each piece's own start (4 us together).  The lines below come from sweeps of
// ns = 1 .. 8 on causal and full masks (us, forward / dQ / dK+dV; bf16 and causal
// unless said; W = workgroups without pieces):
//   B1 H12 T1531 d64  (W 144):  37 / 36 / 39   -> 27.5 / 28 / 33  at 3
//   B1 H8 T4095 d128  (W 256):  110 / 120 / 139 -> 82 / 96 / 116  at 2
//   B1 H1 T8192 d64   (W 64):   132 / 134 / 160 -> 44 / 57 / 45   at 4
//   B1 H8 T2048 d256  (W 128):  99 / 170 / 238 -> 61 / 108 / 128  at 3
//   B2 H8 T1531 d64, full (W 192): 35 -> 37 at 2 and 3, 35 at 4: no gain left
//   B4 H8 T395 d128   (W 128):  17 -> 22 at 2: lists of 7 tiles are too short
//   B2 H8 T4096 d64   (W 512):  80 -> 79 at 2, 81 at 3: no pieces from here on
//   fp32 B1 H8 T2048 d128 (W 256): 170 / 230 / 296 -> 102 / 145 / 188 at 3
//   fp32 B4 H8 T777 d64   (W 448): 60 / 77 / 90 -> 49 / 64 / 78 at 2
//   fp32 B8 H8 T395 d128  (W 512): 59 -> 63 at 2, full 75 -> 95
//   fp32 B2 H8 T4096 d128 (W 1024): 647 -> 626 at 2: long causal lists only
// 16-bit: pieces of two tiles or more while each has a CU to itself, of six or
// more up to two a CU (at d = 256, where one fills a CU, up to one and a half).
// fp32 (two workgroups a block, a tile takes four times as long): one tile a
// piece, up to two (d = 256), three (128) or four workgroups a CU.  And what a
// piece saves has to be 1.45 times what it costs.
int split_pieces(const AttnArgs& a, SplitPass pass) {
  const bool f32 = use_simt(a);
  const int nT = (a.T + 63) / 64, nblk = (nT + 1) / 2;
  const int64_t rows = int64_t(a.B) * a.H * a.T, W = int64_t(a.B) * a.H * nblk * (f32 ? 2 : 1);
  const int d = a.D <= 32 ? 0 : a.D == 64 ? 1 : a.D == 128 ? 2 : 3;
  // us a tile step takes a workgroup that has its CU to itself
  constexpr float step16[4] = {1.0f, 1.0f, 1.7f, 3.0f}, step32[4] = {2.0f, 3.0f, 5.3f, 10.6f};
  constexpr float pass16[3] = {1.0f, 1.1f, 1.25f}, pass32[3] = {1.0f, 1.3f, 1.8f};
  constexpr int64_t room32[4] = {1024, 1024, 768, 512};
  const float step = f32 ? step32[d] * pass32[pass] : step16[d] * pass16[pass];
  const int outs = pass == SPLIT_DKDV ? 2 : 1;
  for (int ns = f32 ? 6 : 4; ns > 1; --ns) {
    const int64_t wg = W * ns;
    const bool room = f32 ? nT >= ns && (wg <= (ns > 4 ? 256 : room32[d]) || (wg <= 2048 && nT >= 32 * ns))
                          : (wg <= 256 && nT >= 2 * ns) || (wg <= (a.D == 256 ? 384 : 512) && nT >= 6 * ns);
    const float saved = step * float(nT) * (1.f - 1.f / float(ns));
    const float cost = 4.f + 1.4e-6f * float(ns * outs) * float(rows) * float(a.D);
    if (room && saved > 1.45f * cost) return ns;
  }
  return 1;
}

int64_t split_floats(const AttnArgs& a, SplitPass pass) {
  const int64_t ns = split_pieces(a, pass), rows = int64_t(a.B) * a.H * a.T;
  if (ns == 1) return 0;
  return ns * rows * (pass == SPLIT_FWD ? a.D + 2 : pass == SPLIT_DQ ? a.D : 2 * a.D);
}

int launch_combine_fwd(const AttnArgs& a, const SplitArgs& sp, hipStream_t st) {
  CombineArgs c = combine_args(a, sp);
  c.ml = split_ml(a, sp);
  c.lse = a.lse;
  c.out[0] = out_row(a.o, a.o_strides, a.o_lo, 1.f, nullptr);
  return launch(a, c, true, 1, st);
}

int launch_combine_dq(const AttnArgs& a, const SplitArgs& sp, hipStream_t st) {
  CombineArgs c = combine_args(a, sp);
  c.out[0] = out_row(a.dq, a.dq_strides, a.dq_lo, a.sm_scale, a.dqk_signs);
  return launch(a, c, false, 1, st);
}

int launch_combine_dkdv(const AttnArgs& a, const SplitArgs& sp, hipStream_t st) {
  CombineArgs c = combine_args(a, sp);
  c.out[0] = out_row(a.dv, a.dv_strides, a.dv_lo, 1.f, nullptr);
  c.out[1] = out_row(a.dk, a.dk_strides, a.dk_lo, a.sm_scale, a.dqk_signs);
  return launch(a, c, false, 2, st);
}

}  // namespace kd
