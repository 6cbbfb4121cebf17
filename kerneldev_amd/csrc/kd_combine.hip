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

// How many pieces.  A block's list is a serial chain of up to nT = T / 64 tile
// steps, so with fewer workgroups than the chip holds the longest list is the
// kernel's time.  Pieces shorten it, and cost the partial results' way through
// memory (ns rows D floats written and read), a second launch, each piece's own
// start, and more workgroups on a CU.  The count is the one with the least of
//   steps of a piece x us a step x (1 + crowd (k - 1) share) + starts + cost
// where k = workgroups a CU (256 CUs), crowd what each further one on a CU costs a
// step (full masks, us a step at one, two, three and four workgroups a CU: fp32 d64
// forward 3.1, 4.9, 6.9, 9.0; bf16 d64 dQ 1.07, 2.06; bf16 d128 dK/dV, whose LDS holds
// one, 2.2, 5.3), and share how much of that is met by lists of uneven length,
// where a long list runs beside short ones: all of it for full masks (every list as
// long), a quarter where an XCD's first 64 workgroups are one head's, longest
// first, so that the upper half of its lists runs beside the lower, about half to two
// thirds elsewhere.  It has to save a tenth of the uncut time.
//
// Fitted to and checked on every pass of 648 shapes (B 1 and 4, W = 4 .. 1536
// workgroups, T 512 .. 8192, d 32 .. 256, bf16 and fp32) under full, causal and
// cocktail masks, timed at each count: 1.26 times faster than uncut in the geometric
// mean, and 5 of 5832 slower by more than 1.5% (the worst 1.04 x).  The rule before it
// knew neither k nor the mask: 1.24 times faster, 361 slower, up to 1.43 x.  Some, us
// (forward / dQ / dK+dV):
//   bf16 B1 H8 T4096 d128 causal (W 256): 96 / 102 / 135 -> 77 / 88 / 114 at 2
//   bf16 B1 H16 T2048 d64 causal (W 256): 39 / 36 / 50, 42 / 41 / 56 at 2: uncut
//   bf16 B1 H12 T1400 d128 full (W 132): dK+dV 53, 76 at 2: uncut
//   bf16 B1 H1 T8192 d64 causal (W 64): 132 / 134 / 160 -> 44 / 57 / 45 at 4
//   fp32 B1 H8 T2048 d128 causal (W 256): 168 / 222 / 299 -> 123 / 161 / 214 at 2
//   fp32 B1 H32 T512 d64 causal (W 256): 28.7 / 35 / 48, 35 / 42 / 51 at 4: uncut
int split_pieces(const AttnArgs& a, SplitPass pass) {
  const bool f32 = use_simt(a), full = a.lists == KD_LISTS_FULL;
  const int nT = (a.T + 63) / 64, nblk = (nT + 1) / 2;
  const int64_t rows = int64_t(a.B) * a.H * a.T, per_head = int64_t(a.B) * nblk * (f32 ? 2 : 1), W = per_head * a.H;
  const int d = a.D <= 32 ? 0 : a.D == 64 ? 1 : a.D == 128 ? 2 : 3, outs = pass == SPLIT_DKDV ? 2 : 1;
  if (W > (f32 ? 2048 : 512)) return 1;  // (several a CU already; 16-bit lists are cut in three and more there at a loss)
  constexpr float step16[4][3] = {{1.0f, 0.85f, 1.2f}, {1.15f, 1.07f, 1.55f}, {1.6f, 1.7f, 2.2f}, {3.0f, 5.2f, 6.7f}};
  constexpr float crowd16[4][3] = {
      {0.5f, 0.55f, 0.65f}, {0.75f, 0.95f, 0.95f}, {0.95f, 1.15f, 1.5f}, {1.2f, 1.25f, 1.2f}};
  constexpr float step32[4] = {2.1f, 3.1f, 5.3f, 10.2f}, pass32[3] = {1.0f, 1.27f, 1.75f};
  constexpr float crowd32[4] = {0.5f, 0.65f, 0.83f, 1.02f};
  const float single = a.precision == KD_PREC_SINGLE ? 0.7f : 1.f;  // P and dS rounded once: fewer products
  const float step = f32 ? step32[d] * pass32[pass] : step16[d][pass] * single, crowd = f32 ? crowd32[d] : crowd16[d][pass];
  const float start = (f32 ? 0.75f : 0.5f) * (1.f + 0.4f * float(d));
  auto us = [&](int ns) {
    const int k = int((W * ns + 255) / 256);
    float share = 1.f;
    if (!full) {
      if (ns == 1) share = k == 2 ? 0.35f : 0.67f;
      else if (k > 2) share = 0.67f;
      else if (a.H % 8 == 0 && per_head * ns >= 64 && nT >= 16) share = 0.25f;
      else share = pass == SPLIT_FWD && !f32 ? 0.6f : 0.5f;
    }
    const float t = float((nT + ns - 1) / ns) * step * (1.f + crowd * float(k - 1) * share) + start * float(k);
    return ns == 1 ? t : t + 4.5f + 1.4e-6f * float(ns * outs) * float(rows) * float(a.D);
  };
  const float whole = us(1);
  float least = 0.9f * whole;
  int best = 1;
  for (int ns = 2; ns <= (f32 ? 6 : 4); ++ns) {
    // two steps a piece; fp32, whose steps are longer, one where each piece has its CU to itself
    if (nT < (f32 && W * ns <= 256 ? 1 : 2) * ns) continue;
    if (const float t = us(ns); t < least) least = t, best = ns;
  }
  // fp32 lists of uneven length and 64 steps or more, whole heads an XCD: the lists of
  // an XCD's last head are the kernel's tail however many come before.  Causal, forward
  // and whole backward: B2 H8 T4096 d128 (W 1024) 647 / 2060 -> 625 / 1969, B1 H8 T8192 d128
  // 1278 / 4069 -> 1192 / 3746, B1 H16 T4096 d64 433 / 1263 -> 351 / 1125.  Not at d = 256 (1364 -> 1435).
  if (best == 1 && f32 && !full && a.D <= 128 && a.H % 8 == 0 && nT >= 64 && W <= 1024) best = 2;
  return best;
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
