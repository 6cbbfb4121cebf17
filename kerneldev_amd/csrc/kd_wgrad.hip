// Weight gradients of the block's projections: dW [N, K] = dY^T X over M
// tokens, dY [M, N] and X [M, K] in bf16 or fp16, row-major.
//
// The contraction runs over the tokens, the slow dimension of both operands,
// and the result is small (768 x 768 .. 2048 x 768 against 16384 tokens), so a
// product needs its tokens split to fill the chip.  A workgroup takes 128 x 128
// of dW over one piece of the tokens: 64 tokens a step of both operands go to
// LDS (two slots of 2 x 16 KiB, so two workgroups share a CU), and both MFMA
// operands are read transposed from there (ds_read_b64_tr_b16), four waves
// taking 64 x 64 each: one operand read a MFMA, at which the LDS keeps the
// matrix cores about three quarters busy.  The pieces' fp32 results are added
// in ascending order by a second kernel and rounded once.  Items are
// piece-major, so an XCD's workgroups read the same tokens through its L2.
#include <cmath>

#include "kd_tile.h"

namespace kd {
namespace {

constexpr int WT = 128;  // rows and columns of dW a workgroup takes

struct WgradArgs {
  const void *dy, *x;
  float* part;      // [S][N][K]
  int M, N, K, S;   // S pieces of the tokens
  int tn, tk;       // tiles of dW
};

template <class E>
__global__ __launch_bounds__(256, 2) void k_wgrad(WgradArgs w) {
  using TL = Tile<WT, 4>;
  __shared__ __attribute__((aligned(1024))) uint8_t s_y[2][TL::BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t s_x[2][TL::BYTES];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, hf = lane >> 5,
            c = lane & 31;
  const int item = xcd_remap(blockIdx.x, gridDim.x), tiles = w.tn * w.tk;
  const int piece = item / tiles, tile = item - piece * tiles;
  const int n0 = (tile / w.tk) * WT, k0 = (tile - (tile / w.tk) * w.tk) * WT;
  const int steps_all = (w.M + 63) / 64;
  const int e0 = int(int64_t(steps_all) * piece / w.S), e1 = int(int64_t(steps_all) * (piece + 1) / w.S);
  const uint32_t yrb = uint32_t(w.N) * 2u, xrb = uint32_t(w.K) * 2u;
  const u32x4 rs_y = rsrc_words(w.dy, uint32_t(w.M) * yrb), rs_x = rsrc_words(w.x, uint32_t(w.M) * xrb);
  uint32_t yoff[TL::LOADS_PER_WAVE], xoff[TL::LOADS_PER_WAVE];  // (columns past N, K read as zeros)
  TL::load_offsets(wave, lane, yrb, yoff, yrb - uint32_t(n0) * 2u);
  TL::load_offsets(wave, lane, xrb, xoff, xrb - uint32_t(k0) * 2u);
  auto load = [&](int e, int slot) {
    TL::load_async(rs_y, uint32_t(e) * 64u * yrb + uint32_t(n0) * 2u, yoff, lds_addr(s_y[slot]), wave);
    TL::load_async(rs_x, uint32_t(e) * 64u * xrb + uint32_t(k0) * 2u, xoff, lds_addr(s_x[slot]), wave);
  };
  // this wave's 64 x 64: column blocks 2 wn, 2 wn + 1 of the dY tile against 2 wk, 2 wk + 1 of the X tile
  const int wn = wave >> 1, wk = wave & 1;
  int ya[2][2], xa[2][2];  // transposed-read offsets [column block][half], a k-step adds 16 rows
  {
    const int i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int r = 8 * (g >> 1) + 4 * half + (i >> 2), ch = 2 * (g & 1) + ((i & 3) >> 1);
        ya[b][half] = TL::at(r, 4 * (2 * wn + b) + ch) + 8 * (i & 1);
        xa[b][half] = TL::at(r, 4 * (2 * wk + b) + ch) + 8 * (i & 1);
      }
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x16{};

  if (e0 < e1) load(e0, 0);
  auto step = [&](int e, auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
    wait_vmem();
    barrier_raw();  // step e's tiles landed for every wave; every wave is done with the other slot
    if (e + 1 < e1) load(e + 1, slot ^ 1);
    lds_u8 *ty = to_lds(s_y[slot]), *tx = to_lds(s_x[slot]);
    auto read = [&](lds_u8* t, const int (&at)[2], int ks) {
      const u32x2 lo = ds_read_tr16(t + at[0] + ks * 16 * TL::ROWB);
      const u32x2 hi = ds_read_tr16(t + at[1] + ks * 16 * TL::ROWB);
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
    // operands of k-step ks + 1 are read before the MFMAs of k-step ks
    u32x4 av[2][2], bv[2][2];  // [k-step parity][block]
#pragma unroll
    for (int b = 0; b < 2; ++b) av[0][b] = read(ty, ya[b], 0), bv[0][b] = read(tx, xa[b], 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      __builtin_amdgcn_sched_barrier(0x406);
      if (ks + 1 < 4) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
          av[(ks + 1) & 1][b] = read(ty, ya[b], ks + 1), bv[(ks + 1) & 1][b] = read(tx, xa[b], ks + 1);
      }
      __builtin_amdgcn_sched_barrier(0x406);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mfma32x32x16<E>(av[ks & 1][a], bv[ks & 1][b], acc[a][b]);
    }
    __builtin_amdgcn_sched_barrier(0x406);
  };
  for (int e = e0; e < e1; e += 2) {
    step(e, std::integral_constant<int, 0>{});
    if (e + 1 < e1) step(e + 1, std::integral_constant<int, 1>{});
  }
  float* out = w.part + int64_t(piece) * w.N * w.K;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = k0 + 64 * wk + 32 * b + c;
#pragma unroll
      for (int r = 0; r < 16; ++r) {  // register r: row 8 (r / 4) + 4 hf + r % 4 of the 32 x 32 block
        const int n = n0 + 64 * wn + 32 * a + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (n < w.N && k < w.K) out[int64_t(n) * w.K + k] = acc[a][b][r];
      }
    }
}

// dW = the pieces' sum, rounded once; eight elements a thread (N K is a multiple of 64)
template <class E>
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* __restrict__ part, uint16_t* __restrict__ dw, int64_t n,
                                                   int S) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i >= n) return;
  float f[8] = {};
#pragma unroll 4
  for (int s = 0; s < S; ++s) {
    const f32x4* p = reinterpret_cast<const f32x4*>(part + s * n + i);
    const f32x4 u = p[0], v = p[1];
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] += u[k], f[4 + k] += v[k];
  }
  *reinterpret_cast<u32x4*>(dw + i) = pack8<E>(f);
}

}  // namespace

// Pieces: a step of 64 tokens takes a workgroup 0.45 us with two on a CU, and a
// piece's N K floats go to memory and back at about 5 TB/s; steps / S * 0.45 us +
// S N K 1.6e-6 us is least at the root below.  No more than two workgroups a CU.
int wgrad_pieces(int M, int N, int K) {
  const int tiles = ((N + WT - 1) / WT) * ((K + WT - 1) / WT), steps = (M + 63) / 64;
  const int best = int(std::sqrt(281250.0 * steps / (double(N) * K)) + 0.5);
  return std::max(1, std::min(std::min(best, steps), 512 / tiles));
}

int launch_wgrad(const void* dy, const void* x, void* dw, float* part, int M, int N, int K, int dtype, hipStream_t st) {
  WgradArgs w{dy, x, part, M, N, K, wgrad_pieces(M, N, K), (N + WT - 1) / WT, (K + WT - 1) / WT};
  const int64_t n = int64_t(N) * K;
  auto go = [&](auto e) {
    using E = decltype(e);
    hipLaunchKernelGGL(k_wgrad<E>, dim3(unsigned(w.tn * w.tk * w.S)), dim3(256), 0, st, w);
    hipLaunchKernelGGL(k_wgrad_sum<E>, dim3(unsigned((n / 8 + 255) / 256)), dim3(256), 0, st, part,
                       static_cast<uint16_t*>(dw), n, w.S);
  };
  if (dtype == KD_BF16) go(BF16{});
  else go(F16{});
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

}  // namespace kd
