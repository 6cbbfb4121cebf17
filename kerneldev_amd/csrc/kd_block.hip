// The elementwise parts of the transformer block (model.py:31-52): RMSNorm
// without a weight, y = x rsqrt(mean(x^2) + eps), and the SwiGLU gate,
// y = silu(a) b, forward and backward, for bf16 and fp16.
//
// All four are bound by memory: each input is read once and each output
// written once, 16 bytes a lane, with fp32 arithmetic between and one rounding
// at the end (the eager forms round after every operation and move each
// intermediate through memory; B8 T2048, D 768 and hidden 2048, bf16, us:
// norm 36 -> 10 forward, 100 -> 14 backward; gate 61 -> 33 and 96 -> 51).
#include <algorithm>

#include "kd_internal.h"

namespace kd {
namespace {

template <class E>
KD_DEV void unpack8(const u32x4& v, float (&f)[8]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f[2 * w] = to_f32<E>(uint16_t(v[w] & 0xFFFFu));
    f[2 * w + 1] = to_f32<E>(uint16_t(v[w] >> 16));
  }
}

KD_DEV float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// One wave a row of D = 8 n columns (n <= 64 NCH): lane l holds the 16-byte
// words l, l + 64, ...; the row stays in registers between its sum and its
// output.  rstd [rows] is kept for the backward.
template <class E, int NCH>
__global__ __launch_bounds__(256) void k_rms_fwd(const u32x4* __restrict__ x, u32x4* __restrict__ y,
                                                 float* __restrict__ rstd, int64_t rows, int words, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const u32x4* p = x + row * words;
  float f[NCH][8], sum = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int w = lane + 64 * c;
    unpack8<E>(w < words ? p[w] : u32x4{}, f[c]);
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = __builtin_fmaf(f[c][i], f[c][i], sum);
  const float r = 1.f / sqrtf(wave_sum(sum) / float(8 * words) + eps);
  if (lane == 0 && rstd != nullptr) rstd[row] = r;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int w = lane + 64 * c;
#pragma unroll
    for (int i = 0; i < 8; ++i) f[c][i] *= r;
    if (w < words) y[row * words + w] = pack8<E>(f[c]);
  }
}

// dx = r (dy - x r^2 mean(dy x))
template <class E, int NCH>
__global__ __launch_bounds__(256) void k_rms_bwd(const u32x4* __restrict__ x, const u32x4* __restrict__ dy,
                                                 const float* __restrict__ rstd, u32x4* __restrict__ dx, int64_t rows,
                                                 int words) {
  const int lane = threadIdx.x & 63;
  const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float f[NCH][8], g[NCH][8], dot = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int w = lane + 64 * c;
    unpack8<E>(w < words ? x[row * words + w] : u32x4{}, f[c]);
    unpack8<E>(w < words ? dy[row * words + w] : u32x4{}, g[c]);
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) dot = __builtin_fmaf(f[c][i], g[c][i], dot);
  const float r = rstd[row], m = wave_sum(dot) / float(8 * words) * r * r;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int w = lane + 64 * c;
#pragma unroll
    for (int i = 0; i < 8; ++i) g[c][i] = r * (g[c][i] - f[c][i] * m);
    if (w < words) dx[row * words + w] = pack8<E>(g[c]);
  }
}

KD_DEV float sigmoid(float x) { return 1.f / (1.f + fast_exp2(x * -1.4426950408889634f)); }

// one 16-byte word of each operand a thread; the last n % 8 elements one by one
template <class E>
__global__ __launch_bounds__(256) void k_gate_fwd(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
                                                  uint16_t* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i + 8 <= n) {
    float u[8], v[8];
    unpack8<E>(*reinterpret_cast<const u32x4*>(a + i), u);
    unpack8<E>(*reinterpret_cast<const u32x4*>(b + i), v);
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = u[k] * sigmoid(u[k]) * v[k];
    *reinterpret_cast<u32x4*>(y + i) = pack8<E>(u);
  } else {
    for (int64_t j = i; j < n; ++j) {
      const float u = to_f32<E>(a[j]);
      y[j] = uint16_t(pack2<E>(u * sigmoid(u) * to_f32<E>(b[j]), 0.f) & 0xFFFFu);
    }
  }
}

// da = dy b s (1 + a (1 - s)), db = dy a s, s = sigmoid(a)
template <class E>
__global__ __launch_bounds__(256) void k_gate_bwd(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
                                                  const uint16_t* __restrict__ dy, uint16_t* __restrict__ da,
                                                  uint16_t* __restrict__ db, int64_t n) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 8;
  auto one = [](float u, float v, float g, float* gu, float* gv) {
    const float s = sigmoid(u);
    *gu = g * v * s * (1.f + u * (1.f - s));
    *gv = g * (u * s);
  };
  if (i + 8 <= n) {
    float u[8], v[8], g[8];
    unpack8<E>(*reinterpret_cast<const u32x4*>(a + i), u);
    unpack8<E>(*reinterpret_cast<const u32x4*>(b + i), v);
    unpack8<E>(*reinterpret_cast<const u32x4*>(dy + i), g);
#pragma unroll
    for (int k = 0; k < 8; ++k) one(u[k], v[k], g[k], &u[k], &v[k]);
    *reinterpret_cast<u32x4*>(da + i) = pack8<E>(u);
    *reinterpret_cast<u32x4*>(db + i) = pack8<E>(v);
  } else {
    for (int64_t j = i; j < n; ++j) {
      float gu, gv;
      one(to_f32<E>(a[j]), to_f32<E>(b[j]), to_f32<E>(dy[j]), &gu, &gv);
      da[j] = uint16_t(pack2<E>(gu, 0.f) & 0xFFFFu);
      db[j] = uint16_t(pack2<E>(gv, 0.f) & 0xFFFFu);
    }
  }
}

template <class F>
int by_type(int dtype, F f) {
  if (dtype == KD_BF16) f(BF16{});
  else f(F16{});
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

// A launch holds less than 2^32 threads: longer inputs go in several.  f(first, count)
template <class F>
void in_launches(int64_t n, int64_t most, F f) {
  for (int64_t i = 0; i < n; i += most) f(i, std::min(most, n - i));
}
constexpr int64_t LAUNCH_ROWS = int64_t(1) << 25;   // 64 threads a row
constexpr int64_t LAUNCH_WORDS = int64_t(1) << 31;  // a thread a word of eight

}  // namespace

int launch_rms_fwd(const void* x, void* y, float* rstd, int64_t rows, int D, int dtype, float eps, hipStream_t st) {
  return by_type(dtype, [&](auto e) {
    using E = decltype(e);
    const int words = D / 8;
    auto go = [&](auto k) {
      in_launches(rows, LAUNCH_ROWS, [&](int64_t r, int64_t n) {
        hipLaunchKernelGGL(k, dim3(unsigned((n + 3) / 4)), dim3(256), 0, st, static_cast<const u32x4*>(x) + r * words,
                           static_cast<u32x4*>(y) + r * words, rstd == nullptr ? rstd : rstd + r, n, words, eps);
      });
    };
    if (words <= 64) go(k_rms_fwd<E, 1>);
    else if (words <= 128) go(k_rms_fwd<E, 2>);
    else go(k_rms_fwd<E, 4>);
  });
}

int launch_rms_bwd(const void* x, const void* dy, const float* rstd, void* dx, int64_t rows, int D, int dtype,
                   hipStream_t st) {
  return by_type(dtype, [&](auto e) {
    using E = decltype(e);
    const int words = D / 8;
    auto go = [&](auto k) {
      in_launches(rows, LAUNCH_ROWS, [&](int64_t r, int64_t n) {
        hipLaunchKernelGGL(k, dim3(unsigned((n + 3) / 4)), dim3(256), 0, st, static_cast<const u32x4*>(x) + r * words,
                           static_cast<const u32x4*>(dy) + r * words, rstd + r, static_cast<u32x4*>(dx) + r * words, n,
                           words);
      });
    };
    if (words <= 64) go(k_rms_bwd<E, 1>);
    else if (words <= 128) go(k_rms_bwd<E, 2>);
    else go(k_rms_bwd<E, 4>);
  });
}

int launch_gate_fwd(const void* a, const void* b, void* y, int64_t n, int dtype, hipStream_t st) {
  return by_type(dtype, [&](auto e) {
    in_launches(n, 8 * LAUNCH_WORDS, [&](int64_t i, int64_t m) {
      hipLaunchKernelGGL(k_gate_fwd<decltype(e)>, dim3(unsigned((m + 2047) / 2048)), dim3(256), 0, st,
                         static_cast<const uint16_t*>(a) + i, static_cast<const uint16_t*>(b) + i,
                         static_cast<uint16_t*>(y) + i, m);
    });
  });
}

int launch_gate_bwd(const void* a, const void* b, const void* dy, void* da, void* db, int64_t n, int dtype,
                    hipStream_t st) {
  return by_type(dtype, [&](auto e) {
    in_launches(n, 8 * LAUNCH_WORDS, [&](int64_t i, int64_t m) {
      hipLaunchKernelGGL(k_gate_bwd<decltype(e)>, dim3(unsigned((m + 2047) / 2048)), dim3(256), 0, st,
                         static_cast<const uint16_t*>(a) + i, static_cast<const uint16_t*>(b) + i,
                         static_cast<const uint16_t*>(dy) + i, static_cast<uint16_t*>(da) + i,
                         static_cast<uint16_t*>(db) + i, m);
    });
  });
}

}  // namespace kd
