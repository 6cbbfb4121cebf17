// Cocktail-party head on gfx950: first-[MASK] context vector, span-interior
// means and their scores (model.py:263-298), forward and backward.
//
// The reference builds h_spans with a Python double loop over rows and over
// the zipped [SPAN] / [ES] position lists, taking x_embed[i, st+1:ed].mean(0)
// when st + 1 < ed (model.py:287-293), and scores each span by its dot
// product with the hidden state at the row's first [MASK] (:264-270, :296).
// Here, where one_launch says so, one workgroup per (row, span)
// finds its own span's markers (block scans give the j-th [SPAN] and the j-th
// [ES] of the row), sums the interior in fp32 (eight waves over interleaved
// rows, combined in a fixed order) and dots the mean with the context vector:
// one launch of 10.7 us at B8 T2048 D768 with 8 spans, where the same in three
// (k_span_find, k_span_pool, k_span_score) takes 20 us.  The backward spreads
// d score over the interior rows and the [MASK] row in a fixed order, so the
// results are deterministic.
#include "kd_internal.h"

namespace kd {

namespace {

constexpr int TOK_MASK = 2, TOK_SPAN = 3, TOK_ES = 4;  // data_builder.py:44-52

KD_DEV int64_t token_at(const kd_span_args& a, int b, int t) {
  const int64_t off = int64_t(b) * a.tokens_strides[0] + int64_t(t) * a.tokens_strides[1];
  return a.tokens_dtype == KD_I64 ? static_cast<const int64_t*>(a.tokens)[off]
                                  : int64_t(static_cast<const int32_t*>(a.tokens)[off]);
}

template <class E>
KD_DEV float h_at(const kd_span_args& a, int b, int t, int d) {
  const uint16_t* p = static_cast<const uint16_t*>(a.h) + int64_t(b) * a.h_strides[0] + int64_t(t) * a.h_strides[1] + d;
  return to_f32<E>(*p);
}

// One workgroup (1024 threads) per row: positions of the j-th [SPAN] and the
// j-th [ES], then the interiors [lo, hi) of the zipped pairs and the first [MASK].
__global__ __launch_bounds__(1024) void k_span_find(kd_span_args a) {
  extern __shared__ int s_pos[];  // [0, n): j-th [SPAN] position, [n, 2n): j-th [ES] position
  __shared__ int s_warp[16];
  __shared__ int s_mask;
  const int b = blockIdx.x, n = a.n_spans, T = a.T;
  for (int j = threadIdx.x; j < 2 * n; j += blockDim.x) s_pos[j] = -1;
  if (threadIdx.x == 0) s_mask = T;
  __syncthreads();
  // contiguous chunk of positions per thread, so ordinals follow position order
  const int per = (T + blockDim.x - 1) / blockDim.x;
  const int t0 = threadIdx.x * per, t1 = min(T, t0 + per);
  int ns = 0, ne = 0, first_mask = T;
  for (int t = t0; t < t1; ++t) {
    const int64_t tok = token_at(a, b, t);
    ns += tok == TOK_SPAN;
    ne += tok == TOK_ES;
    if (tok == TOK_MASK && first_mask == T) first_mask = t;
  }
  const int js = block_scan(ns, s_warp) - ns;  // exclusive: ordinal of this chunk's first [SPAN]
  const int je = block_scan(ne, s_warp) - ne;
  if (first_mask < T) atomicMin(&s_mask, first_mask);
  int cs = js, ce = je;
  for (int t = t0; t < t1; ++t) {
    const int64_t tok = token_at(a, b, t);
    if (tok == TOK_SPAN) {
      if (cs < n) s_pos[cs] = t;  // spans past n_spans are dropped
      ++cs;
    } else if (tok == TOK_ES) {
      if (ce < n) s_pos[n + ce] = t;
      ++ce;
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const int st = s_pos[j], ed = s_pos[n + j];
    const bool ok = st >= 0 && ed >= 0 && st + 1 < ed;  // zip pairs only; `if st + 1 < ed` (model.py:292)
    a.span_lo[int64_t(b) * n + j] = ok ? st + 1 : 0;
    a.span_hi[int64_t(b) * n + j] = ok ? ed : 0;
  }
  if (threadIdx.x == 0) a.mask_pos[b] = s_mask < T ? s_mask : -1;
}

// grid (ceil(B / 4)): [SPAN] tokens of each row, one wave a row
__global__ __launch_bounds__(256) void k_span_count(kd_span_args a, int32_t* counts) {
  const int lane = threadIdx.x & 63, b = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= a.B) return;
  int n = 0;
#pragma unroll 8
  for (int t = lane; t < a.T; t += 64) n += token_at(a, b, t) == TOK_SPAN;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  if (lane == 0) counts[b] = n;
}

// Fixed-order block sum (256 threads) of one float per thread.
KD_DEV float block_sum256(float v, float* s_red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) s_red[wave] = v;
  __syncthreads();
  const float r = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
  __syncthreads();
  return r;
}

// grid (n_spans + 1, B, ceil(D / 256)): block (j < n, b, c) averages span j's
// interior over the columns [256 c, 256 c + 256); block (n, b, c) copies
// those columns of h_ctx.  Wave w of 8 sums the rows lo + w, lo + w + 8, ...
// (lane l: columns 256 c + l + 64 k, k < 4) and the eight partials combine in
// a fixed order, ((w0 + w1) + (w2 + w3)) + ((w4 + w5) + (w6 + w7)).
template <class E>
__global__ __launch_bounds__(512) void k_span_pool(kd_span_args a) {
  __shared__ float s_part[8][256];
  const int j = blockIdx.x, b = blockIdx.y, n = a.n_spans, D = a.D, d0 = blockIdx.z * 256;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (j == n) {
    const int mp = a.mask_pos[b];
    const int d = d0 + int(threadIdx.x);
    if (threadIdx.x < 256 && d < D) a.h_ctx[int64_t(b) * D + d] = mp >= 0 ? h_at<E>(a, b, mp, d) : 0.f;
    return;
  }
  const int lo = a.span_lo[int64_t(b) * n + j], hi = a.span_hi[int64_t(b) * n + j];
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int t = lo + wave; t < hi; t += 8) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int d = d0 + lane + 64 * k;
      if (d < D) acc[k] += h_at<E>(a, b, t, d);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) s_part[wave][lane + 64 * k] = acc[k];
  __syncthreads();
  const int d = d0 + int(threadIdx.x);
  if (threadIdx.x < 256 && d < D) {
    const int i = threadIdx.x;
    const float sum = ((s_part[0][i] + s_part[1][i]) + (s_part[2][i] + s_part[3][i])) +
                      ((s_part[4][i] + s_part[5][i]) + (s_part[6][i] + s_part[7][i]));
    a.h_spans[(int64_t(b) * n + j) * D + d] = hi > lo ? sum / float(hi - lo) : 0.f;
  }
}

// grid (n_spans, B): score of span j = sum_d h_span_j[d] h_ctx[d], thread i
// over d = i + 256 k in ascending k, then a fixed-order block sum.
__global__ __launch_bounds__(256) void k_span_score(kd_span_args a) {
  __shared__ float s_red[4];
  const int j = blockIdx.x, b = blockIdx.y, n = a.n_spans, D = a.D;
  const float* hs = a.h_spans + (int64_t(b) * n + j) * D;
  const float* hc = a.h_ctx + int64_t(b) * D;
  float part = 0.f;
  for (int d = threadIdx.x; d < D; d += 256) part = __builtin_fmaf(hs[d], hc[d], part);
  const float s = block_sum256(part, s_red);
  if (threadIdx.x == 0) a.scores[int64_t(b) * n + j] = s;
}

// k_span_find, k_span_pool and k_span_score in one launch (where: one_launch),
// grid (n_spans + 1, B), 512 threads.  Block (j, b) scans row b itself (thread i
// a contiguous run of tokens, two block scans for the ordinals), keeps the
// positions of the j-th [SPAN] and [ES] and the first [MASK], then sums its
// interior 256 columns at a time (wave w the rows lo + w, lo + w + 8, ..., lane l
// the columns 4 l .. 4 l + 3) and its score.  The sums run in the order of the
// three kernels.  Block (n, b) writes h_ctx.
template <class E, bool VEC>
__global__ __launch_bounds__(512) void k_span_all(kd_span_args a) {
  __shared__ float s_part[8][256];
  __shared__ float s_red[4];
  __shared__ int s_warp[16];
  __shared__ int s_st, s_ed, s_mask;
  const int j = blockIdx.x, b = blockIdx.y, n = a.n_spans, D = a.D, T = a.T, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_st = s_ed = -1, s_mask = T;
  const int per = (T + 511) / 512, t0 = tid * per, t1 = min(T, t0 + per);
  int ns = 0, ne = 0, first_mask = T;
  for (int t = t0; t < t1; ++t) {
    const int64_t tok = token_at(a, b, t);
    ns += tok == TOK_SPAN;
    ne += tok == TOK_ES;
    if (tok == TOK_MASK && first_mask == T) first_mask = t;
  }
  const int js = block_scan(ns, s_warp) - ns, je = block_scan(ne, s_warp) - ne;  // (their barriers order s_st's start)
  if (first_mask < T) atomicMin(&s_mask, first_mask);
  if ((js <= j && j < js + ns) || (je <= j && j < je + ne)) {  // this run holds one of span j's markers
    int cs = js, ce = je;
    for (int t = t0; t < t1; ++t) {
      const int64_t tok = token_at(a, b, t);
      if (tok == TOK_SPAN && cs++ == j) s_st = t;
      if (tok == TOK_ES && ce++ == j) s_ed = t;
    }
  }
  __syncthreads();
  const int mp = s_mask < T ? s_mask : -1;
  if (j == n) {
    if (tid == 0) a.mask_pos[b] = mp;
    for (int d = tid; d < D; d += 512) a.h_ctx[int64_t(b) * D + d] = mp >= 0 ? h_at<E>(a, b, mp, d) : 0.f;
    return;
  }
  const bool ok = s_st >= 0 && s_ed >= 0 && s_st + 1 < s_ed;  // (model.py:292)
  const int lo = ok ? s_st + 1 : 0, hi = ok ? s_ed : 0;
  if (tid == 0) a.span_lo[int64_t(b) * n + j] = lo, a.span_hi[int64_t(b) * n + j] = hi;
  float part = 0.f;
  for (int d0 = 0; d0 < D; d0 += 256) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const int dl = d0 + 4 * lane;
    if (VEC) {
      if (dl < D) {  // (VEC: D is a multiple of 4)
        const uint16_t* p = static_cast<const uint16_t*>(a.h) + int64_t(b) * a.h_strides[0] + dl;
#pragma unroll 4
        for (int t = lo + wave; t < hi; t += 8) {
          const u32x2 v = *reinterpret_cast<const u32x2*>(p + int64_t(t) * a.h_strides[1]);
          acc[0] += to_f32<E>(uint16_t(v[0] & 0xFFFFu));
          acc[1] += to_f32<E>(uint16_t(v[0] >> 16));
          acc[2] += to_f32<E>(uint16_t(v[1] & 0xFFFFu));
          acc[3] += to_f32<E>(uint16_t(v[1] >> 16));
        }
      }
    } else {
      for (int t = lo + wave; t < hi; t += 8)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (dl + k < D) acc[k] += h_at<E>(a, b, t, dl + k);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) s_part[wave][4 * lane + k] = acc[k];
    __syncthreads();
    const int d = d0 + tid;
    if (tid < 256 && d < D) {
      const float sum = ((s_part[0][tid] + s_part[1][tid]) + (s_part[2][tid] + s_part[3][tid])) +
                        ((s_part[4][tid] + s_part[5][tid]) + (s_part[6][tid] + s_part[7][tid]));
      const float mean = hi > lo ? sum / float(hi - lo) : 0.f;
      a.h_spans[(int64_t(b) * n + j) * D + d] = mean;
      part = __builtin_fmaf(mean, mp >= 0 ? h_at<E>(a, b, mp, d) : 0.f, part);
    }
    __syncthreads();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if (lane == 0 && wave < 4) s_red[wave] = part;
  __syncthreads();
  if (tid == 0) a.scores[int64_t(b) * n + j] = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
}

// grid (ceil(T / (4 BWD_R)), B), one wave per BWD_R rows t of dh, each written in full:
//   dh[t] = sum_{j: lo_j <= t < hi_j} ds_j h_ctx / (hi_j - lo_j)   (ascending j)
//         + [t == mask] sum_j ds_j h_span_j                          (ascending j)
// Columns go in groups of 512.  The spans containing t are found 64 at a time
// by a wave ballot over j and added in ascending j; a row in no span (most
// rows) is written as zeros.  Bound by dh's way to memory, and by the chain of
// loads before a row's first store, which several rows a wave share.  With VEC a
// lane holds the eight consecutive columns d0 + 8 l (16-byte accesses), where D,
// dh's strides and every base allow it; without, columns d0 + l + 64 k.  25 MB of
// dh at B8 T2048 D768: 32 us with one row a wave and 2-byte stores, 23.6 with
// 16-byte stores, 14.6 with four rows a wave and the [MASK] row's loads overlapped.
template <class E, bool VEC, int BWD_R>
__global__ __launch_bounds__(256) void k_span_bwd(kd_span_args a) {
  const int lane = threadIdx.x & 63;
  const int b = blockIdx.y, n = a.n_spans, D = a.D;
  const int mp = a.mask_pos[b];
  const int32_t* lo = a.span_lo + int64_t(b) * n;
  const int32_t* hi = a.span_hi + int64_t(b) * n;
  const float* ds = a.dscores + int64_t(b) * n;
  const int first = (blockIdx.x * 4 + (threadIdx.x >> 6)) * BWD_R, last = min(a.T, first + BWD_R);
  for (int d0 = 0; d0 < D; d0 += 512) {
    auto col = [&](int k) { return VEC ? d0 + 8 * lane + k : d0 + lane + 64 * k; };
    auto load8 = [&](const float* p, float (&x)[8]) {  // this lane's columns of a row p of D floats, 0 past D
      if (VEC) {
        const bool in = col(0) < D;  // (VEC: D is a multiple of 8)
        const f32x4 u = in ? *reinterpret_cast<const f32x4*>(p + col(0)) : f32x4{};
        const f32x4 v = in ? *reinterpret_cast<const f32x4*>(p + col(4)) : f32x4{};
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = u[k], x[4 + k] = v[k];
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = col(k) < D ? p[col(k)] : 0.f;
      }
    };
    float c[8];
    load8(a.h_ctx + int64_t(b) * D, c);
    for (int t = first; t < last; ++t) {
      float g[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) g[k] = 0.f;
      for (int j0 = 0; j0 < n; j0 += 64) {
        const int jl = j0 + lane;
        const bool in = jl < n && lo[jl] <= t && t < hi[jl];
        for (uint64_t m = __builtin_amdgcn_ballot_w64(in); m; m &= m - 1) {
          const int j = j0 + __builtin_ctzll(m);
          const float dsj = ds[j], len = float(hi[j] - lo[j]);
#pragma unroll
          for (int k = 0; k < 8; ++k) g[k] += dsj * c[k] / len;
        }
      }
      if (t == mp)
#pragma unroll 4
        for (int j = 0; j < n; ++j) {
          float hs[8];
          load8(a.h_spans + (int64_t(b) * n + j) * D, hs);
          const float dsj = ds[j];
#pragma unroll
          for (int k = 0; k < 8; ++k) g[k] = __builtin_fmaf(dsj, hs[k], g[k]);
        }
      uint16_t* out = static_cast<uint16_t*>(a.dh) + int64_t(b) * a.dh_strides[0] + int64_t(t) * a.dh_strides[1];
      if (VEC) {
        if (col(0) < D)
          *reinterpret_cast<u32x4*>(out + col(0)) =
              u32x4{pack2<E>(g[0], g[1]), pack2<E>(g[2], g[3]), pack2<E>(g[4], g[5]), pack2<E>(g[6], g[7])};
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (col(k) < D) out[col(k)] = uint16_t(pack2<E>(g[k], 0.f) & 0xFFFFu);
      }
    }
  }
}

bool multiple(const void* p, const int64_t* strides, int D, int of) {  // a base of 2 of bytes, rows and D of `of` elements
  return reinterpret_cast<uintptr_t>(p) % (2 * of) == 0 && strides[0] % of == 0 && strides[1] % of == 0 && D % of == 0;
}

// Where one launch is the faster one.  Each of its (n + 1) B workgroups scans its
// row's T tokens and walks the columns 256 at a time, where k_span_find scans a
// row once and k_span_pool has a workgroup for every 256 columns; without 8-byte
// loads (vec) its columns take up to six times as long.  So the scans have to be
// few (2^21 tokens) or small beside the columns that a row is pooled over, and the
// columns one group without vec, four with it, eight where the workgroups fill a
// quarter of the chip.  us, one launch / three: B8 T2048 D768 n8 8.9 / 15.4; B1 T2048
// n1 L1945 D768 47 / 112, D2048 209 / 109, D770 290 / 108; B64 T16384 n60 D64 274 / 70;
// B64 T4096 n4 D2048 124 / 366.  Over 1902 timed shapes none is slower than three
// launches by 2%.
bool one_launch(const kd_span_args& a, bool vec) {
  const int64_t n = a.n_spans, blocks = (n + 1) * a.B;
  const bool small_scan = 16 * (n + 1) <= a.D;
  if (a.T > 16384 || n * a.T > (1 << 20)) return false;
  if (a.D <= (vec ? 1024 : 256)) return blocks * a.T <= (1 << 21) || small_scan;
  return vec && a.D <= 2048 && blocks >= 64 && small_scan;
}

template <class E>
void launch_span_e(const kd_span_args& a, hipStream_t st) {
  const bool vec = multiple(a.h, a.h_strides, a.D, 4);
  if (one_launch(a, vec)) {
    const dim3 grid(unsigned(a.n_spans + 1), unsigned(a.B));
    if (vec) hipLaunchKernelGGL((k_span_all<E, true>), grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((k_span_all<E, false>), grid, dim3(512), 0, st, a);
    return;
  }
  hipLaunchKernelGGL(k_span_find, dim3(unsigned(a.B)), dim3(1024), size_t(2) * a.n_spans * sizeof(int), st, a);
  const dim3 pool(unsigned(a.n_spans + 1), unsigned(a.B), unsigned((a.D + 255) / 256));
  hipLaunchKernelGGL(k_span_pool<E>, pool, dim3(512), 0, st, a);
  hipLaunchKernelGGL(k_span_score, dim3(unsigned(a.n_spans), unsigned(a.B)), dim3(256), 0, st, a);
}

template <class E, int R>
void launch_span_bwd_r(const kd_span_args& a, hipStream_t st) {
  const dim3 grid(unsigned((a.T + 4 * R - 1) / (4 * R)), unsigned(a.B));
  auto aligned = [](const float* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (multiple(a.dh, a.dh_strides, a.D, 8) && aligned(a.h_ctx) && aligned(a.h_spans))
    hipLaunchKernelGGL((k_span_bwd<E, true, R>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_span_bwd<E, false, R>), grid, dim3(256), 0, st, a);
}

// Up to 8192 rows a wave takes one, so that there are waves for every CU: us, one
// row a wave / four: B1 T2048 D768 6.5 / 8.0, D2048 6.8 / 14.3, B4 T2048 D2048 11.3 / 18; B16 T1024 D1024 with 60
// spans 34 / 27, B64 T2048 D768 63 / 58.
template <class E>
void launch_span_bwd_e(const kd_span_args& a, hipStream_t st) {
  if (int64_t(a.B) * a.T <= 8192) launch_span_bwd_r<E, 1>(a, st);
  else launch_span_bwd_r<E, 4>(a, st);
}

}  // namespace

int launch_span_count(const kd_span_args& a, int32_t* counts, hipStream_t st) {
  hipLaunchKernelGGL(k_span_count, dim3(unsigned((a.B + 3) / 4)), dim3(256), 0, st, a, counts);
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

int launch_span(const kd_span_args& a, hipStream_t st) {
  if (a.dtype == KD_BF16) launch_span_e<BF16>(a, st);
  else launch_span_e<F16>(a, st);
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

int launch_span_bwd(const kd_span_args& a, hipStream_t st) {
  if (a.dtype == KD_BF16) launch_span_bwd_e<BF16>(a, st);
  else launch_span_bwd_e<F16>(a, st);
  return hipGetLastError() == hipSuccess ? KD_OK : KD_ERR_LAUNCH;
}

}  // namespace kd
