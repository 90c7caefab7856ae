// Causal depthwise conv1d (+ SiLU) over channel-major rows, forward and
// backward, for gfx950.
//
//   pre[b,c,t] = bias[c] + sum_{j<K} w[c,j] * x[b,c,t-(K-1)+j]   (x = 0 for t < 0)
//   out        = silu(pre) (or pre)
//
// This is the prefill convolution of the Mamba layer (nn.Conv1d with
// groups = channels, padding K-1, first L outputs kept, then SiLU;
// modules/mamba.py:37-44,138-139 of the reference), computed in the
// (batch, channels, seqlen) layout the scan reads, with the activation fused.
//
// Memory-bound: one workgroup streams one (b, c) row; each thread owns chunks
// of 8 consecutive positions (one 16-byte load for bf16, two for fp32) plus
// the K-1 elements before it, which the cache serves.  The backward recomputes
// pre over the K-1 positions past its chunk, writes dx, and leaves per-row
// partial sums of dw / dbias that a second kernel adds over the batch in a
// fixed order (deterministic, no atomics).  All loads of a chunk go through
// buffer ranges that end at the row, so none waits behind a bounds check, and
// issue before the taps are waited for: one memory round trip a chunk.  Rows
// that are not whole 16-byte pieces take the same chunks (ConvRow, store_chunk);
// position by position, with K loads forward and K (K + 1) backward each, a
// pass over (4, 2048, 2047) in bf16 with 4 taps took 61.5 us forward and 151.5
// backward, now 18.3 and 31.0 (2048 positions: 15.8 and 27.1, 4.2 and 3.7 TB/s;
// with the loads behind branches 18.3 and 30.4).
#include "ss_common.cuh"
#include "ss_io.cuh"
#include "ss_prof.h"

namespace ssm {

namespace {

constexpr int kConvThreads = 256;
constexpr int kConvChunk = 8;
constexpr int kMaxWidth = 8;

template <typename T>
__device__ __forceinline__ void store8(T* __restrict__ p, const float* v);

template <>
__device__ __forceinline__ void store8<float>(float* __restrict__ p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}

template <>
__device__ __forceinline__ void store8<__hip_bfloat16>(__hip_bfloat16* __restrict__ p, const float* v) {
  uint4 x;
  x.x = pack_bf16x2(v[0], v[1]);
  x.y = pack_bf16x2(v[2], v[3]);
  x.z = pack_bf16x2(v[4], v[5]);
  x.w = pack_bf16x2(v[6], v[7]);
  *reinterpret_cast<uint4*>(p) = x;
}

// The elements a workgroup reads of a row for the positions [i0, i0 + kConvSpan):
// from 8 before to 8 after, as one buffer range that ends with the row.  kVec:
// rows of a multiple of 8 elements at 16-byte aligned addresses.  Otherwise any
// element alignment (RowRange): fp32 at dword alignment, bf16 as the dwords that
// hold the elements, shifted into place.
constexpr int kConvSpan = kConvThreads * kConvChunk;

template <typename T, bool kVec>
struct ConvRow {
  static constexpr bool kShift = !kVec && sizeof(T) == 2;
  // dwords that hold N elements (an array of one where there are none)
  template <int N> static constexpr int words() { return N ? N * (int)sizeof(T) / 4 + (kShift ? 1 : 0) : 1; }
  __amdgpu_buffer_rsrc_t r;
  uint32_t extra = 0;  // bytes from the (dword aligned) base to the first element: 0 or 2
  int s, L;

  __device__ __forceinline__ ConvRow(const T* row, int L_, int i0) : s(max(i0 - kConvChunk, 0)), L(L_) {
    const uint64_t a = reinterpret_cast<uint64_t>(row + s);
    const uint32_t bytes = (uint32_t)min(L - s, kConvSpan + 2 * kConvChunk) * (uint32_t)sizeof(T);
    if constexpr (kShift) extra = __builtin_amdgcn_readfirstlane((uint32_t)a & 2u);
    r = raw_rsrc(reinterpret_cast<void*>(kShift ? a & ~(uint64_t)3 : a),
                 kShift ? (extra + bytes + 3u) & ~3u : bytes);
  }
  // N elements (4, 8, or none) from position t, a multiple of 4; zero outside
  // the row, but past its end the next row's where it does not end with the range
  template <int N> __device__ __forceinline__ void load(uint32_t* w, int t) const {
    const int off = t >= 0 ? (t - s) * (int)sizeof(T) : (int)kOffDrop;
    constexpr int W = words<N>();
    if constexpr (N > 0) {
#pragma unroll
      for (int q = 0; q + 4 <= W; q += 4) {
        const u32x4_v v = __builtin_amdgcn_raw_buffer_load_b128(r, off + 4 * q, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[q + i] = v[i];
      }
      if constexpr (W % 4 == 1) {
        w[W - 1] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * (W - 1), 0, 0);
      } else if constexpr (W % 4 == 2) {
        const u32x2_v v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        w[0] = v.x; w[1] = v.y;
      } else if constexpr (W % 4 == 3) {
        typedef unsigned int u32x3_v __attribute__((ext_vector_type(3)));
        const u32x3_v v = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
        w[0] = v.x; w[1] = v.y; w[2] = v.z;
      }
    }
  }
  // their values; kEnd: zero at and past the row's end
  template <int N, bool kEnd> __device__ __forceinline__ void decode(const uint32_t* w, int t, float* v) const {
    if constexpr (N > 0) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if constexpr (sizeof(T) == 4) {
          v[i] = __uint_as_float(w[i]);
        } else {
          uint32_t p;
          if constexpr (kShift) p = __builtin_amdgcn_alignbyte(w[i / 2 + 1], w[i / 2], extra);
          else p = w[i / 2];
          v[i] = i % 2 ? bf16_hi(p) : bf16_lo(p);
        }
        if constexpr (kEnd && !kVec) v[i] = t + i < L ? v[i] : 0.0f;
      }
    }
  }
};

// Elements read on either side of a chunk.
template <int K> constexpr int conv_halo() { return K == 1 ? 0 : K <= 5 ? 4 : 8; }

// The chunk at t0 of a row into its output (positions below L).  Every thread
// of the workgroup calls it.  kVec as above.  Otherwise 16 bytes a lane at dword
// alignment too: in a bf16 row that starts between dwords each lane writes the
// last element of the lane before and its own first seven; first and last lanes
// and the row's end write element by element.
template <typename T, bool kVec>
__device__ __forceinline__ void store_chunk(T* __restrict__ row, int L, int i0, const float (&v)[kConvChunk]) {
  const int t0 = i0 + threadIdx.x * kConvChunk;
  if constexpr (kVec) {
    if (t0 < L) store8<T>(row + t0, v);
  } else {
    const uint64_t a = reinterpret_cast<uint64_t>(row + i0);
    const uint32_t extra = __builtin_amdgcn_readfirstlane((uint32_t)a & 2u);
    const uint32_t n = (uint32_t)min(L - i0, kConvSpan);
    const __amdgpu_buffer_rsrc_t r =
        raw_rsrc(reinterpret_cast<void*>(a & ~(uint64_t)3), extra + n * (uint32_t)sizeof(T));
    const int off = (int)extra + (t0 - i0) * (int)sizeof(T);
    auto at = [&](bool ok, int o) { return ok ? o : (int)kOffDrop; };
    if constexpr (sizeof(T) == 4) {
      const bool whole = t0 + kConvChunk <= L;
#pragma unroll
      for (int q = 0; q < kConvChunk; q += 4) {
        const u32x4_v d = {__float_as_uint(v[q]), __float_as_uint(v[q + 1]), __float_as_uint(v[q + 2]),
                           __float_as_uint(v[q + 3])};
        __builtin_amdgcn_raw_buffer_store_b128(d, r, at(whole, off + 4 * q), 0, 0);
      }
      if (!whole && t0 < L) {
#pragma unroll
        for (int j = 0; j < kConvChunk; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[j]), r, at(t0 + j < L, off + 4 * j), 0, 0);
      }
    } else {
      const int lane = threadIdx.x & 63;
      const u32x4_v p = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                         pack_bf16x2(v[6], v[7])};
      auto one = [&](int j, bool ok) {
        const uint32_t w = p[j / 2];
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(j & 1 ? w >> 16 : w), r,
                                              at(ok && t0 + j < L, off + 2 * j), 0, 0);
      };
      bool whole;
      if (extra) {
        const uint32_t before = __shfl_up(p[3], 1, 64);
        const u32x4_v d = {__builtin_amdgcn_alignbyte(p[0], before, 2),
                           __builtin_amdgcn_alignbyte(p[1], p[0], 2),
                           __builtin_amdgcn_alignbyte(p[2], p[1], 2),
                           __builtin_amdgcn_alignbyte(p[3], p[2], 2)};
        whole = lane > 0 && t0 + kConvChunk - 1 <= L;
        __builtin_amdgcn_raw_buffer_store_b128(d, r, at(whole, off - 2), 0, 0);
        one(7, !(lane < 63 && t0 + 2 * kConvChunk - 1 <= L));
      } else {
        whole = t0 + kConvChunk <= L;
        __builtin_amdgcn_raw_buffer_store_b128(p, r, at(whole, off), 0, 0);
        one(7, !whole);
      }
      if (!whole && t0 < L) {
#pragma unroll
        for (int j = 0; j < kConvChunk - 1; ++j) one(j, true);
      }
    }
  }
}

template <int K, typename T>
__device__ __forceinline__ void load_taps(const T* __restrict__ w, const T* __restrict__ bias, int c,
                                          float (&wk)[K], float& bs) {
#pragma unroll
  for (int j = 0; j < K; ++j) wk[j] = Elem<T>::load1(w + (size_t)c * K + j);
  // an absent bias reads a valid stand-in and is dropped: a load in a branch
  // would be waited for there
  bs = Elem<T>::load1(bias ? bias + c : w);
  if (!bias) bs = 0.0f;
}

// Sum of K+1 per-thread values over the workgroup; thread 0 gets the totals.
template <int K>
__device__ __forceinline__ void block_sum(float (&v)[K + 1], float* red) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j <= K; ++j) {
    float s = v[j];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) red[wave * (K + 1) + j] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j <= K; ++j) {
      float s = 0.0f;
      for (int q = 0; q < kConvThreads / 64; ++q) s += red[q * (K + 1) + j];
      v[j] = s;
    }
  }
}

// window (nullable): the decode cache of the row, the K-1 inputs ending at
// position len-1 (len = lengths[b] clamped to [0, L], or L), zero where the
// window starts before the row (the conv context the reference keeps after a
// prefill, modules/mamba.py:113-135).  x's batch rows are xbs elements apart
// (a channel slice of a larger activation); out is contiguous.
template <typename T, int K, bool kVec>
__global__ __launch_bounds__(kConvThreads) void causal_conv1d_fwd_kernel(
    const T* __restrict__ x, int64_t xbs, const T* __restrict__ w, const T* __restrict__ bias,
    T* __restrict__ out, int dim, int L, int silu, const int64_t* __restrict__ lengths,
    T* __restrict__ window) {
  const size_t row = blockIdx.x;
  const int c = (int)(row % (size_t)dim);
  const T* __restrict__ xr = x + (row / (size_t)dim) * (size_t)xbs + (size_t)c * L;
  T* __restrict__ orow = out + row * (size_t)L;
  float wk[K], bs;
  // the decode cache's row length, fetched now and used after the main loop
  const int64_t len_in = lengths ? lengths[row / (size_t)dim] : (int64_t)L;
  constexpr int H = conv_halo<K>();
  using R = ConvRow<T, kVec>;
  uint32_t w0[R::template words<kConvChunk>()], wp[R::template words<H>()];
  for (int i0 = 0; i0 < L; i0 += kConvSpan) {
    const R in(xr, L, i0);
    const int t0 = i0 + threadIdx.x * kConvChunk;
    in.template load<kConvChunk>(w0, t0);
    in.template load<H>(wp, t0 - H);
    if (i0 == 0) load_taps<K>(w, bias, c, wk, bs);
    float v[H + kConvChunk], o[kConvChunk];
    in.template decode<H, false>(wp, t0 - H, v);
    in.template decode<kConvChunk, false>(w0, t0, v + H);
#pragma unroll
    for (int i = 0; i < kConvChunk; ++i) {
      float acc = bs;
#pragma unroll
      for (int j = 0; j < K; ++j) acc = fmaf(wk[j], v[H + i - (K - 1) + j], acc);
      o[i] = silu ? silu_f(acc) : acc;
    }
    store_chunk<T, kVec>(orow, L, i0, o);
  }
  // the decode cache last, off the main stream's path
  if (K > 1 && window && threadIdx.x < K - 1) {
    const int len = (int)min<int64_t>(max<int64_t>(len_in, 0), L);
    const int idx = len - (K - 1) + (int)threadIdx.x;
    const float v = Elem<T>::load1(xr + max(idx, 0));
    Elem<T>::store1(window + row * (K - 1) + threadIdx.x, idx >= 0 ? v : 0.0f);
  }
}

// dx and per-row partials part[row*(K+1) + j] = sum_t g_t x_{t-(K-1)+j} (j < K)
// and part[row*(K+1) + K] = sum_t g_t, with g = dout * dact(pre).
template <typename T, int K, bool kVec>
__global__ __launch_bounds__(kConvThreads) void causal_conv1d_bwd_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ bias,
    const T* __restrict__ dout, T* __restrict__ dx, float* __restrict__ part, int dim, int L,
    int silu) {
  __shared__ float red[(kConvThreads / 64) * (kMaxWidth + 1)];
  const size_t row = blockIdx.x;
  const int c = (int)(row % (size_t)dim);
  const T* __restrict__ xr = x + row * (size_t)L;
  const T* __restrict__ gr = dout + row * (size_t)L;
  T* __restrict__ dxr = dx + row * (size_t)L;
  float wk[K], bs;
  float acc[K + 1];
#pragma unroll
  for (int j = 0; j <= K; ++j) acc[j] = 0.0f;

  auto act_grad = [&](float pre) { return silu ? silu_grad_f(pre) : 1.0f; };

  constexpr int E = kConvChunk, H = conv_halo<K>();
  using R = ConvRow<T, kVec>;
  uint32_t x0[R::template words<E>()], d0[R::template words<E>()];
  uint32_t xp[R::template words<H>()], xn[R::template words<H>()], dn[R::template words<H>()];
  for (int i0 = 0; i0 < L; i0 += kConvSpan) {
    const R xin(xr, L, i0), din(gr, L, i0);
    const int t0 = i0 + threadIdx.x * E;
    // x over [t0-H, t0+E+H), dout over [t0, t0+E+H)
    xin.template load<E>(x0, t0);
    din.template load<E>(d0, t0);
    xin.template load<H>(xp, t0 < L ? t0 - H : -1);  // (lanes past the row: all zero)
    xin.template load<H>(xn, t0 + E);
    din.template load<H>(dn, t0 + E);
    if (i0 == 0) load_taps<K>(w, bias, c, wk, bs);
    float xv[E + 2 * H], dv[E + H];
    xin.template decode<H, false>(xp, t0 - H, xv);
    xin.template decode<E, true>(x0, t0, xv + H);
    xin.template decode<H, true>(xn, t0 + E, xv + H + E);
    din.template decode<E, true>(d0, t0, dv);
    din.template decode<H, true>(dn, t0 + E, dv + E);
    // g at positions t0 + m, m < E + K - 1 (zero past the row end: dv = 0 there)
    float g[E + K - 1];
#pragma unroll
    for (int m = 0; m < E + K - 1; ++m) {
      float pre = bs;
#pragma unroll
      for (int j = 0; j < K; ++j) pre = fmaf(wk[j], xv[H + m - (K - 1) + j], pre);
      g[m] = dv[m] * act_grad(pre);
    }
    float o[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      float s = 0.0f;
#pragma unroll
      for (int j = 0; j < K; ++j) s = fmaf(wk[j], g[i + (K - 1) - j], s);
      o[i] = s;
#pragma unroll
      for (int j = 0; j < K; ++j) acc[j] = fmaf(g[i], xv[H + i - (K - 1) + j], acc[j]);
      acc[K] += g[i];
    }
    store_chunk<T, kVec>(dxr, L, i0, o);
  }
  block_sum<K>(acc, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j <= K; ++j) part[row * (K + 1) + j] = acc[j];
  }
}

// dw[c,j] = sum_b part[(b*dim + c)*(K+1) + j]; dbias[c] likewise at j = K.
template <typename T>
__global__ __launch_bounds__(256) void causal_conv1d_wgrad_kernel(const float* __restrict__ part,
                                                                  T* __restrict__ dw,
                                                                  T* __restrict__ dbias, int batch,
                                                                  int dim, int K) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // c*(K+1) + j
  if (i >= dim * (K + 1)) return;
  const int c = i / (K + 1);
  const int j = i - c * (K + 1);
  float s = 0.0f;
  for (int b = 0; b < batch; ++b) s += part[((size_t)b * dim + c) * (K + 1) + j];
  if (j < K) {
    Elem<T>::store1(dw + (size_t)c * K + j, s);
  } else if (dbias) {
    Elem<T>::store1(dbias + c, s);
  }
}

template <typename T, int K>
hipError_t launch_fwd_k(int batch, int dim, int L, const void* x, int64_t xbs, const void* w,
                        const void* bias, int silu, void* out, const int64_t* lengths, void* window,
                        bool vec, hipStream_t st) {
  ProfScope prof("causal_conv1d_fwd", st);
  const dim3 grid((unsigned)((size_t)batch * dim));
  auto* xp = static_cast<const T*>(x);
  auto* wp = static_cast<const T*>(w);
  auto* bp = static_cast<const T*>(bias);
  auto* op = static_cast<T*>(out);
  auto* wo = static_cast<T*>(window);
  if (vec)
    hipLaunchKernelGGL((causal_conv1d_fwd_kernel<T, K, true>), grid, dim3(kConvThreads), 0, st, xp,
                       xbs, wp, bp, op, dim, L, silu, lengths, wo);
  else
    hipLaunchKernelGGL((causal_conv1d_fwd_kernel<T, K, false>), grid, dim3(kConvThreads), 0, st, xp,
                       xbs, wp, bp, op, dim, L, silu, lengths, wo);
  return hipGetLastError();
}

template <typename T, int K>
hipError_t launch_bwd_k(int batch, int dim, int L, const void* x, const void* w, const void* bias,
                        const void* dout, int silu, void* dx, void* dw, void* dbias, float* part,
                        bool vec, hipStream_t st) {
  const dim3 grid((unsigned)((size_t)batch * dim));
  auto* xp = static_cast<const T*>(x);
  auto* wp = static_cast<const T*>(w);
  auto* bp = static_cast<const T*>(bias);
  auto* gp = static_cast<const T*>(dout);
  auto* dxp = static_cast<T*>(dx);
  {
    ProfScope prof("causal_conv1d_bwd", st);
    if (vec)
      hipLaunchKernelGGL((causal_conv1d_bwd_kernel<T, K, true>), grid, dim3(kConvThreads), 0, st,
                         xp, wp, bp, gp, dxp, part, dim, L, silu);
    else
      hipLaunchKernelGGL((causal_conv1d_bwd_kernel<T, K, false>), grid, dim3(kConvThreads), 0, st,
                         xp, wp, bp, gp, dxp, part, dim, L, silu);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  ProfScope prof("causal_conv1d_wgrad", st);
  const int n = dim * (K + 1);
  hipLaunchKernelGGL((causal_conv1d_wgrad_kernel<T>), dim3((n + 255) / 256), dim3(256), 0, st,
                     part, static_cast<T*>(dw), static_cast<T*>(dbias), batch, dim, K);
  return hipGetLastError();
}

template <typename T>
hipError_t dispatch_fwd(int batch, int dim, int L, int K, const void* x, int64_t xbs, const void* w,
                        const void* bias, int silu, void* out, const int64_t* lengths,
                        void* window, bool vec, hipStream_t st) {
  switch (K) {
    case 1: return launch_fwd_k<T, 1>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 2: return launch_fwd_k<T, 2>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 3: return launch_fwd_k<T, 3>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 4: return launch_fwd_k<T, 4>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 5: return launch_fwd_k<T, 5>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 6: return launch_fwd_k<T, 6>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 7: return launch_fwd_k<T, 7>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    case 8: return launch_fwd_k<T, 8>(batch, dim, L, x, xbs, w, bias, silu, out, lengths, window, vec, st);
    default: return hipErrorInvalidValue;
  }
}

template <typename T>
hipError_t dispatch_bwd(int batch, int dim, int L, int K, const void* x, const void* w,
                        const void* bias, const void* dout, int silu, void* dx, void* dw,
                        void* dbias, float* part, bool vec, hipStream_t st) {
  switch (K) {
#define SSM_CONV_BWD_CASE(k)                                                                 \
  case k:                                                                                    \
    return launch_bwd_k<T, k>(batch, dim, L, x, w, bias, dout, silu, dx, dw, dbias, part, vec, \
                              st);
    SSM_CONV_BWD_CASE(1)
    SSM_CONV_BWD_CASE(2)
    SSM_CONV_BWD_CASE(3)
    SSM_CONV_BWD_CASE(4)
    SSM_CONV_BWD_CASE(5)
    SSM_CONV_BWD_CASE(6)
    SSM_CONV_BWD_CASE(7)
    SSM_CONV_BWD_CASE(8)
#undef SSM_CONV_BWD_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int conv1d_max_width() { return kMaxWidth; }

hipError_t launch_causal_conv1d_fwd(int batch, int dim, int L, int K, int dtype_bf16,
                                    const void* x, int64_t xbs, const void* w, const void* bias,
                                    int silu, void* out, const int64_t* lengths, void* window,
                                    bool vec, hipStream_t st) {
  return dtype_bf16 ? dispatch_fwd<__hip_bfloat16>(batch, dim, L, K, x, xbs, w, bias, silu, out,
                                                   lengths, window, vec, st)
                    : dispatch_fwd<float>(batch, dim, L, K, x, xbs, w, bias, silu, out, lengths,
                                          window, vec, st);
}

hipError_t launch_causal_conv1d_bwd(int batch, int dim, int L, int K, int dtype_bf16,
                                    const void* x, const void* w, const void* bias,
                                    const void* dout, int silu, void* dx, void* dw, void* dbias,
                                    float* part, bool vec, hipStream_t st) {
  return dtype_bf16 ? dispatch_bwd<__hip_bfloat16>(batch, dim, L, K, x, w, bias, dout, silu, dx, dw,
                                                   dbias, part, vec, st)
                    : dispatch_bwd<float>(batch, dim, L, K, x, w, bias, dout, silu, dx, dw, dbias,
                                          part, vec, st);
}

}  // namespace ssm
