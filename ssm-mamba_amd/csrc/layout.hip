// The boundary between token-major activations (batch, L, C), the layout of the
// reference's Block (modules/block.py:78-90), and the channel-major layout
// (batch, C, L) the conv and scan kernels stream, for gfx950:
//
//   rms_norm_tc_kernel      RMSNorm of token-major x, written channel-major (and
//                           token-major for the weight gradients' products)
//   rms_norm_tc_bwd_kernel  its backward: channel-major dh to token-major dx, the
//                           residual's gradient added, and the weight gradient
//   transpose_kernel        (batch, R, S) -> (batch, S, R)
//   batch_sum_kernel        sum over the batch, optionally transposed
//   scan_params_kernel      the scan's fp32 parameters from the stored ones, and back
//
// All are memory-bound; each reads and writes every element once.  Measured at
// (4, 2048, 1024) in bf16 (16.8 MB a tensor, 3.2 us at the copy rate): the norm
// 9.5 us (11.0 with a copy of x for the layer's sum, in place of a device copy
// of 6.5; 13.6 with the token-major result too), its backward 19 + 4 us, a
// transposition 5.4 to 5.7 us, a batch sum of four 2048 x 1024 matrices 4 us.  They
// replace strided copies of 42 us on either side of a layer and, in a training
// step, about 25 elementwise and reduction kernels of the norm (290 us).
//
// Split: the norm kernels hold 32 tokens x all channels per workgroup, so the
// statistics need no second pass over memory and 8192 tokens are 256
// workgroups; the transposition itself goes through LDS.
#include "ss_common.cuh"
#include "ss_io.cuh"
#include "ss_prof.h"

namespace ssm {

namespace {

constexpr int kTcThreads = 1024;                 // 16 waves
constexpr int kTcTok = 32;                       // tokens of a workgroup
constexpr int kTcGroups = kTcThreads / 64 / 2;   // waves over the channels (x 2 token halves)

// A 16-byte chunk of a row.
template <typename T> struct TcChunk;
template <> struct TcChunk<float> {
  static constexpr int E = 4;
  __device__ static __forceinline__ void cvt(const u32x4_v r, float* v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
  }
  __device__ static __forceinline__ u32x4_v pack(const float* v) {
    return u32x4_v{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                   __float_as_uint(v[3])};
  }
};
template <> struct TcChunk<__hip_bfloat16> {
  static constexpr int E = 8;
  __device__ static __forceinline__ void cvt(const u32x4_v r, float* v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf16_lo(r[i]);
      v[2 * i + 1] = bf16_hi(r[i]);
    }
  }
  __device__ static __forceinline__ u32x4_v pack(const float* v) {
    return u32x4_v{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                   pack_bf16x2(v[6], v[7])};
  }
};

// The workgroup's tile in LDS, channel rows of 32 tokens.  A lane of the
// token-major side holds chunk cl = lane % 8 of a 128-byte row piece for a pair
// of adjacent tokens, so it writes (reads) one token pair of E channel rows; a
// lane of the channel-major side moves 16 bytes of one row.  In bf16 a row is
// 16 words of token pairs: word p of channel c sits at word p ^ 4 ((c / 8) % 4)
// of row c ^ ((c / 32) % 2), which spreads the 8 chunks x 8 pairs of a wave
// over the 32 banks (two lanes each) and keeps 16-byte pieces whole.  In fp32 a
// row is 32 words: pair p at words 2 p ^ 4 ((c / 4) % 8).
template <typename T, int kMaxC> struct TcTile;
template <int kMaxC> struct TcTile<__hip_bfloat16, kMaxC> {
  static constexpr int kPieces = 4;  // 16-byte pieces of a row
  uint32_t w[kMaxC * 16];
  __device__ __forceinline__ uint32_t* word(int c, int p) {
    return &w[(c ^ ((c >> 5) & 1)) * 16 + (p ^ (4 * ((c >> 3) & 3)))];
  }
  __device__ __forceinline__ void put_pair(int c, int p, float a, float b) {
    *word(c, p) = pack_bf16x2(a, b);
  }
  __device__ __forceinline__ void get_pair(int c, int p, float& a, float& b) {
    const uint32_t v = *word(c, p);
    a = bf16_lo(v);
    b = bf16_hi(v);
  }
  __device__ __forceinline__ u32x4_v* piece(int c, int j) {
    return reinterpret_cast<u32x4_v*>(word(c, 4 * j));
  }
};
template <int kMaxC> struct TcTile<float, kMaxC> {
  static constexpr int kPieces = 8;
  uint32_t w[kMaxC * 32];
  __device__ __forceinline__ uint32_t* word(int c, int t) {
    return &w[c * 32 + (t ^ (4 * ((c >> 2) & 7)))];
  }
  __device__ __forceinline__ void put_pair(int c, int p, float a, float b) {
    *reinterpret_cast<u32x2_v*>(word(c, 2 * p)) = u32x2_v{__float_as_uint(a), __float_as_uint(b)};
  }
  __device__ __forceinline__ void get_pair(int c, int p, float& a, float& b) {
    const u32x2_v v = *reinterpret_cast<u32x2_v*>(word(c, 2 * p));
    a = __uint_as_float(v[0]);
    b = __uint_as_float(v[1]);
  }
  __device__ __forceinline__ u32x4_v* piece(int c, int j) {
    return reinterpret_cast<u32x4_v*>(word(c, 4 * j));
  }
};

// Thread geometry shared by the two norm kernels: wave = (token half, channel
// group), lane = (token pair of the half, chunk of a 128-byte row piece).
struct TcLane {
  int p, cl, grp, half;  // pair within the 32 tokens, chunk lane, channel group, token half
  __device__ __forceinline__ TcLane() {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    half = wave / kTcGroups;
    grp = wave % kTcGroups;
    p = 8 * half + (lane >> 3);
    cl = lane & 7;
  }
};

// Sum over the 8 chunk lanes and the 8 channel groups of a token pair's two
// values: the sums of tokens 2p, 2p + 1 in every lane (fixed order).
__device__ __forceinline__ void tc_token_sums(const TcLane& g, float (*red)[kTcTok], float& a, float& b) {
#pragma unroll
  for (int m = 1; m < 8; m <<= 1) {
    a += __shfl_xor(a, m, 64);
    b += __shfl_xor(b, m, 64);
  }
  if (g.cl == 0) {
    red[g.grp][2 * g.p] = a;
    red[g.grp][2 * g.p + 1] = b;
  }
  __syncthreads();
  a = b = 0.0f;
#pragma unroll
  for (int i = 0; i < kTcGroups; ++i) {
    a += red[i][2 * g.p];
    b += red[i][2 * g.p + 1];
  }
}

// The 32-token tile of the workgroup: consecutive tiles of a row, two of which
// share the 128-byte lines of the channel-major rows in bf16, on one XCD
// (workgroup i runs on XCD i % 8), so each line meets in one L2.
__device__ __forceinline__ bool tc_tile(int tiles_per_row, int ntiles, int& b, int& t0) {
  const int g = blockIdx.x;
  const int tile = (g / 16) * 16 + (g % 8) * 2 + (g % 16) / 8;
  if (tile >= ntiles) return false;
  b = tile / tiles_per_row;
  t0 = (tile - b * tiles_per_row) * kTcTok;
  return true;
}

// h[b, :, t] = x[b, t, :] * rsqrt(mean_c x^2 + eps) * (1 + w), fp32 statistics
// (modules/rms_norm.py:11-31).  C a multiple of E, rows 16-byte aligned.
// kVec: L a multiple of E and h_cm 16-byte aligned, so a row piece of a tile is
// wholly inside the row or past its end; otherwise element stores.
template <typename T, int kMaxC, bool kVec>
__global__ __launch_bounds__(kTcThreads) void rms_norm_tc_kernel(
    const T* __restrict__ x, const T* __restrict__ w, float eps, T* __restrict__ h_cm,
    T* __restrict__ h_tm, float* __restrict__ rstd, T* __restrict__ x_copy, int C, int L,
    int tiles_per_row, int ntiles) {
  using K = TcChunk<T>;
  constexpr int E = K::E;
  constexpr int kIter = (kMaxC + kTcGroups * 8 * E - 1) / (kTcGroups * 8 * E);
  __shared__ TcTile<T, kMaxC> tile;
  __shared__ float red[kTcGroups][kTcTok];
  int b, t0;
  if (!tc_tile(tiles_per_row, ntiles, b, t0)) return;  // whole workgroup, before any barrier
  const TcLane g;
  const int t = t0 + 2 * g.p;
  const bool ok0 = t < L, ok1 = t + 1 < L;
  const T* r0 = x + ((size_t)b * L + min(t, L - 1)) * C;
  const T* r1 = x + ((size_t)b * L + min(t + 1, L - 1)) * C;
  auto chan = [&](int i) { return ((i * kTcGroups + g.grp) * 8 + g.cl) * E; };
  // every load first, from clamped addresses (chunks past C count zero)
  u32x4_v v0[kIter], v1[kIter], wv[kIter];
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const int c = min(chan(i), C - E);
    v0[i] = *reinterpret_cast<const u32x4_v*>(r0 + c);
    v1[i] = *reinterpret_cast<const u32x4_v*>(r1 + c);
    wv[i] = *reinterpret_cast<const u32x4_v*>(w + c);
  }
  sched_fence();
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const uint32_t keep = chan(i) < C ? ~0u : 0u;
    v0[i] &= keep;
    v1[i] &= keep;
    float a[E], c[E];
    K::cvt(v0[i], a);
    K::cvt(v1[i], c);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      s0 = fmaf(a[j], a[j], s0);
      s1 = fmaf(c[j], c[j], s1);
    }
  }
  tc_token_sums(g, red, s0, s1);
  const float q0 = rsqrtf(s0 / (float)C + eps), q1 = rsqrtf(s1 / (float)C + eps);
  if (rstd && g.grp == 0 && g.cl == 0) {
    if (ok0) rstd[(size_t)b * L + t] = q0;
    if (ok1) rstd[(size_t)b * L + t + 1] = q1;
  }
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const int c = chan(i);
    if (c >= C) continue;
    float a[E], d[E], ww[E];
    K::cvt(v0[i], a);
    K::cvt(v1[i], d);
    K::cvt(wv[i], ww);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const float s = 1.0f + ww[j];
      a[j] = a[j] * q0 * s;
      d[j] = d[j] * q1 * s;
      tile.put_pair(c + j, g.p, a[j], d[j]);
    }
    if (x_copy) {
      if (ok0) *reinterpret_cast<u32x4_v*>(x_copy + ((size_t)b * L + t) * C + c) = v0[i];
      if (ok1) *reinterpret_cast<u32x4_v*>(x_copy + ((size_t)b * L + t + 1) * C + c) = v1[i];
    }
    if (h_tm) {
      if (ok0) *reinterpret_cast<u32x4_v*>(h_tm + ((size_t)b * L + t) * C + c) = K::pack(a);
      if (ok1) *reinterpret_cast<u32x4_v*>(h_tm + ((size_t)b * L + t + 1) * C + c) = K::pack(d);
    }
  }
  __syncthreads();
  // channel rows out, 16 bytes a lane
  constexpr int P = TcTile<T, kMaxC>::kPieces;
  for (int i = threadIdx.x; i < C * P; i += kTcThreads) {
    const int c = i / P, j = i % P, tt = t0 + j * E;
    const u32x4_v v = *tile.piece(c, j);
    T* dst = h_cm + ((size_t)b * C + c) * L + tt;
    if constexpr (kVec) {
      if (tt < L) *reinterpret_cast<u32x4_v*>(dst) = v;
    } else {
      float f[E];
      K::cvt(v, f);
#pragma unroll
      for (int k = 0; k < E; ++k)
        if (tt + k < L) Elem<T>::store1(dst + k, f[k]);
    }
  }
}

// With xh = x rstd, g = dh (1 + w) and m = mean_c g xh:
//   dx = dres + rstd (g - xh m),   dw[c] = sum_{b,t} dh xh
// (the derivative of the forward above).  part: two rows of C per workgroup (one
// per token half) with its sums of dh xh, added by norm_dw_kernel.
template <typename T, int kMaxC, bool kVec>
__global__ __launch_bounds__(kTcThreads) void rms_norm_tc_bwd_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ rstd,
    const T* __restrict__ dh, const T* __restrict__ dres, T* __restrict__ dx,
    float* __restrict__ part, int C, int L, int tiles_per_row, int ntiles) {
  using K = TcChunk<T>;
  constexpr int E = K::E;
  constexpr int kIter = (kMaxC + kTcGroups * 8 * E - 1) / (kTcGroups * 8 * E);
  constexpr int P = TcTile<T, kMaxC>::kPieces;
  constexpr int kLoad = (kMaxC * P + kTcThreads - 1) / kTcThreads;
  __shared__ TcTile<T, kMaxC> tile;
  __shared__ float red[kTcGroups][kTcTok];
  int b, t0;
  if (!tc_tile(tiles_per_row, ntiles, b, t0)) return;  // whole workgroup, before any barrier
  const int tile_id = b * tiles_per_row + t0 / kTcTok;
  const TcLane g;
  const int t = t0 + 2 * g.p;
  const bool ok0 = t < L, ok1 = t + 1 < L;
  const size_t o0 = ((size_t)b * L + min(t, L - 1)) * C, o1 = ((size_t)b * L + min(t + 1, L - 1)) * C;
  auto chan = [&](int i) { return ((i * kTcGroups + g.grp) * 8 + g.cl) * E; };
  // the channel-major tile and this lane's x chunks, all loads first
  u32x4_v dv[kLoad], v0[kIter], v1[kIter];
#pragma unroll
  for (int i = 0; i < kLoad; ++i) {
    const int it = min((int)threadIdx.x + i * kTcThreads, C * P - 1);
    const int c = it / P, tt = t0 + (it % P) * E;
    const T* src = dh + ((size_t)b * C + c) * L;
    if constexpr (kVec) {
      dv[i] = *reinterpret_cast<const u32x4_v*>(src + min(tt, L - E));
    } else {
      float f[E];
#pragma unroll
      for (int k = 0; k < E; ++k) f[k] = Elem<T>::load1(src + min(tt + k, L - 1));
      dv[i] = K::pack(f);
    }
  }
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const int c = min(chan(i), C - E);
    v0[i] = *reinterpret_cast<const u32x4_v*>(x + o0 + c);
    v1[i] = *reinterpret_cast<const u32x4_v*>(x + o1 + c);
  }
  const float q0 = rstd[(size_t)b * L + min(t, L - 1)], q1 = rstd[(size_t)b * L + min(t + 1, L - 1)];
  sched_fence();
#pragma unroll
  for (int i = 0; i < kLoad; ++i) {
    const int it = threadIdx.x + i * kTcThreads;
    if (it < C * P) *tile.piece(it / P, it % P) = dv[i];
  }
  __syncthreads();
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const int c = chan(i);
    const bool in = c < C;
    float a[E], d[E], ww[E], acc[E];
    K::cvt(v0[i], a);
    K::cvt(v1[i], d);
    K::cvt(*reinterpret_cast<const u32x4_v*>(w + min(c, C - E)), ww);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      float h0, h1;
      tile.get_pair(min(c, C - E) + j, g.p, h0, h1);
      // tokens past the end (clamped rows of other tokens) count nothing
      h0 = in && ok0 ? h0 * (a[j] * q0) : 0.0f;
      h1 = in && ok1 ? h1 * (d[j] * q1) : 0.0f;
      acc[j] = h0 + h1;
      s0 = fmaf(h0, 1.0f + ww[j], s0);
      s1 = fmaf(h1, 1.0f + ww[j], s1);
    }
    // sum of the half's 8 token pairs (lane bits 3..5): a reduce-scatter of
    // the E channels
    const int lane = threadIdx.x & 63;
    int idx = 0;
#pragma unroll
    for (int lv = 0, n = E; lv < 3; ++lv) {
      const int m = 8 << lv;
      const bool bit = (lane & m) != 0;
      if (n > 1) {
        n >>= 1;
#pragma unroll
        for (int k = 0; k < n; ++k) {
          const float keep = bit ? acc[k + n] : acc[k], send = bit ? acc[k] : acc[k + n];
          acc[k] = keep + __shfl_xor(send, m, 64);
        }
        idx += bit ? n : 0;
      } else {
        acc[0] += __shfl_xor(acc[0], m, 64);
      }
    }
    // (fp32: four channels over eight lanes, the pairs of lanes agree)
    if (in) part[((size_t)tile_id * 2 + g.half) * C + c + idx] = acc[0];
  }
  tc_token_sums(g, red, s0, s1);
  const float m0 = s0 / (float)C, m1 = s1 / (float)C;
#pragma unroll
  for (int i = 0; i < kIter; ++i) {
    const int c = chan(i);
    if (c >= C) continue;
    float a[E], d[E], ww[E], r0[E], r1[E];
    K::cvt(v0[i], a);
    K::cvt(v1[i], d);
    K::cvt(*reinterpret_cast<const u32x4_v*>(w + c), ww);
    if (dres) {
      K::cvt(*reinterpret_cast<const u32x4_v*>(dres + o0 + c), r0);
      K::cvt(*reinterpret_cast<const u32x4_v*>(dres + o1 + c), r1);
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) r0[j] = r1[j] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {
      float h0, h1;
      tile.get_pair(c + j, g.p, h0, h1);
      r0[j] = fmaf(q0, fmaf(-(a[j] * q0), m0, h0 * (1.0f + ww[j])), r0[j]);
      r1[j] = fmaf(q1, fmaf(-(d[j] * q1), m1, h1 * (1.0f + ww[j])), r1[j]);
    }
    if (ok0) *reinterpret_cast<u32x4_v*>(dx + o0 + c) = K::pack(r0);
    if (ok1) *reinterpret_cast<u32x4_v*>(dx + o1 + c) = K::pack(r1);
  }
}

// dw[c] = sum of `rows` partial rows, in a fixed order: 16 row groups of a
// workgroup (one wave each, 64 channels), then the groups.
template <typename T>
__global__ __launch_bounds__(1024) void norm_dw_kernel(const float* __restrict__ part,
                                                       T* __restrict__ dw, int rows, int C) {
  __shared__ float s[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const float* p = part + min(c, C - 1);
  float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  int r = wave;
  for (; r + 48 < rows; r += 64) {
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] += p[(size_t)(r + 16 * k) * C];
  }
  for (; r < rows; r += 16) a[0] += p[(size_t)r * C];
  s[wave][lane] = (a[0] + a[1]) + (a[2] + a[3]);
  __syncthreads();
  if (wave == 0 && c < C) {
    float v = s[0][lane];
#pragma unroll
    for (int i = 1; i < 16; ++i) v += s[i][lane];
    Elem<T>::store1(dw + c, v);
  }
}

// ---------------------------------------------------------------- transpositions

// out[b, s, r] = in[b, r, s], 64 x 64 elements per workgroup of 256 threads.
// kVec: R and S multiples of E, in and out 16-byte aligned (ibs a multiple of
// E): a lane moves 16-byte chunks of two adjacent rows, packed into row pairs
// in LDS (as TcTile: the swizzle spreads a wave's writes over the banks);
// otherwise element by element.
template <typename T, bool kVec>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ in, int64_t ibs,
                                                        T* __restrict__ out, int R, int S) {
  constexpr int E = TcChunk<T>::E;
  constexpr int kW = 64 * (int)sizeof(T) / 4;  // words of a 64-element row
  __shared__ uint32_t tile[64 * (kVec ? kW : 65)];
  const int r0 = blockIdx.y * 64, s0 = blockIdx.x * 64;
  const T* src = in + (size_t)blockIdx.z * ibs;
  T* dst = out + (size_t)blockIdx.z * R * S;
  if constexpr (kVec) {
    constexpr int kCh = 64 / E;  // chunks of a row: 8 (bf16) or 16 (fp32)
    constexpr int kPer = 32 * kCh / 256;
    // word w of column s at w ^ 4 (chunk of s % 8)
    auto word = [&](int s, int w) { return &tile[s * kW + (w ^ (4 * ((s / E) & 7)))]; };
    u32x4_v a[kPer], b[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int it = threadIdx.x + 256 * i, rp = it / kCh, ch = it % kCh;
      const int r = r0 + 2 * rp, s = min(s0 + ch * E, S - E);
      a[i] = *reinterpret_cast<const u32x4_v*>(src + (size_t)min(r, R - 1) * S + s);
      b[i] = *reinterpret_cast<const u32x4_v*>(src + (size_t)min(r + 1, R - 1) * S + s);
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int it = threadIdx.x + 256 * i, rp = it / kCh, ch = it % kCh;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        if constexpr (sizeof(T) == 2) {
          const uint32_t lo = a[i][k / 2], hi = b[i][k / 2];
          *word(ch * E + k, rp) = k % 2 ? (lo >> 16) | (hi & 0xffff0000u) : (lo & 0xffffu) | (hi << 16);
        } else {
          *reinterpret_cast<u32x2_v*>(word(ch * E + k, 2 * rp)) = u32x2_v{a[i][k], b[i][k]};
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * kPer; ++i) {
      const int it = threadIdx.x + 256 * i, s = it / kCh, ch = it % kCh;
      const int r = r0 + ch * E;
      if (s0 + s < S && r < R)
        *reinterpret_cast<u32x4_v*>(dst + (size_t)(s0 + s) * R + r) =
            *reinterpret_cast<const u32x4_v*>(word(s, 4 * ch));
    }
  } else {
    for (int it = threadIdx.x; it < 64 * 64; it += 256) {
      const int r = r0 + it / 64, s = s0 + it % 64;
      tile[(it / 64) * 65 + it % 64] =
          elem_bits(src[(size_t)min(r, R - 1) * S + min(s, S - 1)]);
    }
    __syncthreads();
    for (int it = threadIdx.x; it < 64 * 64; it += 256) {
      const int s = it / 64, r = it % 64;
      if (s0 + s < S && r0 + r < R)
        Elem<T>::store1(dst + (size_t)(s0 + s) * R + r0 + r, bits_to_f32<T>(tile[r * 65 + s]));
    }
  }
}

// out = sum over the batch of in (B, R, S), fp32 sums in batch order, rounded
// once; kTrans: out (S, R), else (R, S).  32 x 64 elements per workgroup (a weight
// gradient of 2048 x 1024 is 1024 workgroups).  kVec: S (and with kTrans R) a
// multiple of E, in and out 16-byte aligned: a thread sums E columns of a row,
// four batch rows' loads in flight; element by element otherwise.
template <typename T, bool kTrans, bool kVec>
__global__ __launch_bounds__(256) void batch_sum_kernel(const T* __restrict__ in,
                                                        T* __restrict__ out, int B, int R, int S) {
  constexpr int E = kVec ? TcChunk<T>::E : 1;
  constexpr int kCh = 64 / E, kPer = 32 * kCh / 256;
  constexpr int kIn = kVec ? 4 : 1;
  __shared__ float tile[kTrans ? 32 * 65 : 1];
  const int r0 = blockIdx.y * 32, s0 = blockIdx.x * 64;
  const size_t bs = (size_t)R * S;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int it = threadIdx.x + 256 * i, rl = it / kCh, sl = (it % kCh) * E;
    const T* p = in + (size_t)min(r0 + rl, R - 1) * S + min(s0 + sl, S - E);
    float v[E];
#pragma unroll
    for (int k = 0; k < E; ++k) v[k] = 0.0f;
    for (int b0 = 0; b0 < B; b0 += kIn) {
      float q[kIn][E];
#pragma unroll
      for (int u = 0; u < kIn; ++u) {
        const T* pb = p + (size_t)min(b0 + u, B - 1) * bs;
        if constexpr (kVec) TcChunk<T>::cvt(*reinterpret_cast<const u32x4_v*>(pb), q[u]);
        else q[u][0] = Elem<T>::load1(pb);
      }
#pragma unroll
      for (int u = 0; u < kIn; ++u)
#pragma unroll
        for (int k = 0; k < E; ++k) v[k] += b0 + u < B ? q[u][k] : 0.0f;
    }
    if constexpr (kTrans) {
#pragma unroll
      for (int k = 0; k < E; ++k) tile[rl * 65 + sl + k] = v[k];
    } else if (r0 + rl < R && s0 + sl < S) {
      T* dst = out + (size_t)(r0 + rl) * S + s0 + sl;
      if constexpr (kVec) *reinterpret_cast<u32x4_v*>(dst) = TcChunk<T>::pack(v);
      else Elem<T>::store1(dst, v[0]);
    }
  }
  if constexpr (kTrans) {
    __syncthreads();
    constexpr int kRc = 32 / E;  // row chunks of an output row
#pragma unroll
    for (int i = 0; i < 64 * kRc / 256 + (64 * kRc < 256); ++i) {
      const int it = threadIdx.x + 256 * i, sl = it / kRc, rl = (it % kRc) * E;
      if (sl >= 64 || s0 + sl >= S || r0 + rl >= R) continue;
      float v[E];
#pragma unroll
      for (int k = 0; k < E; ++k) v[k] = tile[(rl + k) * 65 + sl];
      T* dst = out + (size_t)(s0 + sl) * R + r0 + rl;
      if constexpr (kVec) *reinterpret_cast<u32x4_v*>(dst) = TcChunk<T>::pack(v);
      else Elem<T>::store1(dst, v[0]);
    }
  }
}

template <typename T, int kMaxC>
void launch_norm_fwd_c(const void* x, const void* w, float eps, void* h_cm, void* h_tm, float* rstd,
                       void* x_copy, int B, int L, int C, bool vec, hipStream_t st) {
  const int tpr = (L + kTcTok - 1) / kTcTok, nt = B * tpr;
  const dim3 grid((nt + 15) / 16 * 16);
#define SSM_NORM_TC(v)                                                                          \
  hipLaunchKernelGGL((rms_norm_tc_kernel<T, kMaxC, v>), grid, dim3(kTcThreads), 0, st,          \
                     static_cast<const T*>(x), static_cast<const T*>(w), eps,                   \
                     static_cast<T*>(h_cm), static_cast<T*>(h_tm), rstd,                        \
                     static_cast<T*>(x_copy), C, L, tpr, nt)
  if (vec) SSM_NORM_TC(true);
  else SSM_NORM_TC(false);
#undef SSM_NORM_TC
}

template <typename T, int kMaxC>
void launch_norm_bwd_c(const void* x, const void* w, const float* rstd, const void* dh,
                       const void* dres, void* dx, float* part, int B, int L, int C, bool vec,
                       hipStream_t st) {
  const int tpr = (L + kTcTok - 1) / kTcTok, nt = B * tpr;
  const dim3 grid((nt + 15) / 16 * 16);
#define SSM_NORM_TC(v)                                                                          \
  hipLaunchKernelGGL((rms_norm_tc_bwd_kernel<T, kMaxC, v>), grid, dim3(kTcThreads), 0, st,      \
                     static_cast<const T*>(x), static_cast<const T*>(w), rstd,                  \
                     static_cast<const T*>(dh), static_cast<const T*>(dres),                    \
                     static_cast<T*>(dx), part, C, L, tpr, nt)
  if (vec) SSM_NORM_TC(true);
  else SSM_NORM_TC(false);
#undef SSM_NORM_TC
}

// ---------------------------------------------------------------- scan parameters

// A = -exp(log_A) and the fp32 copies of D and the step-size bias (kBwd: dlog_A
// = dA * A and the gradients' casts).  A few 100 KB: what it costs is its
// launch, so all three go in one, an element per thread.  As torch ops a
// training step of a layer made 12 launches of 3.2 to 4.2 us for them (cast,
// exp and negation forward, the casts again in the backward, negation, product
// and three casts for the gradients): with two, the step at (4, 2048, 1024) bf16
// went from 938 to 892 us.
template <typename T, bool kBwd>
__global__ __launch_bounds__(256) void scan_params_kernel(
    const void* __restrict__ a_in, const float* __restrict__ A, const void* __restrict__ d_in,
    const void* __restrict__ b_in, void* __restrict__ a_out, void* __restrict__ d_out,
    void* __restrict__ b_out, const int nA, const int dim) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if constexpr (kBwd) {
    if (a_out && i < nA)
      Elem<T>::store1(static_cast<T*>(a_out) + i, static_cast<const float*>(a_in)[i] * A[i]);
    if (d_out && i < dim) Elem<T>::store1(static_cast<T*>(d_out) + i, static_cast<const float*>(d_in)[i]);
    if (b_out && i < dim) Elem<T>::store1(static_cast<T*>(b_out) + i, static_cast<const float*>(b_in)[i]);
  } else {
    if (i < nA) static_cast<float*>(a_out)[i] = -expf(Elem<T>::load1(static_cast<const T*>(a_in) + i));
    if (d_out && i < dim) static_cast<float*>(d_out)[i] = Elem<T>::load1(static_cast<const T*>(d_in) + i);
    if (b_out && i < dim) static_cast<float*>(b_out)[i] = Elem<T>::load1(static_cast<const T*>(b_in) + i);
  }
}

}  // namespace

// Channels the tile of 32 tokens holds in LDS: 128 KB at the largest.
int rms_norm_tc_max_channels(int bf16) { return bf16 ? 2048 : 1024; }

int rms_norm_tc_part_rows(int B, int L) { return 2 * B * ((L + kTcTok - 1) / kTcTok); }

hipError_t launch_rms_norm_tc(int bf16, const void* x, const void* w, float eps, void* h_cm,
                              void* h_tm, float* rstd, void* x_copy, int B, int L, int C, bool vec,
                              hipStream_t st) {
  ProfScope prof("rms_norm_tc", st);
  // the smallest tile that holds the channels: 64 KB tiles leave room for two
  // workgroups of a CU
  if (bf16) {
    if (C <= 1024) launch_norm_fwd_c<__hip_bfloat16, 1024>(x, w, eps, h_cm, h_tm, rstd, x_copy, B, L, C, vec, st);
    else launch_norm_fwd_c<__hip_bfloat16, 2048>(x, w, eps, h_cm, h_tm, rstd, x_copy, B, L, C, vec, st);
  } else {
    if (C <= 512) launch_norm_fwd_c<float, 512>(x, w, eps, h_cm, h_tm, rstd, x_copy, B, L, C, vec, st);
    else launch_norm_fwd_c<float, 1024>(x, w, eps, h_cm, h_tm, rstd, x_copy, B, L, C, vec, st);
  }
  return hipGetLastError();
}

hipError_t launch_rms_norm_tc_bwd(int bf16, const void* x, const void* w, const float* rstd,
                                  const void* dh, const void* dres, void* dx, void* dw, float* part,
                                  int B, int L, int C, bool vec, hipStream_t st) {
  {
    ProfScope prof("rms_norm_tc_bwd", st);
    if (bf16) {
      if (C <= 1024) launch_norm_bwd_c<__hip_bfloat16, 1024>(x, w, rstd, dh, dres, dx, part, B, L, C, vec, st);
      else launch_norm_bwd_c<__hip_bfloat16, 2048>(x, w, rstd, dh, dres, dx, part, B, L, C, vec, st);
    } else {
      if (C <= 512) launch_norm_bwd_c<float, 512>(x, w, rstd, dh, dres, dx, part, B, L, C, vec, st);
      else launch_norm_bwd_c<float, 1024>(x, w, rstd, dh, dres, dx, part, B, L, C, vec, st);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  ProfScope prof("norm_dw", st);
  const int rows = rms_norm_tc_part_rows(B, L);
  const dim3 grid((C + 63) / 64);
  if (bf16)
    hipLaunchKernelGGL((norm_dw_kernel<__hip_bfloat16>), grid, dim3(1024), 0, st, part,
                       static_cast<__hip_bfloat16*>(dw), rows, C);
  else
    hipLaunchKernelGGL((norm_dw_kernel<float>), grid, dim3(1024), 0, st, part,
                       static_cast<float*>(dw), rows, C);
  return hipGetLastError();
}

hipError_t launch_transpose(int bf16, const void* in, int64_t ibs, void* out, int B, int R, int S,
                            bool vec, hipStream_t st) {
  ProfScope prof("transpose", st);
  const dim3 grid((S + 63) / 64, (R + 63) / 64, B);
#define SSM_TR(T, v)                                                                            \
  hipLaunchKernelGGL((transpose_kernel<T, v>), grid, dim3(256), 0, st, static_cast<const T*>(in), \
                     ibs, static_cast<T*>(out), R, S)
  if (bf16) {
    if (vec) SSM_TR(__hip_bfloat16, true);
    else SSM_TR(__hip_bfloat16, false);
  } else {
    if (vec) SSM_TR(float, true);
    else SSM_TR(float, false);
  }
#undef SSM_TR
  return hipGetLastError();
}

hipError_t launch_batch_sum(int bf16, const void* in, void* out, int B, int R, int S, bool trans,
                            bool vec, hipStream_t st) {
  ProfScope prof("batch_sum", st);
  const dim3 grid((S + 63) / 64, (R + 31) / 32);
#define SSM_BS(T, t, v)                                                                          \
  hipLaunchKernelGGL((batch_sum_kernel<T, t, v>), grid, dim3(256), 0, st,                        \
                     static_cast<const T*>(in), static_cast<T*>(out), B, R, S)
  switch ((bf16 ? 4 : 0) + (trans ? 2 : 0) + (vec ? 1 : 0)) {
    case 0: SSM_BS(float, false, false); break;
    case 1: SSM_BS(float, false, true); break;
    case 2: SSM_BS(float, true, false); break;
    case 3: SSM_BS(float, true, true); break;
    case 4: SSM_BS(__hip_bfloat16, false, false); break;
    case 5: SSM_BS(__hip_bfloat16, false, true); break;
    case 6: SSM_BS(__hip_bfloat16, true, false); break;
    default: SSM_BS(__hip_bfloat16, true, true); break;
  }
#undef SSM_BS
  return hipGetLastError();
}

// nA, dim >= 1 (nA >= dim); bwd: a_in is dA, else log_A
hipError_t launch_scan_params(int bf16, bool bwd, const void* a_in, const float* A, const void* d_in,
                              const void* b_in, void* a_out, void* d_out, void* b_out, int nA,
                              int dim, hipStream_t st) {
  ProfScope prof("scan_params", st);
  const dim3 grid((nA + 255) / 256);
#define SSM_SP(T, b)                                                                            \
  hipLaunchKernelGGL((scan_params_kernel<T, b>), grid, dim3(256), 0, st, a_in, A, d_in, b_in,   \
                     a_out, d_out, b_out, nA, dim)
  if (bf16) {
    if (bwd) SSM_SP(__hip_bfloat16, true);
    else SSM_SP(__hip_bfloat16, false);
  } else {
    if (bwd) SSM_SP(float, true);
    else SSM_SP(float, false);
  }
#undef SSM_SP
  return hipGetLastError();
}

}  // namespace ssm
