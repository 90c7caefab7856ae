// Decode step of a Mamba block for a batch of sequences past the GEMV kernels'
// reach (9 to 64 rows), for gfx950: the projections of Block.step / Mamba.step
// (modules/block.py:80-86, modules/mamba.py:189-243 of the reference) as
// small matrix products on the matrix cores, with the work around them fused:
//
//   rows_gemm_kernel (norm, conv epilogue)  xz = W_in @ rmsnorm(x); for the x
//                                           half the conv step, SiLU and the
//                                           window roll
//   rows_gemm_kernel                        params = W_x @ xc
//   ssm_step_kernel (decode.hip)            step size, state update, gate
//   rows_gemm_kernel (residual)             x' = x + W_out @ y
//
// What bounds it: the weights, read once for all rows (22 MB of bytes a layer
// at d_model 1024, 4 us at the copy rate), and below that the latency of four
// short launches.  At 9 rows and more the GEMV kernels' fp32 multiply-adds per
// weight (one per row) would exceed the stream; an MFMA takes 16 rows at once.
// Measured at d_model 1024, batch 32, bf16: in-projection 7.8 us, x- and
// out-projection 7.2 each, state update 5.9, 28 us in all (43 at batch 64);
// the same step op by op (29 launches) took 99 us of kernels and 274 us a
// call, host-bound, against 30 now.
//
// Split: a workgroup owns kMT * 16 weight rows and every batch row; its waves
// split K in groups of kU MFMA steps (whole 256-byte pieces of a weight row),
// each wave issuing all loads of a group before its products, and add their
// totals through LDS in wave order, so the result does not depend on timing.
// With 16 rows to a workgroup an in-projection of 4096 rows is 256 workgroups,
// one per CU.  The activations (64 KB at batch 32, K 1024) come from L2
// straight into the operand layout: each wave reads only its K groups.
#include "ss_common.cuh"
#include "ss_io.cuh"
#include "ss_prof.h"

namespace ssm {

hipError_t launch_decode_ssm_step(int bf16, const void* p, int nout, int nparts, int R,
                                  const void* Wdt, const void* dtb, const void* logA, const void* D,
                                  const void* xc, const void* xz, int ld, float* state, void* y,
                                  int B, int dim, int nstate, bool vecR, hipStream_t st);

namespace {

typedef __bf16 rbf16x8_v __attribute__((ext_vector_type(8)));
typedef float rf32x4_v __attribute__((ext_vector_type(4)));

constexpr int kRowsU = 4;        // MFMA steps of a wave's K group
constexpr int kRowsTile = 16;    // weight rows, and batch rows, of one MFMA

struct RowsArgs {
  const void* W;     // (O, K)
  const void* x;     // (B, K)
  const void* nw;    // (K) RMSNorm weight (kNorm)
  float eps;
  const void* bias;  // (O) nullable
  const void* res;   // (B, O) nullable
  void* y;           // (B, O)
  int B, O, K;
  // conv epilogue: rows o < dim are xs; window (B, dim, width-1), weight (dim, width)
  int dim, width;
  void* ctx;
  const void* cw;
  const void* cb;    // nullable
  void* xc;          // (B, dim)
};

// One 16-byte chunk of a weight row against one of an activation row.  Lane l
// supplies row l % 16 of either operand and k positions 16-byte chunk l / 16 of
// the step: bf16 one 16x16x32 product (8 positions a lane), fp32 four 16x16x4
// (position i of every lane's chunk in product i; both operands agree on the
// positions, whose order does not matter to the sum).  The result's element
// r of lane l is weight row 4 (l / 16) + r, batch row l % 16.
template <typename T>
__device__ __forceinline__ rf32x4_v rows_mfma(u32x4_v a, u32x4_v b, rf32x4_v acc) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rbf16x8_v, a),
                                                   __builtin_bit_cast(rbf16x8_v, b), acc, 0, 0, 0);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i]), __uint_as_float(b[i]), acc,
                                                 0, 0, 0);
    return acc;
  }
}

// A chunk of x times (1 + norm weight), in T as the reference's normalised
// activations are (the row's scale multiplies the finished sums), and the sum
// of the chunk's squares.
template <typename T>
__device__ __forceinline__ u32x4_v rows_norm_chunk(u32x4_v x, u32x4_v w, float& ssq) {
  u32x4_v o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 2) {
      const float a = bf16_lo(x[i]), b = bf16_hi(x[i]);
      ssq = fmaf(a, a, ssq);
      ssq = fmaf(b, b, ssq);
      o[i] = pack_bf16x2(a * (1.0f + bf16_lo(w[i])), b * (1.0f + bf16_hi(w[i])));
    } else {
      const float a = __uint_as_float(x[i]);
      ssq = fmaf(a, a, ssq);
      o[i] = __float_as_uint(a * (1.0f + __uint_as_float(w[i])));
    }
  }
  return o;
}

template <typename T>
__device__ __forceinline__ float rows_round(float v) {
  T t;
  Elem<T>::store1(&t, v);
  return Elem<T>::load1(&t);
}

// kNT: batch tiles of 16 rows (B <= 16 kNT); kMT: weight tiles of 16 rows a
// workgroup; kW: waves; kTaps: 0 without the conv epilogue, else the largest
// conv width taken.
template <typename T, int kNT, int kMT, int kW, bool kNorm, int kTaps>
__global__ __launch_bounds__(64 * kW) void rows_gemm_kernel(const RowsArgs a) {
  constexpr int E = 16 / (int)sizeof(T);       // elements of a 16-byte chunk
  constexpr int kNB = kNT * kRowsTile;         // batch rows covered
  constexpr int kOB = kMT * kRowsTile;         // weight rows covered
  constexpr int kItems = (kNB * kOB + 64 * kW - 1) / (64 * kW);  // outputs a thread
  constexpr bool kConv = kTaps > 0;
  constexpr int kT = kConv ? kTaps : 2;
  __shared__ float s_sum[kW][kNB][kOB + 1];    // per-wave totals
  __shared__ float s_ssq[kNorm ? kW : 1][kNB];

  const int lane = threadIdx.x & 63;
  const int w = wave_id_uniform();
  const int o0 = blockIdx.x * kOB;
  const int B = a.B, O = a.O, K = a.K;
  const int lr = lane & 15, lc = lane >> 4;
  const T* __restrict__ W = static_cast<const T*>(a.W);
  const T* __restrict__ x = static_cast<const T*>(a.x);
  const T* __restrict__ nw = static_cast<const T*>(a.nw);

  rf32x4_v acc[kMT][kNT];
  float ssq[kNT];
#pragma unroll
  for (int n = 0; n < kNT; ++n) {
    ssq[n] = 0.0f;
#pragma unroll
    for (int m = 0; m < kMT; ++m) acc[m][n] = {0.0f, 0.0f, 0.0f, 0.0f};
  }

  // operand rows of this lane, clamped (rows past O or B are computed from a
  // valid row and never stored)
  const T* wrow[kMT];
  const T* xrow[kNT];
#pragma unroll
  for (int m = 0; m < kMT; ++m) wrow[m] = W + (size_t)min(o0 + m * kRowsTile + lr, O - 1) * K;
#pragma unroll
  for (int n = 0; n < kNT; ++n) xrow[n] = x + (size_t)min(n * kRowsTile + lr, B - 1) * K;

  // epilogue operands of this thread's outputs, from clamped addresses, ahead
  // of the weight stream (absent ones from a valid stand-in: no load in a branch)
  float e_bias[kItems], e_res[kItems], e_cb[kItems], e_cw[kItems][kT], e_win[kItems][kT - 1];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int it = threadIdx.x + i * 64 * kW;
    const int o = min(o0 + it % kOB, O - 1), n = min(it / kOB, B - 1);
    e_bias[i] = Elem<T>::load1((a.bias ? static_cast<const T*>(a.bias) : W) + o);
    if constexpr (!kConv) {
      e_res[i] = Elem<T>::load1(a.res ? static_cast<const T*>(a.res) + (size_t)n * O + o : W + o);
    } else {
      const int c = min(o, a.dim - 1), wd = a.width;
      const T* cw = static_cast<const T*>(a.cw) + (size_t)c * wd;
      const T* win = static_cast<const T*>(a.ctx) + ((size_t)n * a.dim + c) * (wd - 1);
#pragma unroll
      for (int j = 0; j < kT; ++j) e_cw[i][j] = Elem<T>::load1(cw + min(j, wd - 1));
#pragma unroll
      for (int j = 0; j < kT - 1; ++j) e_win[i][j] = Elem<T>::load1(win + min(j, wd - 2));
      e_cb[i] = Elem<T>::load1(a.cb ? static_cast<const T*>(a.cb) + c : cw);
    }
  }

  const int nstep = (K + 4 * E - 1) / (4 * E);
  for (int s0 = w * kRowsU; s0 < nstep; s0 += kW * kRowsU) {
    // Every load of the group first, from clamped addresses: one memory round
    // trip per group.  The fence keeps them together (left alone, the compiler
    // starts the products after the first loads to reuse their registers, and
    // waits four times: 14.8 against 7.2 us for the x- and out-projections of
    // the layer above).
    u32x4_v wa[kMT][kRowsU], xb[kNT][kRowsU], nv[kNorm ? kRowsU : 1];
#pragma unroll
    for (int u = 0; u < kRowsU; ++u) {
      const int kc = min((s0 + u) * 4 * E + lc * E, K - E);
#pragma unroll
      for (int m = 0; m < kMT; ++m)
        wa[m][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_v*>(wrow[m] + kc));
#pragma unroll
      for (int n = 0; n < kNT; ++n) xb[n][u] = *reinterpret_cast<const u32x4_v*>(xrow[n] + kc);
      if constexpr (kNorm) nv[u] = *reinterpret_cast<const u32x4_v*>(nw + kc);
    }
    sched_fence();
    // chunks past K become zeros in both operands
#pragma unroll
    for (int u = 0; u < kRowsU; ++u) {
      const uint32_t keep = (s0 + u) * 4 * E + lc * E < K ? ~0u : 0u;
#pragma unroll
      for (int m = 0; m < kMT; ++m) wa[m][u] &= keep;
#pragma unroll
      for (int n = 0; n < kNT; ++n) xb[n][u] &= keep;
    }
#pragma unroll
    for (int u = 0; u < kRowsU; ++u) {
#pragma unroll
      for (int n = 0; n < kNT; ++n) {
        u32x4_v v = xb[n][u];
        if constexpr (kNorm) v = rows_norm_chunk<T>(v, nv[u], ssq[n]);
#pragma unroll
        for (int m = 0; m < kMT; ++m) acc[m][n] = rows_mfma<T>(wa[m][u], v, acc[m][n]);
      }
    }
  }

#pragma unroll
  for (int m = 0; m < kMT; ++m)
#pragma unroll
    for (int n = 0; n < kNT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s_sum[w][n * kRowsTile + lr][m * kRowsTile + 4 * lc + r] = acc[m][n][r];
  if constexpr (kNorm) {
    // the four lanes of a batch row hold its chunks 0..3 of every step
#pragma unroll
    for (int n = 0; n < kNT; ++n) {
      float v = ssq[n];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lc == 0) s_ssq[w][n * kRowsTile + lr] = v;
    }
  }
  __syncthreads();

#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int it = threadIdx.x + i * 64 * kW;
    const int ol = it % kOB, n = it / kOB;
    const int o = o0 + ol;
    if (n >= B || o >= O) continue;
    float s = s_sum[0][n][ol];
#pragma unroll
    for (int ww = 1; ww < kW; ++ww) s += s_sum[ww][n][ol];
    if constexpr (kNorm) {
      float q = s_ssq[0][n];
#pragma unroll
      for (int ww = 1; ww < kW; ++ww) q += s_ssq[ww][n];
      s *= rsqrtf(q / (float)K + a.eps);
    }
    if (a.bias) s += e_bias[i];
    T* const yo = static_cast<T*>(a.y) + (size_t)n * O + o;
    if constexpr (!kConv) {
      Elem<T>::store1(yo, a.res ? s + e_res[i] : s);
    } else {
      Elem<T>::store1(yo, s);
      if (o < a.dim) {
        // conv step on the cached window, then the window drops its oldest
        // column and takes xs
        const int wd = a.width;
        const float xs = rows_round<T>(s);
        float cv = a.cb ? e_cb[i] : 0.0f;
        float wlast = 0.0f;
#pragma unroll
        for (int j = 0; j < kT; ++j) {
          if (j < kT - 1 && j < wd - 1) cv = fmaf(e_cw[i][j], e_win[i][min(j, kT - 2)], cv);
          if (j == wd - 1) wlast = e_cw[i][j];
        }
        cv = fmaf(wlast, xs, cv);
        Elem<T>::store1(static_cast<T*>(a.xc) + (size_t)n * a.dim + o, silu_f(cv));
        T* const win = static_cast<T*>(a.ctx) + ((size_t)n * a.dim + o) * (wd - 1);
#pragma unroll
        for (int j = 0; j + 1 < kT - 1; ++j)
          if (j + 1 < wd - 1) Elem<T>::store1(win + j, e_win[i][j + 1]);
        Elem<T>::store1(win + wd - 2, xs);
      }
    }
  }
}

template <typename T, int kNT, int kMT, int kW, bool kNorm, int kTaps>
void launch_rows_n(const RowsArgs& a, hipStream_t st) {
  const dim3 grid((a.O + kMT * kRowsTile - 1) / (kMT * kRowsTile));
  hipLaunchKernelGGL((rows_gemm_kernel<T, kNT, kMT, kW, kNorm, kTaps>), grid, dim3(64 * kW), 0, st, a);
}

// Shapes by the number of weight rows: two tiles to a workgroup for tall
// matrices (the LM head: half the reads of x), else one, with 16 waves where
// the rows alone leave half of the CUs idle or more (K is then split
// further; not with the norm, whose 16-wave form spills at 64 rows), else 8.
template <typename T, int kNT>
hipError_t launch_rows_b(const RowsArgs& a, hipStream_t st) {
  if (a.xc) {
    if (a.width <= 4) {
      if (a.nw) launch_rows_n<T, kNT, 1, 8, true, 4>(a, st);
      else launch_rows_n<T, kNT, 1, 8, false, 4>(a, st);
    } else {
      if (a.nw) launch_rows_n<T, kNT, 1, 8, true, 8>(a, st);
      else launch_rows_n<T, kNT, 1, 8, false, 8>(a, st);
    }
  } else if (a.O >= 16384) {
    if (a.nw) launch_rows_n<T, kNT, 2, 8, true, 0>(a, st);
    else launch_rows_n<T, kNT, 2, 8, false, 0>(a, st);
  } else if (a.nw) {
    launch_rows_n<T, kNT, 1, 8, true, 0>(a, st);
  } else if (a.O <= 2048) {
    launch_rows_n<T, kNT, 1, 16, false, 0>(a, st);
  } else {
    launch_rows_n<T, kNT, 1, 8, false, 0>(a, st);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rows_t(const RowsArgs& a, hipStream_t st) {
  if (a.B <= 16) return launch_rows_b<T, 1>(a, st);
  if (a.B <= 32) return launch_rows_b<T, 2>(a, st);
  return launch_rows_b<T, 4>(a, st);
}

}  // namespace

int decode_rows_max_batch() { return 64; }

hipError_t launch_decode_rows_linear(int bf16, const void* W, const void* x, const void* nw,
                                     float eps, const void* bias, const void* res, void* y, int B,
                                     int O, int K, hipStream_t st) {
  ProfScope prof("decode_rows_linear", st);
  RowsArgs a{};
  a.W = W; a.x = x; a.nw = nw; a.eps = eps; a.bias = bias; a.res = res; a.y = y;
  a.B = B; a.O = O; a.K = K;
  return bf16 ? launch_rows_t<__hip_bfloat16>(a, st) : launch_rows_t<float>(a, st);
}

hipError_t launch_decode_rows_in_proj(int bf16, const void* W, const void* x, const void* nw,
                                      float eps, const void* bias, void* xz, int B, int dim, int K,
                                      int width, void* ctx, const void* cw, const void* cb, void* xc,
                                      hipStream_t st) {
  ProfScope prof("decode_rows_in_proj", st);
  RowsArgs a{};
  a.W = W; a.x = x; a.nw = nw; a.eps = eps; a.bias = bias; a.y = xz;
  a.B = B; a.O = 2 * dim; a.K = K;
  a.dim = dim; a.width = width; a.ctx = ctx; a.cw = cw; a.cb = cb; a.xc = xc;
  return bf16 ? launch_rows_t<__hip_bfloat16>(a, st) : launch_rows_t<float>(a, st);
}

}  // namespace ssm
