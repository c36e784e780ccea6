// fp32 / fp64 engine on gfx950: the matmul / Linear / tensordot of momijo's
// Float32 and Float64 tensor engine (tensor/broadcast.mojo:1397-1900,
// tensor/math.mojo:7838-7880, learn/nn/layers.mojo:383-433).
//
// gemm_fx_kernel<T, TB>: C = epi(A @ B + bias) on v_mfma_f32_16x16x4f32 (T =
// float, full fp32 products) or v_mfma_f64_16x16x4f64 (T = double), a TB x TB
// tile per 256-thread workgroup (64; 128 for problems with enough tiles, where
// each wave then runs 4 x 4 MFMA blocks per LDS fragment read instead of
// 2 x 2; 32 for tiny fp64 products and convolutions, one block per wave; the 128
// and 64 tiles run eight waves, two per SIMD, of TB/2 x TB/4), K stages
// staged through LDS (k-major, padded; 16 deep, 64 (fp32) or 32 (fp64) on the
// 32 x 32 tiles).  Neither the tile size nor the stage depth changes any
// output's summation order.  Tiny fp32 products run gemm_f32_tiny_kernel (rounds of
// 256 k through LDS, the same MFMA sequence), small fp64 ones
// gemm_f64_direct_kernel.  Operands come as (pointer, row stride, column stride),
// which covers the reference's zero-copy transpose views; the loader walks
// whichever dimension has unit stride with consecutive lanes so global reads
// stay coalesced.  A grid dimension over broadcast batch indices serves
// tensordot's batched paths.  The fp32 kernels of this file take the products of
// up to 256^3 multiply-adds with K up to 1024, and all with K up to 16
// (f32s_takes); the others run on split bf16 operands (gemm_f32s.hip).
#include <type_traits>

#include "common.h"
#include "launch.h"

namespace mj {

constexpr int kFBK = 16;

typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4;

template <typename T> struct Acc;
// Both instructions read A[i][k] from lane i + 16 k and B[k][j] from lane
// j + 16 k.  Accumulator item r of lane l holds column l % 16 and row
// 4 (l / 16) + r for fp32, but row 4 r + l / 16 for fp64.
template <> struct Acc<float> {
  typedef f32x4 V;
  static __device__ __forceinline__ V mfma(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
template <> struct Acc<double> {
  typedef f64x4 V;
  static __device__ __forceinline__ V mfma(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
};

// One (batch, 64 x 64 tile) per workgroup: C[b] = epi(A[b] @ B[b] + bias),
// or with accum set C[b] = C[b] + A[b] @ B[b] (gradient accumulation: the old
// value plus the finished product, one rounding).
// The batch index (batch0 + blockIdx.y) is decomposed over up to 5 broadcast
// batch dimensions into element offsets of A and B; C is contiguous per batch.
// CONV: B is the image gathered by cv (above) instead of a strided view.
template <typename T, int TB, int BK = kFBK, bool CONV = false, int NW = 4>
__global__ __launch_bounds__(NW * 64) void gemm_fx_kernel(int M, int N, int K, const T *__restrict__ A,
                                                      int64_t sAm, int64_t sAk,
                                                      const T *__restrict__ B, int64_t sBk,
                                                      int64_t sBn, const T *__restrict__ bias,
                                                      int epi, int accum, T *__restrict__ C,
                                                      int64_t ldc, BatchDesc bd, int64_t batch0,
                                                      ConvDesc cv) {
  constexpr int kFBM = TB, kFBN = TB;
  constexpr int NT = NW * 64;
  constexpr int WGN = NW / 2;        // waves 2 x WGN
  constexpr int NBM = TB / 32;       // 16 x 16 blocks per wave along M
  constexpr int NBN = TB / (16 * WGN);  // and along N
  constexpr int EPT = TB * BK / NT;  // elements of each operand per thread per stage
  constexpr int MF = NT / TB;        // m-fast / n-fast loader: k rows per pass
  constexpr int KF = NT / BK;        // k-fast loader: m (n) columns per pass
  static_assert(EPT >= 1 && BK % 4 == 0 && NBN >= 1, "stage shape");
  __shared__ T As[2][BK][kFBM + 4];
  __shared__ T Bs[2][BK][kFBN + 4];

  {
    const int64_t bi = batch0 + blockIdx.y;
    int64_t b = bi, oa = 0, ob = 0;
    for (int d = bd.rank - 1; d >= 0; --d) {
      const int64_t i = b % bd.shape[d];
      b /= bd.shape[d];
      oa += i * bd.a_stride[d];
      ob += i * bd.b_stride[d];
    }
    A += oa;
    B += ob;
    C += bi * M * ldc;
  }

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN;
  const int tiles_n = (N + kFBN - 1) / kFBN;
  const int m0 = (blockIdx.x / tiles_n) * kFBM;
  const int n0 = (blockIdx.x % tiles_n) * kFBN;

  const bool a_k_fast = (sAk == 1);
  const bool b_n_fast = CONV || (sBn == 1) || (sBk != 1);

  // CONV: a thread's output pixel p = n0 + tid % TB is fixed; element i of
  // its B loads walks k = k0 + tid / TB + MF i, kept as (c, ky, kx) and
  // advanced by one stage after each load
  int cy0 = 0, cx0 = 0, cc[EPT], cky[EPT], ckx[EPT];
  bool cp_ok = false;
  if constexpr (CONV) {
    const int pix = n0 + tid % TB;
    cp_ok = pix < N;
    const int oy = cp_ok ? pix / cv.OW : 0;
    cy0 = oy * cv.sH - cv.pH;
    cx0 = (pix - oy * cv.OW) * cv.sW - cv.pW;
    const int khw = cv.kH * cv.kW;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int k = tid / TB + MF * i;
      cc[i] = k / khw;
      cky[i] = (k - cc[i] * khw) / cv.kW;
      ckx[i] = k - cc[i] * khw - cky[i] * cv.kW;
    }
  }

  T ra[EPT], rb[EPT];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      int m, k;
      if (a_k_fast) { k = tid % BK; m = tid / BK + KF * i; }
      else          { m = tid % TB; k = tid / TB + MF * i; }
      const int gm = m0 + m, gk = k0 + k;
      ra[i] = (gm < M && gk < K) ? A[(int64_t)gm * sAm + (int64_t)gk * sAk] : T(0);
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      if constexpr (CONV) {
        const int iy = cy0 + cky[i], ix = cx0 + ckx[i];
        const bool in = cp_ok && k0 + tid / TB + MF * i < K && (unsigned)iy < (unsigned)cv.H &&
                        (unsigned)ix < (unsigned)cv.W;
        rb[i] = in ? B[((int64_t)cc[i] * cv.H + iy) * cv.W + ix] : T(0);
        // advance (c, ky, kx) by BK: each digit carries at most once
        ckx[i] += cv.dkx;
        const int cx = ckx[i] >= cv.kW;
        ckx[i] -= cx ? cv.kW : 0;
        cky[i] += cv.dky + cx;
        const int cyc = cky[i] >= cv.kH;
        cky[i] -= cyc ? cv.kH : 0;
        cc[i] += cv.dc + cyc;
      } else {
        int n, k;
        if (b_n_fast) { n = tid % TB; k = tid / TB + MF * i; }
        else          { k = tid % BK; n = tid / BK + KF * i; }
        const int gn = n0 + n, gk = k0 + k;
        rb[i] = (gn < N && gk < K) ? B[(int64_t)gk * sBk + (int64_t)gn * sBn] : T(0);
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      int m, k;
      if (a_k_fast) { k = tid % BK; m = tid / BK + KF * i; }
      else          { m = tid % TB; k = tid / TB + MF * i; }
      As[buf][k][m] = ra[i];
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      int n, k;
      if (b_n_fast) { n = tid % TB; k = tid / TB + MF * i; }
      else          { k = tid % BK; n = tid / BK + KF * i; }
      Bs[buf][k][n] = rb[i];
    }
  };

  typename Acc<T>::V acc[NBM][NBN];
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = T(0);

  const int nk = (K + BK - 1) / BK;
  load(0);
  store(0);
  __syncthreads();
  const int fr = lane & 15, fk = lane >> 4;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      T a[NBM], b[NBN];
#pragma unroll
      for (int i = 0; i < NBM; ++i) a[i] = As[buf][kk + fk][wm * (TB / 2) + i * 16 + fr];
#pragma unroll
      for (int j = 0; j < NBN; ++j) b[j] = Bs[buf][kk + fk][wn * (TB / WGN) + j * 16 + fr];
#pragma unroll
      for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) acc[i][j] = Acc<T>::mfma(a[i], b[j], acc[i][j]);
    }
    if (kt + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    const int n = n0 + wn * (TB / WGN) + j * 16 + (lane & 15);
    if (n >= N) continue;
    const T bb = (bias && !CONV) ? bias[n] : T(0);
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * (TB / 2) + i * 16 + Acc<T>::row(lane, r);
        if (m < M) {
          T v = acc[i][j][r];
          if (bias) {
#pragma clang fp contract(off)
            v = v + (CONV ? bias[m] : bb);
          }
          if constexpr (sizeof(T) == sizeof(float)) v = apply_epi(epi, v);  // fp64: none
          T *dst = C + (int64_t)m * ldc + n;
          if (accum) {
#pragma clang fp contract(off)
            v = *dst + v;
          }
          *dst = v;
        }
      }
  }
}

// Tiny fp32 products, which wait on load latency and on the chain of MFMAs that
// the strict k order makes of every output: TB x TB outputs per workgroup (16:
// one wave computes, 32: each of the four a 16 x 16 block), K in rounds of 256
// through LDS.  All four waves load a round (the next one while this one
// multiplies), so a workgroup has 32 KB (TB = 16) in flight, and the computing
// wave reads its fragments 8 MFMAs ahead.  Same MFMA sequence in the same k
// order as gemm_fx_kernel, bit for bit (k past K are zero, as its padding is).
// The computing wave of a 16 x 16 tile alternates with the workgroup, so that
// workgroups on one CU do not queue on one SIMD.  AKF / BKF: k-contiguous
// operands are loaded 16 bytes a lane, others along their rows.  MI355X, against
// one wave per 16 x 16 tile with two batches of 128 k in its registers (both
// operands k-contiguous) and 32 x 32 tiles with 64-deep stages (other layouts),
// graph replays: 256^3 x W^T 6.9 -> 4.6 us, A B 7.9 -> 5.1; 64 x 512 x 512 11.5
// -> 6.5 and 12.3 -> 7.5; 32 x 512 x 1000 21.1 -> 10.9 and 21.5 -> 12.5; 1 x 256
// x 256 6.1 -> 3.9.
template <int TB, bool AKF, bool BKF>
__global__ __launch_bounds__(256) void gemm_f32_tiny_kernel(int M, int N, int K,
                                                            const float *__restrict__ A,
                                                            int64_t sAm, int64_t sAk,
                                                            const float *__restrict__ B,
                                                            int64_t sBk, int64_t sBn,
                                                            const float *__restrict__ bias,
                                                            int epi, int accum,
                                                            float *__restrict__ C, int64_t ldc,
                                                            BatchDesc bd, int64_t batch0) {
  constexpr int RK = 256, LD = RK + 4, NV = TB;  // NV: elements per thread and operand
  __shared__ __align__(16) float As[TB * LD + 64], Bs[TB * LD + 64];
  {
    const int64_t bi = batch0 + blockIdx.y;
    int64_t b = bi, oa = 0, ob = 0;
    for (int d = bd.rank - 1; d >= 0; --d) {
      const int64_t i = b % bd.shape[d];
      b /= bd.shape[d];
      oa += i * bd.a_stride[d];
      ob += i * bd.b_stride[d];
    }
    A += oa;
    B += ob;
    C += bi * M * ldc;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = (N + TB - 1) / TB;
  const int m0 = (int)(blockIdx.x / tiles_n) * TB, n0 = (int)(blockIdx.x % tiles_n) * TB;

  // element i of a thread: k-contiguous: row tid / 16 + 16 (i / 16), k 4 (tid %
  // 16 + 16 (i / 4 % 4)) + i % 4; else row tid % TB, k tid / TB + 256 / TB i
  auto load = [&](const float *X, bool kf, int r0, int R, int64_t sr, int64_t sk, int k0,
                  float (&x)[NV]) __attribute__((always_inline)) {
    if (kf) {
#pragma unroll
      for (int c = 0; c < NV / 4; ++c) {
        const int r = r0 + (tid >> 4) + 16 * (c >> 2);
        const int k = k0 + 4 * ((tid & 15) + 16 * (c & 3));
        const float *q = X + (int64_t)(r < R ? r : R - 1) * sr + k;
        if (k + 4 <= K) {
          typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
          const f32x4u v = *(const f32x4u *)q;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[4 * c + e] = v[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[4 * c + e] = 0.0f;
          if (k < K) {
            x[4 * c] = q[0];
            if (k + 1 < K) x[4 * c + 1] = q[1];
            if (k + 2 < K) x[4 * c + 2] = q[2];
          }
        }
      }
    } else {
      const int r = r0 + tid % TB;
      const float *q = X + (int64_t)(r < R ? r : R - 1) * sr;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int k = k0 + tid / TB + (256 / TB) * i;
        x[i] = k < K ? q[(int64_t)k * sk] : 0.0f;
      }
    }
  };
  auto store = [&](float *S, bool kf, const float (&x)[NV]) __attribute__((always_inline)) {
    if (kf) {
#pragma unroll
      for (int c = 0; c < NV / 4; ++c)
        *(f32x4 *)(S + ((tid >> 4) + 16 * (c >> 2)) * LD + 4 * ((tid & 15) + 16 * (c & 3))) =
            f32x4{x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]};
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) S[(tid % TB) * LD + tid / TB + (256 / TB) * i] = x[i];
    }
  };

  const int fr = lane & 15, fk = lane >> 4;
  const bool mine = TB == 32 || wave == (int)((blockIdx.x + blockIdx.y) & 3);
  const int bm = TB == 32 ? 16 * (wave >> 1) : 0, bn = TB == 32 ? 16 * (wave & 1) : 0;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  float xa[NV], xb[NV];
  load(A, AKF, m0, M, sAm, sAk, 0, xa);
  load(B, BKF, n0, N, sBn, sBk, 0, xb);
  for (int64_t k0 = 0; k0 < K; k0 += RK) {
    store(As, AKF, xa);
    store(Bs, BKF, xb);
    __syncthreads();
    if (k0 + RK < K) {
      load(A, AKF, m0, M, sAm, sAk, (int)k0 + RK, xa);
      load(B, BKF, n0, N, sBn, sBk, (int)k0 + RK, xb);
    }
    if (mine) {
      const float *pa = As + (bm + fr) * LD + fk, *pb = Bs + (bn + fr) * LD + fk;
      const int left = K - (int)k0, nu = ((left < RK ? left : RK) + 31) / 32;
      float a[2][8], b[2][8];
      auto frags = [&](int s, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          a[s][t] = pa[32 * u + 4 * t];
          b[s][t] = pb[32 * u + 4 * t];
        }
      };
      auto mma = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 8; ++t) acc = Acc<float>::mfma(a[s][t], b[s][t], acc);
      };
      frags(0, 0);
      for (int u = 0;;) {  // fragments past the round stay unused
        frags(1, u + 1);
        mma(0);
        if (++u >= nu) break;
        frags(0, u + 1);
        mma(1);
        if (++u >= nu) break;
      }
    }
    __syncthreads();
  }
  const int n = n0 + bn + fr;
  if (!mine || n >= N) return;
  const float bb = bias ? bias[n] : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = m0 + bm + Acc<float>::row(lane, r);
    if (m < M) {
      float v = acc[r];
      if (bias) {
#pragma clang fp contract(off)
        v = v + bb;
      }
      v = apply_epi(epi, v);
      float *dst = C + (int64_t)m * ldc + n;
      if (accum) {
#pragma clang fp contract(off)
        v = *dst + v;
      }
      *dst = v;
    }
  }
}

template <int TB>
static hipError_t launch_tiny(int64_t M, int64_t N, int64_t K, const float *A, int64_t sAm,
                              int64_t sAk, const float *B, int64_t sBk, int64_t sBn,
                              const float *bias, int epi, int accum, float *C, int64_t ldc,
                              const BatchDesc &bd, int64_t batches, hipStream_t stream) {
  // fewer than 64 tiles of 64 x 64 in all: both grid dimensions are small
  const dim3 grid((unsigned)(((M + TB - 1) / TB) * ((N + TB - 1) / TB)), (unsigned)batches);
  auto kernel = sAk == 1 ? (sBk == 1 ? gemm_f32_tiny_kernel<TB, true, true>
                                     : gemm_f32_tiny_kernel<TB, true, false>)
                         : (sBk == 1 ? gemm_f32_tiny_kernel<TB, false, true>
                                     : gemm_f32_tiny_kernel<TB, false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, (int)M, (int)N, (int)K, A, sAm, sAk, B,
                     sBk, sBn, bias, epi, accum, C, ldc, bd, (int64_t)0);
  return hipGetLastError();
}

// fp64 products with too few 64 x 64 tiles to fill the chip: TB x TB outputs per
// workgroup, K in blocks of 32 dealt over its NW waves, fragments loaded straight
// from memory two blocks ahead (a lane's eight k of a block are consecutive; A
// and B take the same k per MFMA, so any assignment of k to MFMAs gives the same
// product).  The waves' sums are added in wave order through LDS: the chain of
// roundings is K / NW + NW long, not K.  AKF / BKF: k-contiguous operands.
// MI355X, against 32 x 32 tiles with 32-deep stages (each stage a load round
// trip): 256^3 A B 9.6 -> 3.8 us, 512^3 29.6 -> 11.1, 59 x 70 x 1779 (x W^T) 50.0
// -> 11.2, 192 x 645 x 1280 36.4 -> 20.2, 186 x 28 x 1332 with both operands'
// rows contiguous 34.8 -> 8.9.  The staged tiles stay for short K in that last
// layout (70 x 1779 x 59: 4.7 against 6.7 us: eight 8-byte loads a block and
// operand, and no reuse of them).
template <int TB, int NW, bool AKF, bool BKF>
__global__ __launch_bounds__(NW * 64) void gemm_f64_direct_kernel(
    int M, int N, int K, const double *__restrict__ A, int64_t sAm, int64_t sAk,
    const double *__restrict__ B, int64_t sBk, int64_t sBn, int accum, double *__restrict__ C,
    int64_t ldc) {
  constexpr int NB = TB / 16, LDT = TB + 2, KB = 32;
  __shared__ double part[NW][TB][LDT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = (N + TB - 1) / TB;
  const int m0 = (int)(blockIdx.x / tiles_n) * TB, n0 = (int)(blockIdx.x % tiles_n) * TB;
  const int fr = lane & 15, fk = lane >> 4;
  const double *pa[NB], *pb[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int m = m0 + 16 * i + fr, n = n0 + 16 * i + fr;
    pa[i] = A + (int64_t)(m < M ? m : M - 1) * sAm;
    pb[i] = B + (int64_t)(n < N ? n : N - 1) * sBn;
  }
  auto fetch = [&](const double *q, bool kf, int64_t sk, int64_t k, double (&x)[8])
                   __attribute__((always_inline)) {
    if (k + 8 <= K) {
      const double *q0 = q + k * (kf ? 1 : sk);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = q0[e * (kf ? 1 : sk)];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = k + e < K ? q[(k + e) * (kf ? 1 : sk)] : 0.0;
    }
  };
  double xa[2][NB][8], xb[2][NB][8];
  auto load = [&](int s, int64_t kb) __attribute__((always_inline)) {
    if (kb * KB >= K) return;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      fetch(pa[i], AKF, sAk, kb * KB + 8 * fk, xa[s][i]);
      fetch(pb[i], BKF, sBk, kb * KB + 8 * fk, xb[s][i]);
    }
  };
  f64x4 acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto mma = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = Acc<double>::mfma(xa[s][i][e], xb[s][j][e], acc[i][j]);
  };
  load(0, wave);
  load(1, wave + NW);
  for (int64_t kb = wave; kb * KB < K; kb += 2 * NW) {
    mma(0);
    load(0, kb + 2 * NW);
    if ((kb + NW) * KB < K) {
      mma(1);
      load(1, kb + 3 * NW);
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[wave][16 * i + Acc<double>::row(lane, r)][16 * j + fr] = acc[i][j][r];
  __syncthreads();
  for (int o = tid; o < TB * TB; o += NW * 64) {
    const int r = o / TB, c = o % TB, m = m0 + r, n = n0 + c;
    if (m >= M || n >= N) continue;
    double v = part[0][r][c];
#pragma unroll
    for (int w = 1; w < NW; ++w) v = v + part[w][r][c];
    double *dst = C + (int64_t)m * ldc + n;
    if (accum) {
#pragma clang fp contract(off)
      v = *dst + v;
    }
    *dst = v;
  }
}

template <int TB, int NW>
static hipError_t launch_f64_direct(int64_t M, int64_t N, int64_t K, const double *A, int64_t sAm,
                                    int64_t sAk, const double *B, int64_t sBk, int64_t sBn,
                                    double *C, int64_t ldc, int accum, hipStream_t stream) {
  const int64_t tiles = ((M + TB - 1) / TB) * ((N + TB - 1) / TB);
  auto kernel = sAk == 1 ? (sBk == 1 ? gemm_f64_direct_kernel<TB, NW, true, true>
                                     : gemm_f64_direct_kernel<TB, NW, true, false>)
                         : (sBk == 1 ? gemm_f64_direct_kernel<TB, NW, false, true>
                                     : gemm_f64_direct_kernel<TB, NW, false, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(NW * 64), 0, stream, (int)M, (int)N,
                     (int)K, A, sAm, sAk, B, sBk, sBn, accum, C, ldc);
  return hipGetLastError();
}

// K per stage of the 32 x 32 tiles: each stage costs a global-load round
// trip that its MFMAs (BK / 4 per wave) cannot cover, so the latency-bound
// tiny problems take deep stages (fp32, convolutions only: 64, 37 KB of LDS; fp64:
// 32, the static LDS limit); per output the k order is the same at any depth
template <typename T>
constexpr int kTinyBK = sizeof(T) == 4 ? 64 : 32;

// Which native tile a product takes (see launch_fx).
struct FxPlan {
  bool big, tiny, wide;
};
template <typename T>
static FxPlan plan_fx(int64_t M, int64_t N, int64_t K, int64_t batches) {
  FxPlan pl;
  const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
  pl.big = M >= 256 && N >= 256 && tiles128 * batches >= 512 && !(K <= 16 && sizeof(T) == 4);
  pl.tiny = !pl.big && ((M + 63) / 64) * ((N + 63) / 64) * batches < 64;
  pl.wide = ((M + 15) / 16) * ((N + 15) / 16) * batches > 512;
  return pl;
}

const char *gemm_f32_kernel_name(int64_t M, int64_t N, int64_t K, int64_t batches, int64_t sAm,
                                 int64_t sBn) {
  if (f32s_takes(M, N, K)) {
    F32Args p;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.sAm = sAm; p.sBn = sBn;
    return f32s_kernel_name(p, batches);
  }
  const FxPlan pl = plan_fx<float>(M, N, K, batches);
  if (!pl.tiny) return pl.big ? "native 128x128" : "native 64x64";
  return pl.wide ? "native tiny 32" : "native tiny 16";
}

template <typename T>
static hipError_t launch_fx(int64_t M, int64_t N, int64_t K, const T *A, int64_t sAm,
                            int64_t sAk, const T *B, int64_t sBk, int64_t sBn, const T *bias,
                            int epi, int accum, T *C, int64_t ldc, const BatchDesc &bd,
                            int64_t batches, hipStream_t stream) {
  if constexpr (sizeof(T) == sizeof(float)) {
    if (f32s_takes(M, N, K)) {
      F32Args p;
      p.M = (int)M; p.N = (int)N; p.K = (int)K;
      p.A = A; p.sAm = sAm; p.sAk = sAk;
      p.B = B; p.sBk = sBk; p.sBn = sBn;
      p.bias = bias; p.epi = epi; p.accum = accum;
      p.C = C; p.ldc = ldc;
      p.bd = bd;
      return launch_gemm_f32s(p, batches, stream);
    }
  }
  // 128 x 128 tiles for matrices of at least 256 x 256 once they still give
  // every CU two workgroups (fp32 with a single stage takes 64 x 64, whose outputs
  // leave earlier: 3000 x 2900 x 16 23.9 -> 15.6 us, 4096 x 4096 x 16 26.7 -> 24.0);
  // problems of fewer than 64 tiles of 64 x 64 take gemm_f32_tiny_kernel in fp32 (16 x 16 tiles up to two workgroups per CU, 32
  // x 32 above); fp64 takes gemm_f64_direct_kernel with the same two tiles up to
  // one 32 x 32 tile per CU, else 32 x 32 staged tiles below 64 tiles of 64 x 64
  // (latency-bound launches: a quarter of the MFMA chain per wave and four times
  // the workgroups); the rest 64 x 64
  const auto [big, tiny, wide] = plan_fx<T>(M, N, K, batches);
  if constexpr (sizeof(T) == sizeof(float)) {
    if (tiny) {
      return wide ? launch_tiny<32>(M, N, K, A, sAm, sAk, B, sBk, sBn, bias, epi, accum, C, ldc,
                                    bd, batches, stream)
                  : launch_tiny<16>(M, N, K, A, sAm, sAk, B, sBk, sBn, bias, epi, accum, C, ldc,
                                    bd, batches, stream);
    }
  } else if (((M + 31) / 32) * ((N + 31) / 32) <= 256 && (sAk == 1 || sBk == 1 || K > 128)) {
    // fp64 comes without batches; a second 32 x 32 tile on a CU costs more than
    // the staged 64 x 64 tiles' load trips (1024^3: 76 us against 62)
    return wide ? launch_f64_direct<32, 4>(M, N, K, A, sAm, sAk, B, sBk, sBn, C, ldc, accum, stream)
                : launch_f64_direct<16, 4>(M, N, K, A, sAm, sAk, B, sBk, sBn, C, ldc, accum,
                                           stream);
  }
  const int TBs = big ? 128 : (tiny ? 32 : 64);
  const int64_t tiles64 = ((M + TBs - 1) / TBs) * ((N + TBs - 1) / TBs);
  if (tiles64 > INT32_MAX) return hipErrorInvalidValue;  // grid.x limit
  const int tiles = (int)tiles64;
  constexpr int64_t kMaxGridY = 65535;
  for (int64_t b0 = 0; b0 < batches; b0 += kMaxGridY) {
    const int64_t nb = batches - b0 < kMaxGridY ? batches - b0 : kMaxGridY;
    // eight waves (two per SIMD) on the 128 x 128 and 64 x 64 tiles, four on
    // the tiny 32 x 32 ones (measured on MI355X against four waves on the same
    // tiles: fp32 Linear.backward 4096 2857 -> 2694 us, fp32 2048^3 220 ->
    // 207 us, 1536^3 130 -> 119 us, fp64 4096^3 3293 -> 2657 us, fp64 2048^3
    // 411 -> 326 us)
    if (big)
      hipLaunchKernelGGL((gemm_fx_kernel<T, 128, kFBK, false, 8>), dim3(tiles, (unsigned)nb),
                         dim3(512), 0, stream, (int)M, (int)N, (int)K, A, sAm, sAk, B, sBk, sBn,
                         bias, epi, accum, C, ldc, bd, b0, ConvDesc{});
    else if (!tiny)
      hipLaunchKernelGGL((gemm_fx_kernel<T, 64, kFBK, false, 8>), dim3(tiles, (unsigned)nb),
                         dim3(512), 0, stream, (int)M, (int)N, (int)K, A, sAm, sAk, B, sBk, sBn,
                         bias, epi, accum, C, ldc, bd, b0, ConvDesc{});
    else if constexpr (sizeof(T) == sizeof(double))
      hipLaunchKernelGGL((gemm_fx_kernel<T, 32, kTinyBK<T>>), dim3(tiles, (unsigned)nb),
                         dim3(256), 0, stream, (int)M, (int)N, (int)K, A, sAm, sAk, B, sBk, sBn,
                         bias, epi, accum, C, ldc, bd, b0, ConvDesc{});
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_gemm_f32(int64_t M, int64_t N, int64_t K, const float *A, int64_t sAm,
                           int64_t sAk, const float *B, int64_t sBk, int64_t sBn,
                           const float *bias, int epi, float *C, int64_t ldc,
                           hipStream_t stream) {
  return launch_fx<float>(M, N, K, A, sAm, sAk, B, sBk, sBn, bias, epi, 0, C, ldc, BatchDesc{},
                          1, stream);
}

hipError_t launch_gemm_f32_accum(int64_t M, int64_t N, int64_t K, const float *A, int64_t sAm,
                                 int64_t sAk, const float *B, int64_t sBk, int64_t sBn, float *C,
                                 int64_t ldc, int accum, hipStream_t stream) {
  return launch_fx<float>(M, N, K, A, sAm, sAk, B, sBk, sBn, nullptr, 0, accum, C, ldc,
                          BatchDesc{}, 1, stream);
}

hipError_t launch_gemm_f32_batched(int64_t M, int64_t N, int64_t K, const float *A, int64_t sAm,
                                   int64_t sAk, const float *B, int64_t sBk, int64_t sBn,
                                   float *C, const BatchDesc &bd, int64_t batches,
                                   hipStream_t stream) {
  return launch_fx<float>(M, N, K, A, sAm, sAk, B, sBk, sBn, nullptr, 0, 0, C, N, bd, batches,
                          stream);
}

hipError_t launch_gemm_f64(int64_t M, int64_t N, int64_t K, const double *A, int64_t sAm,
                           int64_t sAk, const double *B, int64_t sBk, int64_t sBn, double *C,
                           int64_t ldc, int accum, hipStream_t stream) {
  return launch_fx<double>(M, N, K, A, sAm, sAk, B, sBk, sBn, nullptr, 0, accum, C, ldc,
                           BatchDesc{}, 1, stream);
}

// Conv2d.forward with OC >= 64 (conv2d_fx_kernel<NBN>): 64 x TBN tiles of
// (output channel, output pixel of one image), TBN = 32 NBN, eight waves
// 4 x 2 of 16 x 16 NBN, 16-deep K stages through LDS, with the MFMA of
// gemm_fx_kernel in the same k order (k ascending by 4, lane group fk
// supplying k = 4 t + fk): the outputs are bit-identical to it.
// The gather: thread t owns pixel n0 + t % 256 of the tile (t % 256 < TBN)
// and loads 8 k of each stage, waves 0-3 the first 8, waves 4-7 the last 8.
// Element k = (c kH + ky) kW + kx sits at (pixel base) + c H W + ky W + kx in
// the image, pixel base = (oy sH - pH) W + ox sW - pW; the (c, ky, kx) walk
// is the same for every lane of a wave (scalar registers), and an out-of-range
// buffer offset (a tap in the padding, k >= K, a pixel past the image) loads
// zero.  Two stages are in flight in registers while one multiplies from LDS.
// The LDS rows are padded to 16 mod 32 words, so the fragment reads of four
// consecutive k rows (16 lanes each) hit distinct banks.  Against one wave
// per SIMD (four waves of 32 x 16 NBN) the eight waves ran the bench layer
// (32 x 64 x 56 x 56, 3 x 3, pad 1) 116.5 us against 126.8 (MI355X, same
// tile).  Needs C H W and OC C kH kW below 2^29 (32-bit byte offsets).
template <int NBN>
__global__ __launch_bounds__(512) void conv2d_fx_kernel(int M, int Ng, int K,
                                                        const float *__restrict__ w,
                                                        const float *__restrict__ x,
                                                        const float *__restrict__ bias, int epi,
                                                        float *__restrict__ y, int64_t img0,
                                                        int C, ConvDesc cv) {
  constexpr int TBM = 64, TBN = 32 * NBN, BK = 16;
  constexpr int LDA = TBM + 16, LDB = TBN + 16;
  __shared__ float As[2][BK][LDA];
  __shared__ float Bs[2][BK][LDB];
  const int64_t img = img0 + blockIdx.y;
  const int hw = cv.H * cv.W;
  const int64_t chw = (int64_t)C * hw;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x + img * chw, chw * 4);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, (int64_t)M * K * 4);
  y += img * (int64_t)M * Ng;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_n = (Ng + TBN - 1) / TBN;
  const int m0 = (blockIdx.x / tiles_n) * TBM;
  const int n0 = (blockIdx.x % tiles_n) * TBN;

  const int kg = wave >> 2;      // k group of the B gather (wave-uniform)
  const int px = tid & 255;
  int iy0 = -(1 << 28), ix0 = 0, pbase = 0;
  if (px < TBN && n0 + px < Ng) {
    const int pix = n0 + px;
    const int oy = pix / cv.OW;
    iy0 = oy * cv.sH - cv.pH;
    ix0 = (pix - oy * cv.OW) * cv.sW - cv.pW;
    pbase = iy0 * cv.W + ix0;
  }
  // walk state: the (c, ky, kx) of k = 8 kg of the next stage to load
  const int khw = cv.kH * cv.kW;
  int wc = (8 * kg) / khw;
  int wky = (8 * kg - wc * khw) / cv.kW;
  int wkx = 8 * kg - wc * khw - wky * cv.kW;
  const int ak = tid & 15, am = tid >> 4;

  float ra[2][2], rb[2][8];
  auto step = [&]() {
    if (++wkx == cv.kW) {
      wkx = 0;
      if (++wky == cv.kH) {
        wky = 0;
        ++wc;
      }
    }
  };
  auto load = [&](int k0, auto slot_c) {
    constexpr int SL = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + am + 32 * i, k = k0 + ak;
      const uint32_t off = (m < M && k < K) ? (uint32_t)(m * K + k) * 4u : kOobOffset;
      ra[SL][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rw, off, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int iy = iy0 + wky, ix = ix0 + wkx;
      const bool in = (unsigned)iy < (unsigned)cv.H && (unsigned)ix < (unsigned)cv.W &&
                      k0 + 8 * kg + i < K;
      const uint32_t off = in ? (uint32_t)(pbase + wc * hw + wky * cv.W + wkx) * 4u : kOobOffset;
      rb[SL][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, off, 0, 0));
      step();
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) step();
  };
  auto store = [&](int buf, auto slot_c) {
    constexpr int SL = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < 2; ++i) As[buf][ak][am + 32 * i] = ra[SL][i];
    if (px < TBN) {
#pragma unroll
      for (int i = 0; i < 8; ++i) Bs[buf][8 * kg + i][px] = rb[SL][i];
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  f32x4 acc[NBN];
#pragma unroll
  for (int j = 0; j < NBN; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int nk = (K + BK - 1) / BK;
  const int fr = lane & 15, fk = lane >> 4;
  auto mma = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const float a = As[buf][kk + fk][wm * 16 + fr];
      float b[NBN];
#pragma unroll
      for (int j = 0; j < NBN; ++j) b[j] = Bs[buf][kk + fk][wn * 16 * NBN + j * 16 + fr];
#pragma unroll
      for (int j = 0; j < NBN; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[j], acc[j], 0, 0, 0);
    }
  };
  load(0, S0());
  if (nk > 1) load(BK, S1());
  store(0, S0());
  __syncthreads();
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    if (kt + 2 < nk) load((kt + 2) * BK, S0());
    mma(0);
    store(1, S1());
    __syncthreads();
    if (kt + 3 < nk) load((kt + 3) * BK, S1());
    mma(1);
    if (kt + 2 < nk) store(0, S0());
    __syncthreads();
  }
  if (kt < nk) mma(0);

#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    const int n = n0 + wn * 16 * NBN + j * 16 + fr;
    if (n >= Ng) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * 16 + 4 * fk + r;
      if (m < M) {
        float v = acc[j][r];
        if (bias) {
#pragma clang fp contract(off)
          v = v + bias[m];
        }
        y[(int64_t)m * Ng + n] = apply_epi(epi, v);
      }
    }
  }
}

// The native convolution's tile: OC >= 64 and a grid of at least 192 workgroups:
// conv2d_fx_kernel with 224- or 256-pixel tiles, whichever leaves fewer pixel
// columns on the busiest CU (workgroups of all images dealt over 256 CUs; 256 on a
// tie).  Against the square tiles (eight waves), MI355X: 32 x 64 x 56^2 -> 64 (448
// workgroups) 126 against 145 us, 16 x 64 x 56^2 -> 64 (224) 79.5 against 87.5, but
// 8 x 64 x 56^2 -> 64 (112) 74.5 against 49.1 and 16 x 128 x 28^2 -> 128 (128) 139
// against 90.  Narrower tiles of that kernel were slower than the square ones (128
// pixels: 158.6 us on the bench layer).  Returns 256 or 224, or the square tile's
// 128, 64 or 32.
static int plan_conv2d_native(int64_t M, int64_t Ng, int64_t K, int64_t N, int64_t image) {
  if (M >= 64 && image < ((int64_t)1 << 29) && M * K < ((int64_t)1 << 29)) {
    int pick = 0;
    int64_t best = INT64_MAX, wgs_best = 0;
    for (int tbn : {256, 224}) {
      const int64_t wgs = ((M + 63) / 64) * ((Ng + tbn - 1) / tbn) * N;
      const int64_t cost = (wgs + 255) / 256 * tbn;
      if (cost < best) {
        best = cost;
        pick = tbn;
        wgs_best = wgs;
      }
    }
    if (wgs_best >= 192) return pick;
  }
  const int64_t tiles128 = ((M + 127) / 128) * ((Ng + 127) / 128);
  if (M >= 256 && Ng >= 256 && tiles128 * N >= 512) return 128;
  return ((M + 63) / 64) * ((Ng + 63) / 64) * N < 64 ? 32 : 64;
}

const char *conv2d_f32_kernel_name(int64_t N, int64_t C, int64_t H, int64_t W, int64_t OC,
                                   int64_t kH, int64_t kW, int64_t OH, int64_t OW) {
  const int64_t K = C * kH * kW;
  if (f32s_takes(OC, OH * OW, K)) {
    F32Args p;
    p.M = (int)OC; p.N = (int)(OH * OW); p.K = (int)K;
    p.sAm = K;
    p.cv.H = (int)H; p.cv.W = (int)W; p.cv.kH = (int)kH; p.cv.kW = (int)kW;
    p.channels = (int)C;
    return conv2d_f32s_kernel_name(p, N);
  }
  switch (plan_conv2d_native(OC, OH * OW, K, N, C * H * W)) {
    case 256: return "native conv 256";
    case 224: return "native conv 224";
    case 128: return "native 128x128";
    case 64: return "native 64x64";
    default: return "native 32x32";
  }
}

// Conv2d.forward (NCHW) as one implicit GEMM per image: y[n] [OC, OH OW] =
// w [OC, C kH kW] @ im2col(x[n]) [C kH kW, OH OW] + b[oc], the image index
// on the grid's second dimension: conv2d_fx_kernel's 64 x 224 or 64 x 256
// tiles when they apply (below), else the matmul engine's square tiles as
// the matmul picks them (64 x 64, 128 x 128 for large problems, 32 x 32 for
// tiny ones).  Both sum each output in the same k order.
hipError_t launch_conv2d_f32(const float *x, const float *w, const float *b, float *y, int64_t N,
                             int64_t C, int64_t H, int64_t W, int64_t OC, int64_t kH,
                             int64_t kW, int64_t sH, int64_t sW, int64_t pH, int64_t pW,
                             int64_t OH, int64_t OW, int epi, hipStream_t stream) {
  const int64_t M = OC, Ng = OH * OW, K = C * kH * kW;
  constexpr int64_t kMaxGridY = 65535;
  ConvDesc cv;
  cv.H = (int)H; cv.W = (int)W; cv.OW = (int)OW; cv.kH = (int)kH; cv.kW = (int)kW;
  cv.sH = (int)sH; cv.sW = (int)sW; cv.pH = (int)pH; cv.pW = (int)pW;
  if (f32s_takes(M, Ng, K)) {
    F32Args p;
    p.M = (int)M; p.N = (int)Ng; p.K = (int)K;
    p.A = w; p.sAm = K; p.sAk = 1;
    p.B = x; p.sBn = 1;
    p.bias = b; p.epi = epi;
    p.C = y; p.ldc = Ng;
    p.bd.rank = 1;
    p.bd.shape[0] = N;
    p.bd.b_stride[0] = C * H * W;
    p.cv = cv;
    p.channels = (int)C;
    return launch_conv2d_f32s(p, N, stream);
  }
  const int tile = plan_conv2d_native(M, Ng, K, N, C * H * W);
  if (tile >= 224) {
    const int nbn = tile / 32;
    const int64_t tiles_c = ((M + 63) / 64) * ((Ng + 32 * nbn - 1) / (32 * nbn));
    if (tiles_c > INT32_MAX) return hipErrorInvalidValue;
    for (int64_t b0 = 0; b0 < N; b0 += kMaxGridY) {
      const int64_t nb = N - b0 < kMaxGridY ? N - b0 : kMaxGridY;
      const dim3 g((unsigned)tiles_c, (unsigned)nb);
      if (nbn == 8)
        hipLaunchKernelGGL((conv2d_fx_kernel<8>), g, dim3(512), 0, stream, (int)M, (int)Ng,
                           (int)K, w, x, b, epi, y, b0, (int)C, cv);
      else
        hipLaunchKernelGGL((conv2d_fx_kernel<7>), g, dim3(512), 0, stream, (int)M, (int)Ng,
                           (int)K, w, x, b, epi, y, b0, (int)C, cv);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  BatchDesc bd;
  bd.rank = 1;
  bd.shape[0] = N;
  bd.a_stride[0] = 0;
  bd.b_stride[0] = C * H * W;
  const int TBs = tile;
  const bool big = tile == 128, tiny = tile == 32;
  const int BKs = tiny ? kTinyBK<float> : kFBK;
  cv.dc = (int)(BKs / (kH * kW));
  cv.dky = (int)((BKs % (kH * kW)) / kW);
  cv.dkx = (int)(BKs % kW);
  const int64_t tiles64 = ((M + TBs - 1) / TBs) * ((Ng + TBs - 1) / TBs);
  if (tiles64 > INT32_MAX) return hipErrorInvalidValue;
  const int tiles = (int)tiles64;
  for (int64_t b0 = 0; b0 < N; b0 += kMaxGridY) {
    const int64_t nb = N - b0 < kMaxGridY ? N - b0 : kMaxGridY;
    // eight waves on the 128 and 64 tiles, as the matmul (against four:
    // 8 x 32 x 40^2 -> 96 32.4 -> 28.5 us, 4 x 64 x 56^2 -> 64 42.4 -> 32.6,
    // 16 x 128 x 28^2 -> 128 102 -> 90, 8 x 256 x 14^2 -> 256 144 -> 107,
    // 32 x 3 x 224^2 -> 32 (7 x 7, stride 2) 149 -> 143 us on MI355X)
    if (big)
      hipLaunchKernelGGL((gemm_fx_kernel<float, 128, kFBK, true, 8>), dim3(tiles, (unsigned)nb),
                         dim3(512), 0, stream, (int)M, (int)Ng, (int)K, w, K, (int64_t)1, x,
                         (int64_t)0, (int64_t)1, b, epi, 0, y, Ng, bd, b0, cv);
    else if (tiny)
      hipLaunchKernelGGL((gemm_fx_kernel<float, 32, kTinyBK<float>, true>),
                         dim3(tiles, (unsigned)nb), dim3(256), 0, stream, (int)M, (int)Ng, (int)K,
                         w, K, (int64_t)1, x, (int64_t)0, (int64_t)1, b, epi, 0, y, Ng, bd, b0,
                         cv);
    else
      hipLaunchKernelGGL((gemm_fx_kernel<float, 64, kFBK, true, 8>), dim3(tiles, (unsigned)nb),
                         dim3(512), 0, stream, (int)M, (int)Ng, (int)K, w, K, (int64_t)1, x,
                         (int64_t)0, (int64_t)1, b, epi, 0, y, Ng, bd, b0, cv);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Column sums s[o] = sum_n X[n, o] of a row-major [N, OutF] matrix, in
// ascending n within each of `segs` consecutive row segments; a second pass
// adds the segment sums in segment order.  With segs = 1 the order is the
// strict ascending-n order of the reference's db loop.  One thread per
// column: consecutive lanes read consecutive columns of a row.
__global__ __launch_bounds__(256) void colsum_seg_kernel(const float *__restrict__ X, int64_t N,
                                                         int64_t OutF, int64_t seg_len,
                                                         float *__restrict__ out) {
  const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= OutF) return;
  const int64_t n0 = (int64_t)blockIdx.y * seg_len;
  const int64_t n1 = n0 + seg_len < N ? n0 + seg_len : N;
  const float *p = X + o;
  float s = 0.0f;
  int64_t n = n0;
  for (; n + 8 <= n1; n += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(n + u) * OutF];
#pragma unroll
    for (int u = 0; u < 8; ++u) s = s + v[u];
  }
  for (; n < n1; ++n) s = s + p[n * OutF];
  out[(int64_t)blockIdx.y * OutF + o] = s;
}

__global__ __launch_bounds__(256) void colsum_combine_kernel(const float *__restrict__ part,
                                                             int64_t segs, int64_t OutF,
                                                             float *__restrict__ out) {
  const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= OutF) return;
  const float *p = part + o;
  float s = 0.0f;
  int64_t k = 0;
  for (; k + 8 <= segs; k += 8) {  // loads in flight together, adds in order
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(k + u) * OutF];
#pragma unroll
    for (int u = 0; u < 8; ++u) s = s + v[u];
  }
  for (; k < segs; ++k) s = s + p[k * OutF];
  out[o] = s;
}

int64_t colsum_segments(int64_t N, int64_t OutF) {
  const int64_t col_blocks = (OutF + 255) / 256;
  if (N <= 1024 || col_blocks >= 1024) return 1;
  int64_t segs = (1024 + col_blocks - 1) / col_blocks;  // ~1024 workgroups in all
  const int64_t max_segs = (N + 63) / 64;              // at least 64 rows per segment
  if (segs > max_segs) segs = max_segs;
  if (segs > 65535) segs = 65535;
  return segs;
}

hipError_t launch_colsum_f32(const float *X, int64_t N, int64_t OutF, float *out, float *part,
                             int64_t segs, hipStream_t stream) {
  const unsigned cb = (unsigned)((OutF + 255) / 256);
  if (segs <= 1) {
    hipLaunchKernelGGL(colsum_seg_kernel, dim3(cb, 1), dim3(256), 0, stream, X, N, OutF, N, out);
    return hipGetLastError();
  }
  const int64_t seg_len = (N + segs - 1) / segs;
  hipLaunchKernelGGL(colsum_seg_kernel, dim3(cb, (unsigned)segs), dim3(256), 0, stream, X, N,
                     OutF, seg_len, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(colsum_combine_kernel, dim3(cb), dim3(256), 0, stream, part, segs, OutF,
                     out);
  return hipGetLastError();
}

// y[m] = sum_n A[m,n] x[n]: one wave per row, lanes stride over n.
template <typename T>
__global__ __launch_bounds__(256) void matvec_kernel(int M, int N, const T *__restrict__ A,
                                                     int64_t sAm, int64_t sAn,
                                                     const T *__restrict__ x, int64_t sx,
                                                     T *__restrict__ y) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= M) return;
  const T *a = A + (int64_t)row * sAm;
  T acc = T(0);
  for (int n = lane; n < N; n += 64) acc += a[(int64_t)n * sAn] * x[(int64_t)n * sx];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) y[row] = acc;
}

hipError_t launch_matvec_f32(int64_t M, int64_t N, const float *A, int64_t sAm, int64_t sAn,
                             const float *x, int64_t sx, float *y, hipStream_t stream) {
  hipLaunchKernelGGL(matvec_kernel<float>, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, stream,
                     (int)M, (int)N, A, sAm, sAn, x, sx, y);
  return hipGetLastError();
}

hipError_t launch_matvec_f64(int64_t M, int64_t N, const double *A, int64_t sAm, int64_t sAn,
                             const double *x, int64_t sx, double *y, hipStream_t stream) {
  hipLaunchKernelGGL(matvec_kernel<double>, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, stream,
                     (int)M, (int)N, A, sAm, sAn, x, sx, y);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void activation_f32_kernel(int epi, const float *x, float *y,
                                                             int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    y[i] = apply_epi(epi, x[i]);
}

hipError_t launch_activation_f32(int epi, const float *x, float *y, int64_t n,
                                 hipStream_t stream) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(activation_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, epi,
                     x, y, n);
  return hipGetLastError();
}

// Tensor[Float32].maximum_scalar(s) = where(x >= s, x, s)
// (tensor/tensor.mojo:4232): x itself where x >= s (so -0 stays -0 at s = 0),
// else s (NaN >= s is false, so NaN gives s).
__global__ __launch_bounds__(256) void maximum_scalar_f32_kernel(const float *x, float s, float *y,
                                                                 int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float v = x[i];
    y[i] = v >= s ? v : s;
  }
}

hipError_t launch_maximum_scalar_f32(const float *x, float s, float *y, int64_t n,
                                     hipStream_t stream) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(maximum_scalar_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x,
                     s, y, n);
  return hipGetLastError();
}

// astype_f32_from_int (tensor/cast.mojo:5431-5437): Float32(Int) of each
// 64-bit element, rounded to nearest even (the conversion rounds once, from
// the exact integer).
__global__ __launch_bounds__(256) void cast_i64_f32_kernel(const int64_t *x, float *y, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    y[i] = (float)x[i];
}

hipError_t launch_cast_i64_f32(const int64_t *x, float *y, int64_t n, hipStream_t stream) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(cast_i64_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, y, n);
  return hipGetLastError();
}

}  // namespace mj
