// int8 x int8 -> int32 GEMM on gfx950 int8 MFMA (v_mfma_i32_32x32x32_i8):
// matmul_i8_i8_to_i32 (learn/api/functional.mojo:249-279) with the weight
// given in its stored layout w_q [N,K], optionally with the dequantize of
// QuantLinear (learn/nn/layers.mojo:1681-1685) fused into the epilogue.
// Integer products and sums are exact, so the result is bit-identical to
// the reference's i-j-p loop in any summation order (|acc| <= 127*128*K).
//
// gemm_i8_kernel<TB, ANY>: TB x TB tile per 256-thread workgroup, 64-wide K
// stages of int8 in LDS (rows padded to 80 B so 16-byte fragment reads of 16
// lanes hit distinct banks), double-buffered through registers.  The
// one-wave-per-SIMD kernel (gemm_i8_w4_kernel in gemm_nt.hip, 256 x 256 or 256 x
// 128 tiles) is faster at every measured shape it takes: MI355X, bit-identical
// outputs, settled A/B timed alternately, 128 x 128 tiles of this kernel against
// it: 4096^3 114.8 / 59.7 us, 3072 x 4096 x 4096 75.6 / 53.7, 2048 x 4096 x 4096
// 58.4 / 35.3, 1024 x 4096 x 4096 47.3 / 29.9, 512 x 11008 x 4096 53.2 / 33.3,
// 512 x 4096 x 11008 109.5 / 65.1, 1024 x 1024 x 4096 40.7 / 28.4, 1000 x 3000 x
// 1040 20.3 / 16.4, 300 x 520 x 4112 39.7 / 25.1, 512 x 512 x 4096 39.2 / 24.6.
// It runs what that kernel cannot address:
//  * 256 K >= 2^31 (tile offsets past 32 bits; TB = 128);
//  * ANY: rows that start at any byte (K not a multiple of 16, or unaligned
//    operands): 16-byte loads at byte addresses, which the hardware takes, and
//    single bytes where a row's last chunk reaches past K.  Against one thread
//    per output with a byte load per product, QuantLinear calls: 1000^3 3752 ->
//    17.4 us (17.9 at K = 1008 on the w4 kernel), 2000 x 2000 x 2001 32052 ->
//    48.9, 4096 x 4096 x 4095 252907 -> 205, 746 x 19 x 968 112 -> 15.1 (host).
#include "common.h"
#include "launch.h"

namespace mj {

constexpr int kIBK = 64;
constexpr int kILds = kIBK + 16;  // bytes per LDS row

typedef uint32_t u32x4b __attribute__((ext_vector_type(4), aligned(1)));

template <int TB, bool ANY>
__global__ __launch_bounds__(256) void gemm_i8_kernel(const int8_t *__restrict__ A,
                                                      const int8_t *__restrict__ B,
                                                      int32_t *__restrict__ C,
                                                      float *__restrict__ Y, float sf,
                                                      const float *__restrict__ bias, int M,
                                                      int N, int K) {
  constexpr int NB = TB / 64;  // 32 x 32 blocks per wave and dimension, rows per thread
  __shared__ __attribute__((aligned(16))) int8_t As[2][TB * kILds];
  __shared__ __attribute__((aligned(16))) int8_t Bs[2][TB * kILds];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_m = (int)(((int64_t)M + TB - 1) / TB), tiles_n = (int)(((int64_t)N + TB - 1) / TB);
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, 4, tm, tn);
  const int m0 = tm * TB, n0 = tn * TB;

  // 4 chunks of 16 B per 64-byte row: thread -> (row t/4 + 64 i, chunk t%4)
  const int c = tid & 3, r0 = tid >> 2;
  uint4 ra[NB], rb[NB];
  auto chunk = [&](const int8_t *X, int r, int R, int k) __attribute__((always_inline)) {
    if (r >= R || k >= K) return make_uint4(0, 0, 0, 0);
    const int8_t *q = X + (size_t)r * K + k;
    if constexpr (!ANY) return *(const uint4 *)q;
    if (K - k >= 16) {
      const u32x4b v = *(const u32x4b *)q;
      return make_uint4(v[0], v[1], v[2], v[3]);
    }
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 15; ++e)
      if (e < K - k) w[e >> 2] |= (uint32_t)(uint8_t)q[e] << (8 * (e & 3));
    return make_uint4(w[0], w[1], w[2], w[3]);
  };
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      ra[i] = chunk(A, m0 + r0 + 64 * i, M, k0 + c * 16);
      rb[i] = chunk(B, n0 + r0 + 64 * i, N, k0 + c * 16);
    }
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      *(uint4 *)(&As[buf][(r0 + 64 * i) * kILds + c * 16]) = ra[i];
      *(uint4 *)(&Bs[buf][(r0 + 64 * i) * kILds + c * 16]) = rb[i];
    }
  };

  i32x16 acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  const int nk = (int)(((int64_t)K + kIBK - 1) / kIBK);
  load(0);
  store(0);
  __syncthreads();
  const int fr = lane & 31, fk = (lane >> 5) * 16;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * kIBK);
#pragma unroll
    for (int ks = 0; ks < kIBK; ks += 32) {
      i32x4 a[NB], b[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i)
        a[i] = *(const i32x4 *)(&As[buf][(wm * (TB / 2) + i * 32 + fr) * kILds + ks + fk]);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        b[j] = *(const i32x4 *)(&Bs[buf][(wn * (TB / 2) + j * 32 + fr) * kILds + ks + fk]);
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + wn * (TB / 2) + j * 32 + (lane & 31);
    if (n >= N) continue;
    const float bb = Y ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * (TB / 2) + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (m >= M) continue;
        if (Y) {
#pragma clang fp contract(off)
          const float v = (float)acc[i][j][r] * sf;
          Y[(size_t)m * N + n] = v + bb;
        } else {
          C[(size_t)m * N + n] = acc[i][j][r];
        }
      }
  }
}

template <int TB, bool ANY>
static hipError_t launch_i8_tile(const int8_t *A, const int8_t *B, int32_t *C, float *y, float sf,
                                 const float *b, int64_t M, int64_t N, int64_t K,
                                 hipStream_t stream) {
  const int64_t tiles = ((M + TB - 1) / TB) * ((N + TB - 1) / TB);
  if (tiles > INT32_MAX) return hipErrorInvalidValue;  // grid.x limit
  hipLaunchKernelGGL((gemm_i8_kernel<TB, ANY>), dim3((unsigned)tiles), dim3(256), 0, stream, A, B,
                     C, y, sf, b, (int)M, (int)N, (int)K);
  return hipGetLastError();
}

hipError_t launch_gemm_i8(const int8_t *A, const int8_t *B, int32_t *C, float *y, float sf,
                          const float *b, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  if (256 * K < ((int64_t)1 << 31) && K % 16 == 0 && (((uintptr_t)A | (uintptr_t)B) & 15) == 0)
    return launch_gemm_i8_w4(A, B, C, y, sf, b, M, N, K, stream);
  return launch_i8_tile<128, false>(A, B, C, y, sf, b, M, N, K, stream);
}

// The same product for any K and alignment: 128 x 128 tiles where they give
// every CU one, else 64 x 64.
hipError_t launch_gemm_i8_any(const int8_t *A, const int8_t *B, int32_t *C, float *y, float sf,
                              const float *b, int64_t M, int64_t N, int64_t K,
                              hipStream_t stream) {
  if (((M + 127) / 128) * ((N + 127) / 128) >= 256)
    return launch_i8_tile<128, true>(A, B, C, y, sf, b, M, N, K, stream);
  return launch_i8_tile<64, true>(A, B, C, y, sf, b, M, N, K, stream);
}

// The reference's literal indexing bt._data[p*N + j] (functional.mojo:274), B
// read as a row-major [K,N] matrix: one thread per output, exact.
__global__ __launch_bounds__(256) void gemm_i8_literal_kernel(const int8_t *__restrict__ A,
                                                              const int8_t *__restrict__ B,
                                                              int32_t *__restrict__ C,
                                                              float *__restrict__ Y, float sf,
                                                              const float *__restrict__ bias,
                                                              int64_t M, int64_t N, int64_t K) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M * N) return;
  const int64_t i = t / N, j = t - i * N;
  int32_t acc = 0;
  for (int64_t p = 0; p < K; ++p) acc += (int32_t)A[i * K + p] * (int32_t)B[p * N + j];
  if (Y) {
#pragma clang fp contract(off)
    const float v = (float)acc * sf;
    Y[t] = v + bias[j];
  } else {
    C[t] = acc;
  }
}

hipError_t launch_gemm_i8_literal(const int8_t *A, const int8_t *B, int32_t *C, float *y, float sf,
                                  const float *b, int64_t M, int64_t N, int64_t K,
                                  hipStream_t stream) {
  const unsigned blocks = (unsigned)((M * N + 255) / 256);
  hipLaunchKernelGGL(gemm_i8_literal_kernel, dim3(blocks), dim3(256), 0, stream, A, B, C, y, sf, b,
                     M, N, K);
  return hipGetLastError();
}

}  // namespace mj
