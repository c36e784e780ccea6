// fp32 products on gfx950 bf16 MFMA: the matmul / Linear / tensordot / Conv2d
// of momijo's Float32 engine (tensor/broadcast.mojo:1543-1900,
// learn/nn/layers.mojo:383-433, learn/nn/conv.mojo:494-697).
//
// Every fp32 operand x is split into three bf16 numbers, x = h + m + l: h is x
// rounded to bf16, m the rounded rest x - h, l the rounded rest x - h - m (both
// rests are exact in fp32; 3 x 8 bits hold the 24 of x, so the sum is x unless
// l falls below the smallest bf16 denormal, see below).  A product a b is then
// ah bh + (ah bm + am bh) + (ah bl + am bm + al bh), each term exact in fp32;
// the three terms left out are below 2^-26 of it.  One v_mfma_f32_16x16x32_bf16
// does 32 k of one term in the cycles in which v_mfma_f32_16x16x4f32 does 2,
// so the six terms take 3/8 of the native fp32 time.
//
// The sum of every output, in every kernel of this file: for each block of 32 k
// (ascending) the six terms run small to large into a fresh accumulator t,
// then acc += t in fp32.  The order does not depend on the tile, so every kernel gives
// the same bits (Conv2d those of the matmul on its im2col).  t keeps the terms' roundings
// at the size of 32 products instead of the whole sum's, so the result is
// closer to the exact product than the native fp32 MFMA chain (which rounds
// after each product) from K = 3 on (K up to 16 runs natively all the same, see
// f32s_takes): relative error (2-norm) on N(0,1) data against 64 bits
// 4.7e-8 / 7.0e-8 / 1.2e-7 / 2.2e-7 at K = 64 / 256 / 1024 / 4096 against
// 1.4e-7 / 2.9e-7 / 5.7e-7 / 1.1e-6 for v_mfma_f32_16x16x4f32; on |N(0,1)|
// 4.0e-8 / 4.9e-8 / 8.1e-8 / 1.5e-7 against 1.2e-7 / 2.3e-7 / 4.4e-7 / 8.6e-7.
//
// What bounds it: six bf16 terms at the rate of a large bf16 product on this
// card (1440 TFLOP/s) are 240 fp32 TFLOP/s.  MI355X, against the native fp32
// kernels: 4096^3 1335 -> 597 us as x W^T, 630 with W row-major [K, N], 670 with
// both operands' rows contiguous (230 / 218 / 205 TFLOP/s, where the power
// limit holds the clock as in the bf16 GEMM); the training step of a 4096-wide
// Linear on 4096 rows 4002 -> 1945 us; 32 x (300 x 517 x 257) 47.4 -> 35.4 us.
//
// Where the split does not hold: an infinity (inf - inf = NaN in m) or a value
// that rounds to infinity in bf16 makes its outputs non-finite, and an element
// below 2^-110 has bits below 2^-133, the smallest bf16 denormal (which the MFMA
// keeps): it loses up to 2^-134.  The second matters where the rest of the
// output is as small, so an output is computed again on the native fp32 MFMA, in
// ascending k, if it is not finite (unless its row of A or column
// of B holds a NaN: NaN either way), or if its tile of A (of B) holds such an
// element and its magnitude is below 2^24 times what K of them can lose, K 2^-110
// times the largest of its column of B (row of A).  Every other output has lost
// at most 2^-24 of itself on each side, beside the sum's own roundings.
#include <atomic>
#include <cmath>

#include "common.h"
#include "launch.h"

namespace mj {

constexpr int kSBK = 32;               // k per stage: one MFMA deep
constexpr float kExactMin = 0x1p-110f; // h + m + l holds every fp32 number from here on

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// x[0..7] -> the three bf16 planes, packed in pairs; the rounding of
// pack_bf16x2 is to nearest even.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 &h, u32x4 &m, u32x4 &l) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    h[q] = pack_bf16x2(x[2 * q], x[2 * q + 1]);
    const float a = x[2 * q] - __uint_as_float(h[q] << 16);
    const float b = x[2 * q + 1] - __uint_as_float(h[q] & 0xFFFF0000u);
    m[q] = pack_bf16x2(a, b);
    l[q] = pack_bf16x2(a - __uint_as_float(m[q] << 16), b - __uint_as_float(m[q] & 0xFFFF0000u));
  }
}

// Running largest magnitude of a row; NaN once the row holds a NaN.
__device__ __forceinline__ float absmax3(float mx, float x, float y) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, fabsf(x)), fabsf(y));
}

// Operands are swapped (B^T rows feed the first operand), so lane l of a 16 x
// 16 block holds row l % 16 of the tile and columns 4 (l / 16) + r.
__device__ __forceinline__ f32x4 mfma_b16(const u32x4 &b, const u32x4 &a, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b),
                                                 __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
}

// Running smallest nonzero magnitude, as the fp32 bits without the sign times
// two minus one: zero becomes the largest number.
__device__ __forceinline__ uint32_t absmin3(uint32_t mn, float x, float y) {
  const uint32_t u = (__float_as_uint(x) << 1) - 1, v = (__float_as_uint(y) << 1) - 1;
  return __builtin_elementwise_min(__builtin_elementwise_min(mn, u), v);
}
__device__ __forceinline__ bool is_lossy(uint32_t mn) {
  return mn < 2 * __builtin_bit_cast(uint32_t, kExactMin) - 1;
}

// On the bits of a row's largest magnitude (non-negative floats order as their
// bits; NaN above all).
__device__ __forceinline__ bool is_nan(uint32_t mx) { return mx > 0x7F800000u; }
__device__ __forceinline__ bool is_finite(float v) { return fabsf(v) < __builtin_inff(); }

// Largest of the wave's magnitudes (as bits), a NaN taken as infinity: two quad
// permutes and two row rotations leave each 16-lane row's, read out as scalars.
__device__ __forceinline__ uint32_t wave_max_mag(uint32_t v) {
  v = min(v, 0x7F800000u);
#define MJ_DPP_MAX(ctrl) \
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, false))
  MJ_DPP_MAX(0xB1);   // quad_perm [1,0,3,2]
  MJ_DPP_MAX(0x4E);   // quad_perm [2,3,0,1]
  MJ_DPP_MAX(0x124);  // row_ror:4
  MJ_DPP_MAX(0x128);  // row_ror:8
#undef MJ_DPP_MAX
  uint32_t m = 0;
#pragma unroll
  for (int l = 0; l < 64; l += 16) m = max(m, (uint32_t)__builtin_amdgcn_readlane((int)v, l));
  return m;
}

// Whether output v is computed again: ma, mb the largest magnitudes of its row
// of A and column of B, la, lb whether elements of its tile's A, B lose bits (in a
// row or column of zeros they do not matter).  The product by 2^-110 comes first: it
// cannot overflow, and where it underflows the loss is below the smallest fp32
// denormal.
__device__ __forceinline__ bool split_fails(float v, uint32_t ma, uint32_t mb, bool la, bool lb,
                                            int K) {
  if (!is_finite(v)) return !is_nan(ma) && !is_nan(mb);
  const uint32_t mx = ma && mb ? max(la ? mb : 0u, lb ? ma : 0u) : 0u;
  return fabsf(v) < __uint_as_float(mx) * kExactMin * (float)K;
}

// x[c][iy][ix] of one image for k = (c kH + ky) kW + kx and pixel (iy0, ix0):
// zero in the padding.
__device__ __forceinline__ float conv_tap(const float *x, const ConvDesc &cv, int c, int ky, int kx,
                                          int iy0, int ix0) {
  const int iy = iy0 + ky, ix = ix0 + kx;
  const bool in = (unsigned)iy < (unsigned)cv.H && (unsigned)ix < (unsigned)cv.W;
  return in ? x[((int64_t)c * cv.H + iy) * cv.W + ix] : 0.0f;
}

__device__ __forceinline__ void conv_pixel(const ConvDesc &cv, int pix, int &iy0, int &ix0) {
  const int oy = pix / cv.OW;
  iy0 = oy * cv.sH - cv.pH;
  ix0 = (pix - oy * cv.OW) * cv.sW - cv.pW;
}

// Lane fr + 16 j holds 4 consecutive k of row fr, 4 j .. + 3 of a 16-deep chunk; a
// 4 x 4 transpose across the four 16-lane rows (two v_permlane32_swap, then two
// v_permlane16_swap) leaves k = 4 c + j in register c, what the MFMA c of the chunk
// takes from that lane.
__device__ __forceinline__ void transpose4_rows(const f32x4u &v, float *d) {
  const auto s0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]),
                                                   false, false);
  const auto s1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]),
                                                   false, false);
  const auto t0 = __builtin_amdgcn_permlane16_swap(s0[0], s1[0], false, false);
  const auto t1 = __builtin_amdgcn_permlane16_swap(s0[1], s1[1], false, false);
  d[0] = __uint_as_float(t0[0]);
  d[1] = __uint_as_float(t0[1]);
  d[2] = __uint_as_float(t1[0]);
  d[3] = __uint_as_float(t1[1]);
}

// One wave's look through row m of A and column n of B: 4 if the row, 8 if the
// column holds an element that loses bits.
template <bool CONV>
__device__ __forceinline__ uint32_t lossy_pair(const F32Args &p, const float *A, const float *B,
                                               int m, int n, int lane) {
  n = n < p.N ? n : p.N - 1;
  const float *pa = A + (int64_t)(m < p.M ? m : p.M - 1) * p.sAm;
  const float *pb = CONV ? B : B + (int64_t)n * p.sBn;
  const int khw = CONV ? p.cv.kH * p.cv.kW : 1;
  int iy0 = 0, ix0 = 0;
  if constexpr (CONV) conv_pixel(p.cv, n, iy0, ix0);
  uint32_t amin = ~0u, bmin = ~0u;
#pragma unroll 2
  for (int64_t k = lane; k < p.K; k += 64) {
    const float a = pa[k * p.sAk];
    float b;
    if constexpr (CONV) {
      const int c = (int)k / khw, t = (int)k - c * khw;
      b = conv_tap(B, p.cv, c, t / p.cv.kW, t % p.cv.kW, iy0, ix0);
    } else {
      b = pb[k * p.sBk];
    }
    amin = absmin3(amin, a, a);
    bmin = absmin3(bmin, b, b);
  }
  return (__builtin_amdgcn_ballot_w64(is_lossy(amin)) ? 4 : 0) |
         (__builtin_amdgcn_ballot_w64(is_lossy(bmin)) ? 8 : 0);
}

// 16 x 16 outputs from (mb, nb) on the native fp32 MFMA, k ascending, straight
// from memory, 32 k of loads in flight: the direct kernels' rare outputs that the
// split cannot give.
template <bool CONV>
__device__ __forceinline__ f32x4 exact_block(const F32Args &p, const float *A, const float *B,
                                             int mb, int nb, int lane) {
  const int fr = lane & 15, fk = lane >> 4;
  const int m = mb + fr < p.M ? mb + fr : p.M - 1;
  const int n = nb + fr < p.N ? nb + fr : p.N - 1;
  const float *pa = A + (int64_t)m * p.sAm;
  const float *pb = CONV ? B : B + (int64_t)n * p.sBn;
  int iy0 = 0, ix0 = 0;
  if constexpr (CONV) conv_pixel(p.cv, n, iy0, ix0);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = 8;
  float a[U], b[U];
  auto mma = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(b[u], a[u], acc, 0, 0, 0);
  };
  int64_t k0 = 0;
  if constexpr (!CONV) {
    auto fetch = [&](const float *q, int64_t sk, float(&x)[U]) __attribute__((always_inline)) {
      if (sk == 1) {
        f32x4u v[U / 4];
#pragma unroll
        for (int c = 0; c < U / 4; ++c) v[c] = *(const f32x4u *)(q + k0 + 16 * c + 4 * fk);
#pragma unroll
        for (int c = 0; c < U / 4; ++c) transpose4_rows(v[c], x + 4 * c);
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = q[(k0 + 4 * u + fk) * sk];
      }
    };
    for (; k0 + 4 * U <= p.K; k0 += 4 * U) {
      fetch(pa, p.sAk, a);
      fetch(pb, p.sBk, b);
      mma();
    }
  }
  const int khw = CONV ? p.cv.kH * p.cv.kW : 1;
  for (; k0 < p.K; k0 += 4 * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = k0 + 4 * u + fk, kc = k < p.K ? k : p.K - 1;
      a[u] = pa[kc * p.sAk];
      if constexpr (CONV) {
        const int c = (int)kc / khw, t = (int)kc - c * khw;
        b[u] = conv_tap(B, p.cv, c, t / p.cv.kW, t % p.cv.kW, iy0, ix0);
      } else {
        b[u] = pb[kc * p.sBk];
      }
      if (k >= p.K) a[u] = b[u] = 0.0f;
    }
    mma();
  }
  return acc;
}

// Offsets of the batch (or image) blockIdx.y + batch0 in A, B and C.
__device__ __forceinline__ void batch_offsets(const F32Args &p, const float *&A, const float *&B,
                                              float *&C) {
  const int64_t bi = p.batch0 + blockIdx.y;
  int64_t b = bi, oa = 0, ob = 0;
  for (int d = p.bd.rank - 1; d >= 0; --d) {
    // what is left is the first index: no division (64 bits, some hundred
    // instructions before a short tile's first load)
    const int64_t q = d > 0 ? b / p.bd.shape[d] : 0, i = b - q * p.bd.shape[d];
    b = q;
    oa += i * p.bd.a_stride[d];
    ob += i * p.bd.b_stride[d];
  }
  A = p.A + oa;
  B = p.B + ob;
  C = p.C + bi * p.M * p.ldc;
}

// bias, activation, accumulation and store of 4 consecutive columns of a row.
// CONV: the bias is per row (channel).
template <bool CONV>
__device__ __forceinline__ void store4_f32(const F32Args &p, float *C, int m, int n, f32x4 v) {
  float *dst = C + (int64_t)m * p.ldc + n;
  const int cnt = p.N - n < 4 ? p.N - n : 4;
  const float rb = CONV && p.bias ? p.bias[m] : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma clang fp contract(off)
    if (p.bias) v[r] = v[r] + (CONV ? rb : p.bias[r < cnt ? n + r : n]);
  }
  if (p.epi != EPI_NONE) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = apply_epi(p.epi, v[r]);
  }
  if (cnt == 4) {
    if (p.accum) v = *(const f32x4u *)dst + v;
    *(f32x4u *)dst = v;
  } else {
    for (int r = 0; r < cnt; ++r) dst[r] = p.accum ? dst[r] + v[r] : v[r];
  }
}

// ---------------------------------------------------------------- tiles
// TM x TN outputs per workgroup of WGM x WGN waves.  Per 32-deep stage each
// thread holds SA + SB "slots" of 8 consecutive k of one row in registers:
// loaded D + 1 stages ahead as fp32, split in the course of the MFMAs of the
// stage before theirs (16-byte or pairs of 8-byte LDS writes), so no pass over
// the operands comes before the product.  With eight waves the two of a SIMD
// work in opposite halves of a stage (PP): one reads fragments, writes LDS and
// requests loads while the other's MFMAs run, a barrier between the halves;
// 4096^3 on 256 x 128 tiles 696 -> 644 us, on 128 x 128 783 -> 700 us against
// both waves in step.  The split runs in the matrix half between the MFMAs, on
// the 256 x 128 tiles (whose registers are full there) in the memory half.  Counters
// (MFMA busy / VALU busy / LDS busy): 4096^3 64 / 52 / 28 %, under the power limit; 32
// x (300 x 517 x 257) 18 / 35 / 25, the conv of 32 x 64 x 56^2 21 / 50 / 28 on 64 x 64
// tiles, with a fifth of the LDS cycles in bank conflicts.  LDS: rows of 64 bytes per
// plane, their four octets permuted by lds_unit so that writes (4 rows of 4 octets, or
// 16 rows of one) and fragment reads (16 rows of one octet per 16 lanes) spread
// over all banks.
// AKF / BKF: the operand is k-contiguous (rows of the Linear layout): four
// lanes read the 128 bytes of a row's stage.  Otherwise (a stride view, whose
// rows are contiguous unless both strides are above 1) lanes walk the rows and
// the octet is the wave's.
// CONV: B is the image gathered as in exact_block.  A stage's 8 taps are the
// wave's: eight lanes compute tap number and offset of one k each, the wave
// reads them as scalars, and a per-pixel bit mask of the taps in the padding
// turns their loads out of range, which gives zero.  Four vector operations a
// tap; a scalar walk over (c, ky, kx) with the bounds compared per tap made the
// gather the larger half of a stage: 32 x 64 x 56^2 -> 64, 3 x 3 111 -> 79 us on
// MI355X (native fp32 117), 16 x 128 x 28^2 -> 128 52 us (native 90).  The mask is
// built by kernel rows: tap by tap it was a sixth of a short-K launch (32 x 3 x
// 102^2 -> 64, 5 x 5: 76 -> 66 us, native 69; 7 x 7 of stride 2 on 112^2 44 -> 34).
// ANY: kernels of more than 64 taps, which the mask does not hold: bounds
// compared per tap, divisions instead of the reciprocals.
// 16-byte unit of k octet o of row r within a plane.  The hardware serves a
// 16-byte read in groups of 16 lanes, {0-3, 12-15, 20-27} and its complement in
// each half wave; with the octet xor'ed by 0, 2, 3, 1 for rows 0-3, 4-7, 8-11,
// 12-15 such a group covers the 256 bytes of the banks once, and so do 16
// consecutive rows of one octet (measured: no conflicts left; octet-major rows
// padded by 64 bytes had half of the LDS cycles lost to conflicts).
__device__ __forceinline__ int lds_unit(int r, int o) {
  return r * 4 + (o ^ ((0x78 >> ((r >> 1) & 6)) & 3));
}

template <int TM, int TN, int WGM, int WGN>
struct TileS {
  static constexpr int NT = WGM * WGN * 64;
  static constexpr int PA = TM * 4, PB = TN * 4;           // 16-byte units per plane
  static constexpr int STAGE = 3 * (PA + PB) * 16;         // bytes
  static constexpr int LDT = TN + 4;                       // output staging row (floats)
  static constexpr int LDN = kSBK + 4;                     // native stage's row (floats)
  static constexpr int OUT = (TM * LDT > (TM + TN) * LDN ? TM * LDT : (TM + TN) * LDN) * 4;
  static constexpr int TAIL = 2 * STAGE > OUT ? 2 * STAGE : OUT;  // then row maxima and flags
  static constexpr int LDS = TAIL + (TM + TN + 3) * 4;
};

template <int TM, int TN, int WGM, int WGN, int D, bool AKF, bool BKF, bool CONV, bool ANY>
__global__ __launch_bounds__(WGM * WGN * 64, WGM * WGN == 4 ? 3 : 2) void gemm_f32s_kernel(
    F32Args p) {
  using T = TileS<TM, TN, WGM, WGN>;
  constexpr int NW = WGM * WGN, NT = T::NT, PA = T::PA, PB = T::PB;
  constexpr bool PP = NW == 8;
  constexpr int WTM = TM / WGM, WTN = TN / WGN, TMF = WTM / 16, TNF = WTN / 16;
  constexpr int RP = NT / 4;                 // rows per slot pass
  constexpr int SA = TM / RP, SB = TN / RP, NS = SA + SB;
  constexpr bool SM = TM == 256;  // the split in the memory half of a stage
  constexpr int VPM = SM ? 1 : 3; // VALU operations scheduled beside each MFMA
  static_assert(NT >= 256 && SA >= 1 && SB >= 1 && WTM <= 64 && WTN <= 64 && TMF * TNF <= 32,
                "tile shape");
  extern __shared__ __align__(16) char lds[];

  const float *A, *B;
  float *C;
  batch_offsets(p, A, B, C);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  int tm, tn;
  tile_coords(blockIdx.x, (p.M + TM - 1) / TM, (p.N + TN - 1) / TN, 4, tm, tn);
  const int m0 = tm * TM, n0 = tn * TN;
  const int K = p.K;
  const int nk = (int)(((unsigned)K + kSBK - 1) / kSBK);

  // Loader.  A slot is 8 elements of one thread: for a k-contiguous operand 4
  // consecutive k (chunk tid % 8) of two rows NT / 8 apart, so that eight lanes
  // read the 128 bytes of a row's stage; otherwise 8 consecutive k (the wave's
  // octet) of one row.  Row offsets are bytes from the tile's first row.
  const int uoct = wave / (NT / 256);
  const int c4 = tid & 7;
  uint32_t va[SA][2], vb[SB][2];
  int iy0[SB], ix0[SB], pbase[SB];           // CONV: the slot's pixel
  const float *ta = A + (int64_t)m0 * p.sAm, *tb = CONV ? B : B + (int64_t)n0 * p.sBn;
  auto slot_row = [&](bool kf, int s, int h) __attribute__((always_inline)) {
    return kf ? (tid >> 3) + (2 * s + h) * (NT / 8) : tid % RP + s * RP;
  };
#pragma unroll
  for (int s = 0; s < SA; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = slot_row(AKF, s, h), rc = m0 + r < p.M ? r : p.M - 1 - m0;
      va[s][h] = (uint32_t)(rc * (int)p.sAm) * 4u + (AKF ? 16u * c4 : 0u);
    }
#pragma unroll
  for (int s = 0; s < SB; ++s) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = slot_row(BKF && !CONV, s, h), rc = n0 + r < p.N ? r : p.N - 1 - n0;
      if constexpr (CONV) {
        conv_pixel(p.cv, n0 + rc, iy0[s], ix0[s]);
        pbase[s] = iy0[s] * p.cv.W + ix0[s];
      } else {
        vb[s][h] = (uint32_t)(rc * (int)p.sBn) * 4u + (BKF ? 16u * c4 : 0u);
      }
    }
  }
  // CONV: the image as a buffer, and per slot the taps that fall into the padding
  const int hw = CONV ? p.cv.H * p.cv.W : 0, khw = CONV ? p.cv.kH * p.cv.kW : 1;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(B, CONV ? (int64_t)p.channels * hw * 4 : 0);
  uint32_t out[SB][2];
  const uint32_t mc = 0xFFFFFFFFu / (uint32_t)khw + 1, mk = 65535u / (uint32_t)p.cv.kW + 1;
  if constexpr (CONV && !ANY) {
#pragma unroll
    for (int s = 0; s < SB; ++s) {
      // the taps of one kernel row outside the image's width, then row by row
      auto low = [](int n) { return n >= 64 ? ~(uint64_t)0 : ((uint64_t)1 << max(n, 0)) - 1; };
      const uint64_t row = low(p.cv.kW);
      const uint64_t side = row & ~(low(p.cv.W - ix0[s]) & ~low(-ix0[s]));
      uint64_t o = 0;
      for (int ky = 0; ky < p.cv.kH; ++ky)
        o |= ((unsigned)(iy0[s] + ky) < (unsigned)p.cv.H ? side : row) << (ky * p.cv.kW);
      out[s][0] = (uint32_t)o;
      out[s][1] = (uint32_t)(o >> 32);
    }
  }

  uint32_t *rma = (uint32_t *)(lds + T::TAIL), *rmb = rma + TM;  // row maxima as bits
  uint32_t *lossy = rmb + TN;  // an element that loses bits: of A, of B
  uint32_t *again = lossy + 2; // outputs not finite: 1, operands to read again: 2, lossy: 4, 8
  for (int i = tid; i < TM + TN + 3; i += NT) rma[i] = 0;

  float raw[D][NS][8];     // slots as loaded
  u32x4 sp[NS][3];         // and split, on their way to LDS
  float rmax[NS][2];
#pragma unroll
  for (int s = 0; s < NS; ++s) rmax[s][0] = rmax[s][1] = 0.0f;

  // part: the stage at k0 reaches past K; its k are clamped to the last
  // (split_slot clears them)
  auto load_kf = [&](const float *t, const uint32_t (&v)[2], int k0, float (&x)[8], bool part)
                     __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!part) {
        const f32x4u u = *(const f32x4u *)((const char *)(t + k0) + v[h]);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[4 * h + i] = u[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = k0 + 4 * c4 + i < K ? k0 + 4 * c4 + i : K - 1;
          x[4 * h + i] = *(const float *)((const char *)(t + (k - 4 * c4)) + v[h]);
        }
      }
    }
  };
  auto load_rf = [&](const float *t, int64_t sk, uint32_t v, int k0, float (&x)[8], bool part)
                     __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + 8 * uoct + i;
      x[i] = *(const float *)((const char *)(t + (int64_t)(part && k >= K ? K - 1 : k) * sk) + v);
    }
  };
  auto load_slot = [&](float(&x)[8], int s, int k0, bool part) __attribute__((always_inline)) {
    if (s < SA) {
      if constexpr (AKF) load_kf(ta, va[s], k0, x, part);
      else load_rf(ta, p.sAk, va[s][0], k0, x, part);
    } else if constexpr (CONV) {
      // the stage's 8 taps, one per lane: tap number t of channel c and its
      // byte offset from the pixel's first tap, then read out as scalars
      const uint32_t k = (uint32_t)(k0 + 8 * uoct + c4);
      const uint32_t c = khw == 1 ? k : ANY ? k / (uint32_t)khw : __umulhi(k, mc);
      const uint32_t t = k - c * (uint32_t)khw, ky = ANY ? t / (uint32_t)p.cv.kW : (t * mk) >> 16;
      const int off = (int)(c * (uint32_t)hw + t + ky * (uint32_t)(p.cv.W - p.cv.kW));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t o = (uint32_t)(pbase[s - SA] + __builtin_amdgcn_readlane(off, i)) * 4u;
        uint32_t bad;
        if constexpr (ANY) {
          const int y = __builtin_amdgcn_readlane((int)ky, i);
          const int x0 = __builtin_amdgcn_readlane((int)t, i) - y * p.cv.kW;
          bad = (unsigned)(iy0[s - SA] + y) < (unsigned)p.cv.H &&
                        (unsigned)(ix0[s - SA] + x0) < (unsigned)p.cv.W
                    ? 0u
                    : ~0u;
        } else {
          const int ti = __builtin_amdgcn_readlane((int)t, i);
          const uint32_t m = ti < 32 ? out[s - SA][0] : out[s - SA][1];
          bad = (uint32_t)__builtin_amdgcn_sbfe((int)m, ti & 31, 1);
        }
        // channels past the last lie past the buffer and load zero as well
        x[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            rx, (bad & kOobOffset) | (~bad & o), 0, 0));
      }
    } else {
      if constexpr (BKF) load_kf(tb, vb[s - SA], k0, x, part);
      else load_rf(tb, p.sBk, vb[s - SA][0], k0, x, part);
    }
  };
  auto clear_past_k = [&](float(&x)[8], int s, int k0) __attribute__((always_inline)) {
    const bool kf = s < SA ? AKF : BKF && !CONV;
    if (CONV && s >= SA) return;  // loaded as zeros
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (k0 + (kf ? 4 * c4 + i % 4 : 8 * uoct + i) >= K) x[i] = 0.0f;
  };
  auto split_slot = [&](int set, int s, int k0, bool part) __attribute__((always_inline)) {
    float(&x)[8] = raw[set][s];
    const bool kf = s < SA ? AKF : BKF && !CONV;
    if (part) clear_past_k(x, s, k0);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      float &mx = rmax[s][kf ? i / 4 : 0];
      mx = absmax3(mx, x[i], x[i + 1]);
    }
    split8(x, sp[s][0], sp[s][1], sp[s][2]);
  };
  auto write_slot = [&](int s, int buf) __attribute__((always_inline)) {
    u32x4 *d = (u32x4 *)(lds + buf * T::STAGE) + (s < SA ? 0 : 3 * PA);
    const int sl = s < SA ? s : s - SA, ps = s < SA ? PA : PB;
    if (s < SA ? AKF : BKF && !CONV) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint2 *e = (uint2 *)(d + lds_unit(slot_row(true, sl, h), c4 >> 1)) + (c4 & 1);
#pragma unroll
        for (int q = 0; q < 3; ++q)
          e[2 * q * ps] = make_uint2(sp[s][q][2 * h], sp[s][q][2 * h + 1]);
      }
    } else {
      u32x4 *e = d + lds_unit(slot_row(false, sl, 0), uoct);
#pragma unroll
      for (int q = 0; q < 3; ++q) e[q * ps] = sp[s][q];
    }
  };

  const int fr = lane & 15, fo = lane >> 4;
  f32x4 acc[TMF][TNF];
#pragma unroll
  for (int i = 0; i < TMF; ++i)
#pragma unroll
    for (int j = 0; j < TNF; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

  u32x4 fa[3][TMF], fb[3][TNF];
  const int nfull = K / kSBK;
  // Memory half of stage kt (in buffer buf = kt % 2): its fragments from LDS,
  // the next stage's split slots to the other buffer, the loads of stage kt + 1
  // + D requested.  full: all of these stages exist and lie inside K.
  auto stage_mem = [&](int kt, int buf, bool full) __attribute__((always_inline)) {
    const u32x4 *sa = (const u32x4 *)(lds + buf * T::STAGE) + lds_unit(wm * WTM + fr, fo);
    const u32x4 *sb =
        (const u32x4 *)(lds + buf * T::STAGE) + 3 * PA + lds_unit(wn * WTN + fr, fo);
    auto load_next = [&](int s) __attribute__((always_inline)) {
      if (full || kt + 1 + D < nk)
        load_slot(raw[(kt + 1 + D) % D][s], s, (kt + 1 + D) * kSBK,
                  !full && kt + 1 + D >= nfull);
    };
    if constexpr (!SM) {
#pragma unroll
      for (int s = 0; s < NS; ++s) load_next(s);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int j = 0; j < TNF; ++j) fb[q][j] = sb[q * PB + j * 64];
#pragma unroll
      for (int i = 0; i < TMF; ++i) fa[q][i] = sa[q * PA + i * 64];
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (full || kt + 1 < nk) {
        if constexpr (SM)
          split_slot(0, s, (kt + 1) * kSBK, !full && kt + 1 >= nfull);
        write_slot(s, buf ^ 1);
      }
      if constexpr (SM) load_next(s);
    }
  };
  // Matrix half: the MFMAs of stage kt in groups of 2 blocks (two chains of the
  // six terms), between them the sums of the group before and, in the last
  // groups, the split of stage kt + 2.
  auto stage_mma = [&](int kt, bool full) __attribute__((always_inline)) {
    constexpr int NG = TMF * TNF / 2;
    f32x4 t[2][2];
    auto flush = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[2 * g / TNF][2 * g % TNF + j] += t[g & 1][j];
    };
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int i = 2 * g / TNF, j0 = 2 * g % TNF;
      f32x4(&tg)[2] = t[g & 1];
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[0][j0 + j], fa[2][i], zero);
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[2][j0 + j], fa[0][i], tg[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[1][j0 + j], fa[1][i], tg[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[0][j0 + j], fa[1][i], tg[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[1][j0 + j], fa[0][i], tg[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) tg[j] = mfma_b16(fb[0][j0 + j], fa[0][i], tg[j]);
      if (g > 0) flush(g - 1);
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (!SM && NG - NS + s == g && (full || kt + 2 < nk))
          split_slot((kt + 2) % D, s, (kt + 2) * kSBK, !full && kt + 2 >= nfull);
      if (full) {
#pragma unroll
        for (int m = 0; m < 12; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
        }
      }
    }
    flush(NG - 1);
  };
  // LDS only: the loads in flight stay in flight
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stage = [&](int kt, int buf, bool full) __attribute__((always_inline)) {
    stage_mem(kt, buf, full);
    if constexpr (PP) barrier();
    stage_mma(kt, full);
    barrier();
  };

  if (nk > 0) {
    auto load = [&](int st, int set) __attribute__((always_inline)) {
      if (st < nk) {
#pragma unroll
        for (int s = 0; s < NS; ++s) load_slot(raw[set][s], s, st * kSBK, st >= nfull);
      }
    };
    auto split = [&](int st, int set) __attribute__((always_inline)) {
      if (st < nk) {
#pragma unroll
        for (int s = 0; s < NS; ++s) split_slot(set, s, st * kSBK, st >= nfull);
      }
    };
    load(0, 0);
    if (D == 2) load(1, 1);
    split(0, 0);
#pragma unroll
    for (int s = 0; s < NS; ++s) write_slot(s, 0);
    load(D, 0);
    if (!SM) split(1, D - 1);
    barrier();
    if (PP && wave >= NW / 2) barrier();
    int kt = 0;
    for (; kt + 2 + D < nfull; kt += 2) {
      stage(kt, 0, true);
      stage(kt + 1, 1, true);
    }
    for (; kt < nk; kt += 2) {
      stage(kt, 0, false);
      if (kt + 1 < nk) stage(kt + 1, 1, false);
    }
    if (PP && wave < NW / 2) barrier();
  }

  // the finished tile into LDS, the outputs the split cannot give replaced
  // there, then whole rows to memory
  float *ct = (float *)lds;
  float vmin = __builtin_inff(), vmax = 0.0f;  // of this lane's output magnitudes
#pragma unroll
  for (int i = 0; i < TMF; ++i)
#pragma unroll
    for (int j = 0; j < TNF; ++j) {
      const f32x4 v = acc[i][j];
#pragma unroll
      for (int r = 0; r < 4; ++r) vmin = fminf(vmin, fabsf(v[r]));
      vmax = absmax3(absmax3(vmax, v[0], v[1]), v[2], v[3]);
      *(f32x4 *)(ct + (wm * WTM + i * 16 + fr) * T::LDT + wn * WTN + j * 16 + 4 * fo) = v;
    }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const bool kf = s < SA ? AKF : BKF && !CONV;
#pragma unroll
    for (int h = 0; h < (kf ? 2 : 1); ++h)
      atomicMax((s < SA ? rma : rmb) + slot_row(kf, s < SA ? s : s - SA, h),
                __float_as_uint(rmax[s][h]));
  }
  __syncthreads();
  // Whether an element loses bits is not tracked in the K loop (there it cost the
  // 4096-wide training step 5 %, 32 x 64 x 56^2 -> 64, 3 x 3 4 %; 1.5 % and 2 % with
  // zeros taken for such elements): outputs so small that it could matter are rare (a
  // sum of N(0,1) products cancels to zero once in 4e7) and say where to look.
  uint32_t mine = __builtin_amdgcn_ballot_w64(!is_finite(vmax)) ? 1 : 0;
  const float vlim = __uint_as_float(wave_max_mag(max(lane < WTM ? rma[wm * WTM + lane] : 0u,
                                                      lane < WTN ? rmb[wn * WTN + lane] : 0u))) *
                     kExactMin * (float)K;
  if (__builtin_amdgcn_ballot_w64(vmin < vlim)) {
    // the row and column of up to four such outputs are looked through by the
    // wave; with more the tile's operands are read again
    int count = 0, at = 0;
#pragma unroll 4
    for (int b = 0; b < TMF * TNF; ++b) {
      const int ml = wm * WTM + b / TNF * 16 + fr, nl = wn * WTN + b % TNF * 16 + 4 * fo;
      const f32x4 v = *(const f32x4 *)(ct + ml * T::LDT + nl);
      const float a = fminf(fminf(fabsf(v[0]), fabsf(v[1])), fminf(fabsf(v[2]), fabsf(v[3])));
      if (!__builtin_amdgcn_ballot_w64(a < vlim)) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool small =
            is_finite(v[r]) && split_fails(v[r], rma[ml], rmb[nl + r], true, true, K);
        count += small;
        at = small ? 4 * b + r : at;
      }
    }
    uint64_t left = __builtin_amdgcn_ballot_w64(count > 0);
    uint32_t found = 0;
    if (__builtin_popcountll(left) > 4 || __builtin_amdgcn_ballot_w64(count > 1))
      found = 2;
    else
      for (; left; left &= left - 1) {
        const int l = __builtin_ctzll(left), b = __builtin_amdgcn_readlane(at, l);
        found |= lossy_pair<CONV>(p, A, B, m0 + wm * WTM + b / (4 * TNF) * 16 + (l & 15),
                                  n0 + wn * WTN + b / 4 % TNF * 16 + 4 * (l >> 4) + b % 4, lane);
      }
    if (found & 4) lossy[0] = 1;
    if (found & 8) lossy[1] = 1;
    mine |= found;
  }
  if (mine && lane == 0) atomicOr(again, mine);
  __syncthreads();
  const uint32_t todo = __builtin_amdgcn_readfirstlane(*again);
  if (todo) {
    if (todo & 2) {
      constexpr int U = 4;  // stages in flight
      uint32_t amin = ~0u, bmin = ~0u;
      for (int kt = 0; kt < nk; kt += U) {
        float x[U][NS][8];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const int st = kt + u < nk ? kt + u : nk - 1;
            load_slot(x[u][s], s, st * kSBK, st >= nfull);
          }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
              uint32_t &mn = s < SA ? amin : bmin;
              mn = absmin3(mn, x[u][s][e], x[u][s][e + 1]);
            }
      }
      if (is_lossy(amin)) lossy[0] = 1;
      if (is_lossy(bmin)) lossy[1] = 1;
      __syncthreads();
    }
    const bool la = lossy[0], lb = lossy[1];
    if ((todo & 1) || la || lb) {
      // the tile on the native fp32 MFMA, 32 k at a time through LDS, by the waves
      // that hold such an output: 4096^3 with all of A tiny 1891 us (the native
      // kernels 1327; 16 x 16 blocks straight from memory, wave by wave, 14640), with
      // one infinity in B 897 (1291)
      bool fails = false;
#pragma unroll 1
      for (int b = 0; b < TMF * TNF; ++b) {
        const int ml = wm * WTM + b / TNF * 16 + fr, nl = wn * WTN + b % TNF * 16 + 4 * fo;
        const f32x4 v = *(const f32x4 *)(ct + ml * T::LDT + nl);
#pragma unroll
        for (int r = 0; r < 4; ++r) fails |= split_fails(v[r], rma[ml], rmb[nl + r], la, lb, K);
      }
      const bool need = __builtin_amdgcn_ballot_w64(fails) != 0;
      f32x4 nat[TMF][TNF];
#pragma unroll
      for (int i = 0; i < TMF; ++i)
#pragma unroll
        for (int j = 0; j < TNF; ++j) nat[i][j] = zero;
      float x[NS][8];
#pragma unroll
      for (int s = 0; s < NS; ++s) load_slot(x[s], s, 0, nfull == 0);
      for (int kt = 0; kt < nk; ++kt) {
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (kt >= nfull) clear_past_k(x[s], s, kt * kSBK);
          const bool kf = s < SA ? AKF : BKF && !CONV;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int r = (s < SA ? 0 : TM) + slot_row(kf, s < SA ? s : s - SA, h);
            *(f32x4 *)(ct + r * T::LDN + (kf ? 4 * c4 : 8 * uoct + 4 * h)) =
                f32x4{x[s][4 * h], x[s][4 * h + 1], x[s][4 * h + 2], x[s][4 * h + 3]};
          }
        }
        __syncthreads();
        if (kt + 1 < nk) {
#pragma unroll
          for (int s = 0; s < NS; ++s) load_slot(x[s], s, (kt + 1) * kSBK, kt + 1 >= nfull);
        }
        if (!need) continue;
        const float *na = ct + (wm * WTM + fr) * T::LDN + fo;
        const float *nb = ct + (TM + wn * WTN + fr) * T::LDN + fo;
#pragma unroll
        for (int q = 0; q < kSBK; q += 4) {
          float a[TMF], b[TNF];
#pragma unroll
          for (int i = 0; i < TMF; ++i) a[i] = na[i * 16 * T::LDN + q];
#pragma unroll
          for (int j = 0; j < TNF; ++j) b[j] = nb[j * 16 * T::LDN + q];
#pragma unroll
          for (int i = 0; i < TMF; ++i)
#pragma unroll
            for (int j = 0; j < TNF; ++j)
              nat[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], nat[i][j], 0, 0, 0);
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TMF; ++i)
#pragma unroll
        for (int j = 0; j < TNF; ++j) {
          const int ml = wm * WTM + i * 16 + fr, nl = wn * WTN + j * 16 + 4 * fo;
          f32x4 v = acc[i][j];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (split_fails(v[r], rma[ml], rmb[nl + r], la, lb, K)) v[r] = nat[i][j][r];
          *(f32x4 *)(ct + ml * T::LDT + nl) = v;
        }
      __syncthreads();
    }
  }
#pragma unroll 2
  for (int idx = tid; idx < TM * (TN / 4); idx += NT) {
    const int r = idx / (TN / 4), c = idx % (TN / 4) * 4;
    if (m0 + r < p.M && n0 + c < p.N)
      store4_f32<CONV>(p, C, m0 + r, n0 + c, *(const f32x4 *)(ct + r * T::LDT + c));
  }
}

// ---------------------------------------------------------------- small problems
// TB x TB outputs per workgroup, the blocks of 32 k dealt over its NW waves,
// fragments loaded straight from memory (no operand staging): for products
// with too few tiles to fill the chip, which wait on load latency.  Each wave writes
// its blocks' t to LDS and the owners add them in k order, so the sums are
// those of the tiles.
template <int TB, int NW, bool AKF, bool BKF, bool CONV>
__global__ __launch_bounds__(NW * 64) void gemm_f32s_direct_kernel(F32Args p) {
  constexpr int NB = TB / 16, U = 2, NSLOT = NW * U, LDT = TB + 4;
  constexpr int OWN = TB * TB / 4;  // threads that own 4 outputs
  static_assert(OWN <= NW * 64 && NB * NB <= NW, "owners");
  __shared__ __align__(16) float part[NSLOT][TB][LDT];
  __shared__ uint32_t rma[TB], rmb[TB], lossy[2];

  const float *A, *B;
  float *C;
  batch_offsets(p, A, B, C);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = (p.N + TB - 1) / TB;
  const int m0 = (int)(blockIdx.x / tiles_n) * TB, n0 = (int)(blockIdx.x % tiles_n) * TB;
  const int K = p.K;
  const int nkb = (int)(((unsigned)K + kSBK - 1) / kSBK);
  const int fr = lane & 15, fo = lane >> 4;
  if (tid < TB) rma[tid] = rmb[tid] = 0;
  if (tid < 2) lossy[tid] = 0;

  const float *pa[NB], *pb[NB];
  int iy0[NB], ix0[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int m = m0 + 16 * i + fr < p.M ? m0 + 16 * i + fr : p.M - 1;
    const int n = n0 + 16 * i + fr < p.N ? n0 + 16 * i + fr : p.N - 1;
    pa[i] = A + (int64_t)m * p.sAm;
    pb[i] = B;
    if constexpr (CONV) conv_pixel(p.cv, n, iy0[i], ix0[i]);
    else pb[i] = B + (int64_t)n * p.sBn;
  }
  auto fetch = [&](const float *q, bool kf, int64_t sk, int k0, float (&x)[8]) {
    if ((unsigned)k0 + 8 <= (unsigned)K) {  // k0 + 8 can be 2^31
      if (kf) {
        const f32x4u u = *(const f32x4u *)(q + k0), v = *(const f32x4u *)(q + k0 + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[i] = u[i];
          x[4 + i] = v[i];
        }
      } else {
        const float *q0 = q + (int64_t)k0 * sk;
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = q0[i * sk];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        x[i] = k0 + i < K ? q[(int64_t)(k0 + i) * (kf ? 1 : sk)] : 0.0f;
    }
  };
  auto fetch_conv = [&](int i, int k0, float (&x)[8]) {
    const int khw = p.cv.kH * p.cv.kW;
    int c = k0 / khw, ky = (k0 - c * khw) / p.cv.kW, kx = k0 - c * khw - ky * p.cv.kW;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = k0 + e < K ? conv_tap(B, p.cv, c, ky, kx, iy0[i], ix0[i]) : 0.0f;
      if (++kx == p.cv.kW) {
        kx = 0;
        if (++ky == p.cv.kH) {
          ky = 0;
          ++c;
        }
      }
    }
  };
  typedef float Blocks[U][NB][8];
  Blocks xa, xb;
  float mxa[NB], mxb[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) mxa[i] = mxb[i] = 0.0f;
  auto load = [&](int r0, Blocks &xa, Blocks &xb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kb = r0 + u * NW + wave;
      if (kb >= nkb) break;
      const int k0 = kb * kSBK + 8 * fo;
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        fetch(pa[i], AKF, p.sAk, k0, xa[u][i]);
        if constexpr (CONV) fetch_conv(i, k0, xb[u][i]);
        else fetch(pb[i], BKF, p.sBk, k0, xb[u][i]);
      }
    }
  };
  const int orow = tid / (TB / 4), ocol = tid % (TB / 4) * 4;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  load(0, xa, xb);
  for (int r0 = 0; r0 < nkb; r0 += NSLOT) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int slot = u * NW + wave;
      if (r0 + slot >= nkb) break;
      u32x4 a[NB][3], b[NB][3];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          mxa[i] = absmax3(mxa[i], xa[u][i][e], xa[u][i][e + 1]);
          mxb[i] = absmax3(mxb[i], xb[u][i][e], xb[u][i][e + 1]);
        }
        split8(xa[u][i], a[i][0], a[i][1], a[i][2]);
        split8(xb[u][i], b[i][0], b[i][1], b[i][2]);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          f32x4 t = mfma_b16(b[j][0], a[i][2], zero);
          t = mfma_b16(b[j][2], a[i][0], t);
          t = mfma_b16(b[j][1], a[i][1], t);
          t = mfma_b16(b[j][0], a[i][1], t);
          t = mfma_b16(b[j][1], a[i][0], t);
          t = mfma_b16(b[j][0], a[i][0], t);
          *(f32x4 *)&part[slot][16 * i + fr][16 * j + 4 * fo] = t;
        }
    }
    if (r0 + NSLOT < nkb) load(r0 + NSLOT, xa, xb);
    __syncthreads();
    if (tid < OWN) {
      const int cnt = nkb - r0 < NSLOT ? nkb - r0 : NSLOT;
#pragma unroll 8
      for (int s = 0; s < cnt; ++s) acc += *(const f32x4 *)&part[s][orow][ocol];
    }
    __syncthreads();
  }
  // largest magnitudes of the tile's rows
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    atomicMax(&rma[16 * i + fr], __float_as_uint(mxa[i]));
    atomicMax(&rmb[16 * i + fr], __float_as_uint(mxb[i]));
  }
  __syncthreads();
  bool redo[4] = {false, false, false, false};
  auto failing = [&](bool la, bool lb) __attribute__((always_inline)) {
    if (tid < OWN) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        redo[r] = split_fails(acc[r], rma[orow], rmb[ocol + r], la, lb, K);
    }
    return __syncthreads_or(redo[0] || redo[1] || redo[2] || redo[3]);
  };
  bool small = false;
  auto any = failing(true, true);
#pragma unroll
  for (int r = 0; r < 4; ++r) small |= redo[r] && is_finite(acc[r]);
  if (any && __syncthreads_or(small)) {
    // the operands again, to see whether an element loses bits
    uint32_t amin = ~0u, bmin = ~0u;
    for (int r0 = 0; r0 < nkb; r0 += NSLOT) {
      Blocks ya, yb;
      load(r0, ya, yb);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (r0 + u * NW + wave >= nkb) break;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            amin = absmin3(amin, ya[u][i][e], ya[u][i][e + 1]);
            bmin = absmin3(bmin, yb[u][i][e], yb[u][i][e + 1]);
          }
      }
    }
    if (is_lossy(amin)) lossy[0] = 1;
    if (is_lossy(bmin)) lossy[1] = 1;
    __syncthreads();
    any = failing(lossy[0], lossy[1]);
  }
  if (any) {
    if (wave < NB * NB) {
      const int i = wave / NB, j = wave % NB;
      *(f32x4 *)&part[0][16 * i + fr][16 * j + 4 * fo] =
          exact_block<CONV>(p, A, B, m0 + 16 * i, n0 + 16 * j, lane);
    }
    __syncthreads();
    if (tid < OWN) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (redo[r]) acc[r] = part[0][orow][ocol + r];
    }
  }
  if (tid < OWN && m0 + orow < p.M && n0 + ocol < p.N)
    store4_f32<CONV>(p, C, m0 + orow, n0 + ocol, acc);
}

// ---------------------------------------------------------------- launch
constexpr int64_t kMaxGridY = 65535;

template <int TM, int TN, int WGM, int WGN, int D, bool AKF, bool BKF, bool CONV, bool ANY = false>
static hipError_t launch_tile_s(F32Args p, int64_t batches, hipStream_t stream) {
  using T = TileS<TM, TN, WGM, WGN>;
  const auto kernel = gemm_f32s_kernel<TM, TN, WGM, WGN, D, AKF, BKF, CONV, ANY>;
  static std::atomic<uint64_t> attr_set{0};
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const uint64_t bit = dev < 64 ? (uint64_t)1 << dev : 0;
  if (T::LDS > 65536 && (!bit || !(attr_set.load(std::memory_order_acquire) & bit))) {
    if (hipError_t e = hipFuncSetAttribute(
            (const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
        e != hipSuccess)
      return e;
    attr_set.fetch_or(bit, std::memory_order_release);
  }
  const int64_t tiles = ((p.M + (int64_t)TM - 1) / TM) * ((p.N + (int64_t)TN - 1) / TN);
  if (tiles > INT32_MAX) return hipErrorInvalidValue;  // grid.x limit
  for (int64_t b0 = 0; b0 < batches; b0 += kMaxGridY) {
    const int64_t nb = batches - b0 < kMaxGridY ? batches - b0 : kMaxGridY;
    p.batch0 = b0;
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles, (unsigned)nb), dim3(T::NT), T::LDS, stream,
                       p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int TB, int NW, bool AKF, bool BKF, bool CONV>
static hipError_t launch_direct_s(F32Args p, int64_t batches, hipStream_t stream) {
  const int64_t tiles = ((p.M + (int64_t)TB - 1) / TB) * ((p.N + (int64_t)TB - 1) / TB);
  if (tiles > INT32_MAX) return hipErrorInvalidValue;
  for (int64_t b0 = 0; b0 < batches; b0 += kMaxGridY) {
    const int64_t nb = batches - b0 < kMaxGridY ? batches - b0 : kMaxGridY;
    p.batch0 = b0;
    hipLaunchKernelGGL((gemm_f32s_direct_kernel<TB, NW, AKF, BKF, CONV>),
                       dim3((unsigned)tiles, (unsigned)nb), dim3(NW * 64), 0, stream, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Launches one configuration for the layouts that the strides say.
#define MJ_F32S_LAYOUTS(FN, ...)                                                   \
  (akf ? (bkf ? FN<__VA_ARGS__, true, true, false>(p, batches, stream)             \
              : FN<__VA_ARGS__, true, false, false>(p, batches, stream))           \
       : (bkf ? FN<__VA_ARGS__, false, true, false>(p, batches, stream)            \
              : FN<__VA_ARGS__, false, false, false>(p, batches, stream)))

// The tiles hold a row's byte offset from the tile's first row in 32 bits.
constexpr int64_t kMaxRowStride = (int64_t)1 << 21;

enum F32Kernel { F32_256x128, F32_128x128, F32_64x64, F32_DIRECT32, F32_DIRECT16,
                 F32_DIRECT16_W16 };

// Which kernel takes an M x N x K product of `batches` matrices: the smallest
// estimated time.  A tile kernel deals its tiles over the 256 CUs in rounds of
// a fixed part (first loads, output) and a time per 32-deep stage; the direct
// kernels run ceil(stages / (2 NW)) rounds of loads per workgroup, bound by
// latency when few share a CU and by the splits when many do.  The constants
// (us) are fits to MI355X times of N(0,1) operands, e.g. (256 x 128 / 128 x 128
// / 64 x 64 tiles) 4096^3 644 / 700 / -, 2048^3 137 / 100 / 126, 1024^3 73 / 44
// / 25; (64 x 64 / direct 32 / direct 16 of 4 and of 16 waves) 512 x 512 x 4096
// 73 / 45 / 64 / 72, 64 x 4096 x 1024 23 / 15 / 20 / 27, 1 x 4096 x 4096 87 / 38
// / 25 / 21, 256^3 9.7 / 6.7 / 5.0 / 4.9, 32 x (300 x 517 x 257) 40 / 64 / 85 /
// 230.
static F32Kernel plan_f32s(int64_t M, int64_t N, int64_t K, int64_t batches) {
  const double nk = (double)((K + kSBK - 1) / kSBK);
  auto tiles = [&](int tm, int tn) {
    return (double)((M + tm - 1) / tm) * (double)((N + tn - 1) / tn) * (double)batches;
  };
  auto tile_us = [&](int tm, int tn, double fixed, double stage) {
    return std::ceil(tiles(tm, tn) / 256) * (fixed + nk * stage);
  };
  auto direct_us = [&](int tb, int nw, double wait, double work) {
    return std::ceil(nk / (2 * nw)) * (wait + work * tiles(tb, tb) / 256);
  };
  const double us[] = {
      tile_us(256, 128, 14, 2.45),
      tile_us(128, 128, 9, 1.35),
      tile_us(64, 64, 2.5, 0.45) + (tiles(64, 64) <= 256 ? 0.12 * nk : 0),
      direct_us(32, 4, 1.3, 1.6),
      direct_us(16, 4, 0.8, 0.9),
      direct_us(16, 16, 1.0, 4.3),
  };
  int best = 0;
  for (int i = 1; i < 6; ++i)
    if (us[i] < us[best]) best = i;
  return (F32Kernel)best;
}

static F32Kernel choose_f32s(const F32Args &p, int64_t batches) {
  const F32Kernel k = plan_f32s(p.M, p.N, p.K, batches);
  const bool far = (p.M > 1 && p.sAm >= kMaxRowStride) || (p.N > 1 && p.sBn >= kMaxRowStride);
  return k <= F32_64x64 && far ? F32_DIRECT32 : k;
}

static const char *const kF32Names[] = {"split 256x128", "split 128x128", "split 64x64",
                                        "split direct 32", "split direct 16",
                                        "split direct 16, 16 waves"};

const char *f32s_kernel_name(const F32Args &p, int64_t batches) {
  return kF32Names[choose_f32s(p, batches)];
}

hipError_t launch_gemm_f32s(F32Args p, int64_t batches, hipStream_t stream) {
  // a single row (or k) has no row (k) stride
  if (p.M == 1) p.sAm = 1;
  if (p.N == 1) p.sBn = 1;
  if (p.K == 1) p.sAk = p.sBk = 1;
  const bool akf = p.sAk == 1, bkf = p.sBk == 1;
  switch (choose_f32s(p, batches)) {
    case F32_256x128: return MJ_F32S_LAYOUTS(launch_tile_s, 256, 128, 4, 2, 1);
    case F32_128x128: return MJ_F32S_LAYOUTS(launch_tile_s, 128, 128, 2, 4, 2);
    case F32_64x64: return MJ_F32S_LAYOUTS(launch_tile_s, 64, 64, 2, 2, 2);
    case F32_DIRECT32: return MJ_F32S_LAYOUTS(launch_direct_s, 32, 4);
    case F32_DIRECT16: return MJ_F32S_LAYOUTS(launch_direct_s, 16, 4);
    default: return MJ_F32S_LAYOUTS(launch_direct_s, 16, 16);
  }
}

// plan_f32s for a convolution, whose stages are bound by the gather, so that
// several workgroups on a CU gain more than a larger tile: times (us) fitted to
// MI355X, e.g. (64 x 64 / 128 x 128 tiles / direct 32) 32 x 64 x 56^2 -> 64, 3 x 3
// 75 / 153 / 150, -> 128 132 / 161 / -, 32 x 3 x 80^2 -> 128, 5 x 5 76 / 92 / 185,
// 32 x 128 x 28^2 -> 128, 3 x 3 84 / 75 / -, 32 x 16 x 100^2 -> 16, 3 x 3 71 / 133 /
// 109, 2 x 64 x 56^2 -> 64, 3 x 3 20.5 / 39 / 17.6.  64 x 64 tiles go three to a CU;
// what the full rounds leave over goes one, two or three.  The direct kernels have a
// fixed part, a load latency for each round of blocks and the work of all: 1 x 256 x
// 14^2 -> 256, 3 x 3 (direct 16 of 4 / of 16 waves) 27.4 / 16.1.
static F32Kernel plan_conv2d_f32s(int64_t M, int64_t N, int64_t K, int64_t images) {
  const double nk = (double)((K + kSBK - 1) / kSBK);
  auto tiles = [&](int tm, int tn) {
    return (double)((M + tm - 1) / tm) * (double)((N + tn - 1) / tn) * (double)images;
  };
  auto direct_us = [&](int tb, int nw, double fixed, double wait, double tile, double block) {
    return fixed + std::ceil(nk / (2 * nw)) * wait + (tile + nk * block) * tiles(tb, tb) / 256;
  };
  const double stage[] = {0.83, 1.18, 1.25};
  const double t64 = tiles(64, 64), full = std::floor(t64 / 768), rest = t64 - 768 * full;
  double us64 = full * (5.3 + nk * stage[2]);
  if (rest > 0) us64 += 5.3 + nk * stage[(int)std::ceil(rest / 256) - 1];
  const F32Kernel kernel[] = {F32_64x64, F32_128x128, F32_DIRECT32, F32_DIRECT16, F32_DIRECT16_W16};
  const double us[] = {us64, std::ceil(tiles(128, 128) / 256) * (7 + nk * 1.93),
                       direct_us(32, 4, 4.0, 1.2, 1.2, 0.34), direct_us(16, 4, 3.5, 1.8, 0.55, 0.115),
                       direct_us(16, 16, 3.5, 1.8, 0.7, 0.14)};
  int best = 0;
  for (int i = 1; i < 5; ++i)
    if (us[i] < us[best]) best = i;
  return kernel[best];
}

static F32Kernel choose_conv2d_f32s(const F32Args &p, int64_t images) {
  const F32Kernel k = plan_conv2d_f32s(p.M, p.N, p.K, images);
  // the tiles' gather has 31-bit byte offsets within an image (and the at most 32
  // channels that the last stage reaches past it), and a multiplied reciprocal for
  // k / (kH kW), exact for k below 2^26 + 64
  if (k <= F32_64x64 && (p.sAm >= kMaxRowStride || p.K > (1 << 26) ||
                         ((int64_t)p.channels + 32) * p.cv.H * p.cv.W >= ((int64_t)1 << 29)))
    return F32_DIRECT32;
  return k;
}

static bool any_taps(const F32Args &p) { return (int64_t)p.cv.kH * p.cv.kW > 64; }

const char *conv2d_f32s_kernel_name(const F32Args &p, int64_t images) {
  const F32Kernel k = choose_conv2d_f32s(p, images);
  if (k <= F32_64x64 && any_taps(p))
    return k == F32_64x64 ? "split 64x64, any taps" : "split 128x128, any taps";
  return kF32Names[k];
}

// Conv2d.forward with p.cv and p.channels set (A the weights, B the images).
hipError_t launch_conv2d_f32s(F32Args p, int64_t images, hipStream_t stream) {
  const bool any = any_taps(p);
  switch (choose_conv2d_f32s(p, images)) {
    case F32_128x128:
      return any ? launch_tile_s<128, 128, 2, 4, 2, true, false, true, true>(p, images, stream)
                 : launch_tile_s<128, 128, 2, 4, 2, true, false, true>(p, images, stream);
    case F32_64x64:
      return any ? launch_tile_s<64, 64, 2, 2, 2, true, false, true, true>(p, images, stream)
                 : launch_tile_s<64, 64, 2, 2, 2, true, false, true>(p, images, stream);
    case F32_DIRECT32: return launch_direct_s<32, 4, true, false, true>(p, images, stream);
    case F32_DIRECT16: return launch_direct_s<16, 4, true, false, true>(p, images, stream);
    default: return launch_direct_s<16, 16, true, false, true>(p, images, stream);
  }
}

}  // namespace mj
