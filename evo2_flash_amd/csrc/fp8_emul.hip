// Hopper fp8 "fast accumulation" GEMM, modelled exactly on gfx950 VALU.
//
// The released fp8 Evo 2 checkpoints were trained with Transformer Engine's
// forward fp8 GEMM on sm_90, whose tensor-core accumulator is not fp32.  Some
// layers of those checkpoints depend on its rounding (the FP8-surgery
// configs `hyena_fp8_emulated_layers` / `hyena_fp8_emulated_channels`,
// config.py:81-94), so the reference runs a software model of it
// (fp8_emul.py:1-24; arithmetic of fp8_emul_triton.py:46-76).  This file is
// that model as a HIP kernel.  For each group of 32 consecutive k, ascending:
//
//   e   = max( max_k e(a_k) + e(b_k), e(acc) ),   e(x) = floor(log2|x|)
//   s   = trunc(acc 2^(13-e)) 2^(e-13) + sum_k trunc(a_k b_k 2^(13-e)) 2^(e-13)
//   acc = s truncated to 13 fraction bits of its own exponent
//
// then out = bf16((acc * s_in) * s_w).  Every step is exact in fp32 (E4M3
// products are exact; aligned terms are integers below 2^21 times the ulp),
// so the kernel reproduces the reference bit for bit.
//
// Operands: a (N, K) e4m3 activation rows; b_t (K, M) bf16 holding E4M3
// values, K-major, the layout of the surgery checkpoints'
// `in_proj_emul_weight_t` (mixers.py:768-800).
//
// What bounds it: the per-product truncation depends on the output (its e), so
// the sum is no matrix product and costs VALU work per multiply-add.  A plain
// fp32 loop takes ~6.4 instructions each (exponent max 2, product, scale,
// truncate, accumulate; 300 x 4096 x 12288: 3.19 ms).  Here it is 1 VALU
// instruction per multiply-add, the rest on the matrix cores:
//  * e: A-side 2^(6 e(a)) and B-side 2^(6 e(b)) as bf16; an fp32 MFMA sum of
//    at most 32 of their products lies in [64^max, 32 * 64^max], so its
//    exponent field / 6 is the largest e(a) + e(b), and zeros drop out.
//  * truncation: packed f16 products under round-toward-zero.  f16's smallest
//    step is 2^-24, so with the product scaled by 2^(-11-e) the rounding of
//    v_pk_mul_f16 is exactly trunc(a b 2^(13-e)) (8 significant bits, so
//    nothing else rounds).  a enters as a 2^(-Ea-4) (Ea the largest e(a) of
//    the row's group: exact, at least 2^-24), b as b 2^-5 (exact) times
//    2^(Ea-e-2) per output.  That last product truncates b's low bits only
//    where e(b) < e - Ea - 14, so e(a) + e(b) < e - 14, and the term is zero
//    either way.
//  * the sum: one f16 MFMA per eight products of a lane, the truncated terms
//    as operand A against a constant 0 / 2^15 operand that routes each
//    lane group's sum to its own column of the result (f16 subnormals are kept,
//    and every partial sum is a multiple of 2^-24 below 2^-2: exact).
// Groups it cannot take -- a weight that is not an E4M3 value, a NaN, or an
// output whose e is 14 or more below Ea -- go through the plain arithmetic
// (slow_group), the same bits.
#include "common.h"

#pragma clang fp contract(off)

namespace evo2 {

constexpr int FA_G = 32;    // accumulation group (k)
constexpr int FA_F = 13;    // fraction bits kept
constexpr int FA_WAVES = 4; // waves per workgroup, 16 rows each

struct FastAccArgs {
  const uint8_t *a; int64_t sa;    // (N, K) e4m3 rows, row stride (bytes)
  const bf16_t *b; int64_t sb;     // (K, M) bf16 E4M3 values, row stride (elements)
  const float *sx, *sw;            // (1,) dequantisation scales
  void *out; int64_t so;           // (N, M) bf16 (scaled) or fp32 (raw accumulator)
  int out_f32;
  int N, M, K;
};

// OCP e4m3fn byte -> fp32 (exact): bias 7, subnormals m * 2^-9, S.1111.111 NaN.
__device__ __forceinline__ float e4m3_to_f32(uint32_t x) {
  const uint32_t s = (x >> 7) & 1, e = (x >> 3) & 15, m = x & 7;
  if (e == 15 && m == 7) return __uint_as_float(0x7fc00000u);
  float v;
  if (e == 0) v = static_cast<float>(m) * 0.001953125f;  // m * 2^-9
  else v = __uint_as_float(((e + 120u) << 23) | (m << 20));
  return s ? -v : v;
}

// floor(log2|x|) from the exponent field; a very negative sentinel for 0
// (the reference's -100000; a subnormal reads -127 as there).
__device__ __forceinline__ int exp_floor(float x) {
  const int e = static_cast<int>((__float_as_uint(x) >> 23) & 0xFF) - 127;
  return x == 0.0f ? -100000 : e;
}

// 2^e with e clamped to [-126, 127], as the reference clamps.
__device__ __forceinline__ float pow2i(int e) {
  e = min(max(e, -126), 127);
  return __uint_as_float(static_cast<uint32_t>(e + 127) << 23);
}

typedef _Float16 fa_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 fa_h8 __attribute__((ext_vector_type(8)));
typedef __bf16 fa_b8 __attribute__((ext_vector_type(8)));
typedef uint16_t fa_u2 __attribute__((ext_vector_type(2)));
typedef int16_t fa_i2 __attribute__((ext_vector_type(2)));
typedef float fa_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t fa_w4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ fa_h2 as_h2(uint32_t w) { return __builtin_bit_cast(fa_h2, w); }
__device__ __forceinline__ uint32_t as_u32(fa_h2 h) { return __builtin_bit_cast(uint32_t, h); }

// One group of one output by the plain arithmetic.
__device__ __forceinline__ float slow_group(const uint8_t *a, const bf16_t *b, int64_t sb, float acc) {
  int e = exp_floor(acc);
#pragma unroll 1
  for (int kk = 0; kk < FA_G; ++kk)
    e = max(e, exp_floor(e4m3_to_f32(a[kk])) + exp_floor(bf2f(b[kk * sb])));
  const float ulp = pow2i(e - FA_F), inv = pow2i(FA_F - e);
  float s = truncf(acc * inv) * ulp;
#pragma unroll 1
  for (int kk = 0; kk < FA_G; ++kk)
    s = s + truncf((e4m3_to_f32(a[kk]) * bf2f(b[kk * sb])) * inv) * ulp;
  const int es = exp_floor(s);
  return s == 0.0f ? s : truncf(s * pow2i(FA_F - es)) * pow2i(es - FA_F);
}

// Largest e(a) + e(b) of an output from its max product, 2^(6 e - 1) times 1
// to 32: exponent field 126 + 6 e + {0 .. 5} -> e + 127 (a floor division by
// 6); 106, below any e, for no product at all.
__device__ __forceinline__ int product_e(float d) {
  return static_cast<int>(__umul24(__float_as_uint(d) >> 23, 171u) + (106u << 10)) >> 10;
}

__device__ __forceinline__ int field_of(float x) { return (__float_as_uint(x) >> 23) & 0xff; }

// A workgroup owns 16 rows per wave and 64 columns.  For its packed
// products a lane holds column `lane`; the accumulators,
// and everything done once per output, are in the layout the sums arrive in:
// tile R, lane (g, j = 4 rho + c), element v is row 4 R + rho, column
// 16 c + 4 g + v.  The scales 2^(Ea-e-2) cross over through LDS.
//
// Per group of 32 k the workgroup stages b 2^-5 (f16) and 2^(6 e(b)) (bf16) by
// column, a 2^(-Ea-4) and 2^(6 e(a)) by row; the next group's raw operands load
// while this one is computed.  Measured (300 x 4096 x 12288, us): 1153; with
// two column sets a wave 1180, one and two waves a workgroup 1473 and 1465,
// eight 1663 (its last row block mostly empty), two stages 1215.  One row:
// 276 (the plain loop 1606: 48 workgroups).
struct FaStage {
  fa_w4 b0[4][64];  // k octet, column
  fa_w4 bx[4][64];
  fa_w4 a0[16 * FA_WAVES][4];  // row, k octet
  fa_w4 ax[16 * FA_WAVES][4];
  int elow[16 * FA_WAVES];     // Ea - 14, biased as an fp32 exponent field
};

__global__ __launch_bounds__(64 * FA_WAVES, 2) void fast_accum_kernel(FastAccArgs p, int gx, int gy) {
  __shared__ __align__(16) FaStage stage;
  __shared__ __align__(16) fa_w4 zero[64];
  // scales of a wave: [v][4 c + g][rho] of four f16 (R), v padded apart
  constexpr int SV = 512 + 16;  // bytes per v
  __shared__ __align__(16) uint8_t sig[FA_WAVES][4096];  // (or a wave's accumulators)
  __shared__ int not_e4m3;      // set once an operand is no E4M3 value: slow from there on

  // workgroups that share columns run back to back on one XCD (workgroup L on
  // XCD L % 8): its L2 then serves the weight to the other row blocks
  const int j8 = static_cast<int>(blockIdx.x) >> 3;
  const int by = j8 % gy, bx = (j8 / gy) * 8 + (static_cast<int>(blockIdx.x) & 7);
  if (bx >= gx) return;  // uniform: grid padding
  // f16 arithmetic rounds toward zero in this kernel (the truncation above);
  // every other f16 operation here is exact
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3" ::: "memory");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = bx * 64, n0 = by * 16 * FA_WAVES;
  const int g = lane >> 4, c = lane & 3, rho = (lane >> 2) & 3;
  const int nr = min(16, p.N - n0 - 16 * wave);  // this wave's rows (may be <= 0)

  // staging roles: the lane's column and the wave's k octet of b; row and octet of a
  const int srow = tid >> 2, soct = tid & 3;
  const bool bok = m0 + lane < p.M, aok = n0 + srow < p.N;
  const bf16_t *bsrc = p.b + (int64_t)(8 * wave) * p.sb + (bok ? m0 + lane : 0);
  const uint8_t *asrc = p.a + (int64_t)(aok ? n0 + srow : 0) * p.sa + 8 * soct;
  const bool a8 = (p.sa & 7) == 0 && (reinterpret_cast<uintptr_t>(p.a) & 7) == 0;
  uint32_t braw[8];
  uint2 araw;
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) braw[i] = bok ? bsrc[(int64_t)(k0 + i) * p.sb] : 0;
    if (a8) {
      araw = *reinterpret_cast<const uint2 *>(asrc + k0);
    } else {
      uint32_t w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = asrc[k0 + i];
      araw = make_uint2(w[0] | (w[1] << 8) | (w[2] << 16) | (w[3] << 24),
                        w[4] | (w[5] << 8) | (w[6] << 16) | (w[7] << 24));
    }
    if (!aok) araw = make_uint2(0, 0);
  };
  auto put = [&]() __attribute__((always_inline)) {
    // weights: E4M3 values are 0 or have an exponent in [-9, 8] (field 118 ..
    // 135) and no bits below the third mantissa bit
    uint32_t low = 0;
    fa_u2 mn = {0xffff, 0xffff}, mx = {0, 0};
    fa_w4 h, x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = braw[2 * i] | (braw[2 * i + 1] << 16);
      low |= w;
      const fa_u2 m = __builtin_bit_cast(fa_u2, w & 0x7fff7fffu);
      mn = __builtin_elementwise_min(mn, static_cast<fa_u2>(m - fa_u2{1, 1}));
      mx = __builtin_elementwise_max(mx, m);
      // 2^(6 e(b) + 36): exponent field 6 E - 599, 0 for a zero
      fa_i2 f = __builtin_bit_cast(fa_i2, static_cast<fa_u2>(m >> fa_u2{7, 7}));
      f = __builtin_elementwise_max(static_cast<fa_i2>(f * fa_i2{6, 6} - fa_i2{599, 599}), fa_i2{0, 0});
      x[i] = __builtin_bit_cast(uint32_t, static_cast<fa_u2>(__builtin_bit_cast(fa_u2, f) << fa_u2{7, 7}));
      const fa_h2 v = __builtin_bit_cast(
          fa_h2, __builtin_amdgcn_cvt_pkrtz(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)));
      h[i] = as_u32(v * fa_h2{(_Float16)0.03125f, (_Float16)0.03125f});
    }
    stage.b0[wave][lane] = h;
    stage.bx[wave][lane] = x;
    bool bad = (low & 0x000f000fu) != 0 || mn.x < (118 << 7) - 1 || mn.y < (118 << 7) - 1 ||
          mx.x > ((135 << 7) | 0x7f) || mx.y > ((135 << 7) | 0x7f);
    // activations: byte << 7 is the f16 of a 2^-8 (subnormals too)
    uint32_t hv[4];
    fa_u2 am = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t two = (i & 1 ? (i & 2 ? araw.y : araw.x) >> 16 : (i & 2 ? araw.y : araw.x));
      const uint32_t w = ((two & 0xffu) << 8) | ((two & 0xff00u) << 16);
      hv[i] = ((w >> 1) & 0x3f803f80u) | (w & 0x80008000u);
      am = __builtin_elementwise_max(am, __builtin_bit_cast(fa_u2, hv[i] & 0x7fff7fffu));
    }
    int top = max(static_cast<int>(am.x), static_cast<int>(am.y));
    top = max(top, __shfl_xor(top, 1));
    top = max(top, __shfl_xor(top, 2));  // over the row's 32 k (four lanes)
    bad = bad || top >= (0x7f << 7);     // a NaN
    const _Float16 tf = __builtin_bit_cast(_Float16, static_cast<uint16_t>(top)) * (_Float16)256.0f;
    const int E = max(__builtin_bit_cast(uint16_t, tf) >> 10, 6);  // Ea + 15; an all-zero group: -9
    const uint32_t sc1 = static_cast<uint32_t>(26 - E) << 10;      // 2^(-Ea-4)
    const fa_h2 sc = as_h2(sc1 | (sc1 << 16));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const fa_h2 v = as_h2(hv[i]) * fa_h2{(_Float16)256.0f, (_Float16)256.0f};  // a
      h[i] = as_u32(v * sc);
      // 2^(6 e(a) - 37): exponent field 6 (e + 15), 0 for a zero
      const fa_u2 f = __builtin_bit_cast(fa_u2, as_u32(v) & 0x7fff7fffu) >> fa_u2{10, 10};
      x[i] = __builtin_bit_cast(uint32_t, static_cast<fa_u2>(f * fa_u2{768, 768}));
    }
    stage.a0[srow][soct] = h;
    stage.ax[srow][soct] = x;
    if (soct == 0) stage.elow[srow] = E + 98;
    if (bad) not_e4m3 = 1;  // every writer stores the same value
  };

  float acc[4][4];  // R, v
#pragma unroll
  for (int R = 0; R < 4; ++R)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[R][v] = 0.0f;
  // routing operand of row rho: k-slots of lane group g go to column 4 rho + g
  fa_h8 route[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const _Float16 one = (lane & 15) == 4 * r + g ? (_Float16)32768.0f : (_Float16)0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) route[r][i] = one;
  }
  const bool own = c == g;  // this lane carries row exponents in the max product

  auto compute = [&](int k0) __attribute__((always_inline)) {
    // largest e(a) + e(b) of every output: 2^(6 e - 1 + {0 .. 5}) in d
    fa_f4 d[4];
    {
      fa_b8 bop[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) bop[q] = __builtin_bit_cast(fa_b8, stage.bx[q][lane]);
      // rows 4 R + rho at 64 R (in 16-byte units 16 R), or zeros
      const fa_w4 *ap = own ? &stage.ax[16 * wave + rho][0] : zero;
#pragma unroll
      for (int R = 0; R < 4; ++R) {
        d[R] = fa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const fa_b8 aop = __builtin_bit_cast(fa_b8, ap[16 * R + q]);
          d[R] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bop[q], aop, d[R], 0, 0, 0);
        }
      }
    }
    // e of each output (as an fp32 exponent field, at least elow), the scale
    // 2^(Ea - e - 2) = 2^(elow + 12 - e) and the aligned accumulator
    int nx[4][4];  // 140 - e: the shift 13 - e unbiased
    int xm = -1000;
    int el[4];
#pragma unroll
    for (int R = 0; R < 4; ++R) el[R] = stage.elow[16 * wave + 4 * R + rho];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      uint32_t sg[2];
#pragma unroll
      for (int R = 0; R < 4; ++R) {
        const int e = max(max(product_e(d[R][v]), field_of(acc[R][v])), el[R]);
        const int x = el[R] + 12 - e;
        xm = max(xm, x);
        const uint32_t sb16 = __builtin_bit_cast(
            uint16_t, static_cast<_Float16>(__builtin_amdgcn_ldexph((_Float16)1.0f, (short)x)));
        sg[R >> 1] = R & 1 ? sg[R >> 1] | (sb16 << 16) : sb16;
        nx[R][v] = 140 - e;
      }
      *reinterpret_cast<uint2 *>(&sig[wave][v * SV + (4 * c + g) * 32 + rho * 8]) =
          make_uint2(sg[0], sg[1]);
    }
    // the scales cross lanes of this wave only: LDS serves a wave in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    bool slow = not_e4m3 != 0;
    if (__any(xm >= 12)) {  // some e at its lower clamp: check whether the clamp changed it
      int bad = 0;
#pragma unroll
      for (int R = 0; R < 4; ++R)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          bad |= static_cast<int>(max(product_e(d[R][v]), field_of(acc[R][v])) < el[R]) &
                   static_cast<int>((__float_as_uint(d[R][v]) | __float_as_uint(acc[R][v])) != 0);
      slow = slow || __any(bad);
    }
    if (slow) {  // wave-uniform; through LDS, so that the loop need not be unrolled
      float *sp = reinterpret_cast<float *>(sig[wave]) + lane;
#pragma unroll
      for (int i = 0; i < 16; ++i) sp[64 * i] = acc[i >> 2][i & 3];
#pragma unroll 1
      for (int i = 0; i < 16; ++i) {
        const int n = min(n0 + 16 * wave + 4 * (i >> 2) + rho, p.N - 1);
        const int m = min(m0 + 16 * c + 4 * g + (i & 3), p.M - 1);
        sp[64 * i] = slow_group(p.a + (int64_t)n * p.sa + k0, p.b + (int64_t)k0 * p.sb + m, p.sb, sp[64 * i]);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i >> 2][i & 3] = sp[64 * i];
      return;
    }
    // the accumulators aligned to e, in units of 2^-9
    fa_f4 cin[4];
#pragma unroll
    for (int R = 0; R < 4; ++R)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        cin[R][v] = truncf(ldexpf(acc[R][v], nx[R][v])) * 0.001953125f;
    // the scales in column order: lane's column is v = lane & 3 of 4 c + g =
    // lane >> 2; rho's four rows R
    fa_h2 sv[4][2];
    const uint8_t *sp = &sig[wave][(lane & 3) * SV + (lane >> 2) * 32];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const fa_w4 w = *reinterpret_cast<const fa_w4 *>(sp + 16 * i);
#pragma unroll
      for (int t = 0; t < 4; ++t) sv[2 * i + (t >> 1)][t & 1] = as_h2(w[t]);
    }
    fa_w4 bv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bv[q] = stage.b0[q][lane];
    // Row by row: the next row's a is read ahead (rows past the input are
    // zeros in the stage), the scaled b of the row first, then its products.
    const fa_w4 *arow = &stage.a0[16 * wave][0];  // uniform: reads are broadcasts
    fa_w4 av[2][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) av[0][q] = arow[q];
#pragma unroll
    for (int R = 0; R < 4; ++R) {
      if (4 * R >= nr) break;  // wave-uniform: rows past the input
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int cur = r & 1;
        if (4 * R + r + 1 < 16) {
#pragma unroll
          for (int q = 0; q < 4; ++q) av[cur ^ 1][q] = arow[4 * (4 * R + r + 1) + q];
        }
        const _Float16 z = R & 1 ? sv[r][R >> 1].y : sv[r][R >> 1].x;
        const fa_h2 zz = {z, z};
        fa_h2 u[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < 4; ++i) u[q][i] = as_h2(bv[q][i]) * zz;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          fa_w4 t;
#pragma unroll
          for (int i = 0; i < 4; ++i) t[i] = as_u32(u[q][i] * as_h2(av[cur][q][i]));
          cin[R] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(fa_h8, t), route[r],
                                                             cin[R], 0, 0, 0);
        }
      }
    }
    // truncate to 13 fraction bits (drop the low 10 of fp32's 23) and rescale
#pragma unroll
    for (int R = 0; R < 4; ++R)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[R][v] =
            ldexpf(__uint_as_float(__float_as_uint(cin[R][v]) & 0xfffffc00u), 9 - nx[R][v]);
  };

  if (tid < 64) zero[tid] = fa_w4{0, 0, 0, 0};
  if (tid == 0) not_e4m3 = 0;
  __syncthreads();
  if (p.K > 0) {
    load(0);
    put();
  }
  __syncthreads();
  for (int k0 = 0; k0 < p.K; k0 += FA_G) {
    const bool more = k0 + FA_G < p.K;
    if (more) load(k0 + FA_G);
    if (nr > 0) compute(k0);
    __syncthreads();
    if (more) put();
    __syncthreads();
  }

  const float sx = p.out_f32 ? 1.0f : p.sx[0], sw = p.out_f32 ? 1.0f : p.sw[0];
#pragma unroll
  for (int R = 0; R < 4; ++R) {
    const int n = n0 + 16 * wave + 4 * R + rho;
    if (n >= p.N) continue;
    const int m = m0 + 16 * c + 4 * g;
    if (p.out_f32) {
      float *o = static_cast<float *>(p.out) + (int64_t)n * p.so + m;
      if (m + 4 <= p.M && (reinterpret_cast<uintptr_t>(o) & 15) == 0) {
        *reinterpret_cast<float4 *>(o) = make_float4(acc[R][0], acc[R][1], acc[R][2], acc[R][3]);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (m + v < p.M) o[v] = acc[R][v];
      }
    } else {
      bf16_t *o = static_cast<bf16_t *>(p.out) + (int64_t)n * p.so + m;
      float f[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) f[v] = (acc[R][v] * sx) * sw;
      if (m + 4 <= p.M && (reinterpret_cast<uintptr_t>(o) & 7) == 0) {
        *reinterpret_cast<uint2 *>(o) = make_uint2(pack_bf(f[0], f[1]), pack_bf(f[2], f[3]));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (m + v < p.M) o[v] = f2bf(f[v]);
      }
    }
  }
}

}  // namespace evo2

using namespace evo2;

extern "C" int evo2_fp8_fast_accum_gemm(const void *a8, int64_t sa, const void *b_t, int64_t sb,
                                        const float *input_scale, const float *weight_scale,
                                        void *out, int64_t so, int32_t out_f32, int64_t N,
                                        int64_t M, int64_t K, void *stream) {
  if (N < 0 || M < 0 || K < 0 || N > (int64_t(1) << 31) - 1 || M > (int64_t(1) << 31) - 1 ||
      K > (int64_t(1) << 31) - 1)
    return fail(EVO2_ERR_INVALID, "fp8_fast_accum_gemm: bad sizes N=%lld M=%lld K=%lld",
                (long long)N, (long long)M, (long long)K);
  if (K % FA_G)
    return fail(EVO2_ERR_INVALID, "fp8_fast_accum_gemm: K=%lld is not a multiple of %d",
                (long long)K, FA_G);
  if (N == 0 || M == 0) return EVO2_OK;
  if (!a8 || !b_t || !out || (!out_f32 && (!input_scale || !weight_scale)))
    return fail(EVO2_ERR_INVALID, "fp8_fast_accum_gemm: null pointer argument");
  if (sa < K || sb < M || so < M)
    return fail(EVO2_ERR_INVALID, "fp8_fast_accum_gemm: row strides shorter than the rows");
  FastAccArgs a{static_cast<const uint8_t *>(a8), sa, static_cast<const bf16_t *>(b_t), sb,
                input_scale, weight_scale, out, so, out_f32, static_cast<int>(N),
                static_cast<int>(M), static_cast<int>(K)};
  // launches of at most 2^23 workgroups (a grid holds fewer than 2^32 threads)
  const int64_t cols = int64_t(64) << 20;
  for (int64_t c0 = 0; c0 < M; c0 += cols) {
    FastAccArgs b = a;
    b.M = static_cast<int>(M - c0 < cols ? M - c0 : cols);
    b.b += c0;
    const int64_t gx = cdiv(b.M, 64), gxp = 8 * cdiv(gx, 8);
    const int64_t rows = (int64_t(1) << 23) / gxp * (16 * FA_WAVES);
    for (int64_t r0 = 0; r0 < N; r0 += rows) {
      b.N = static_cast<int>(N - r0 < rows ? N - r0 : rows);
      b.a = a.a + r0 * sa;
      b.out = out_f32 ? static_cast<void *>(static_cast<float *>(out) + r0 * so + c0)
                      : static_cast<void *>(static_cast<bf16_t *>(out) + r0 * so + c0);
      const int64_t gy = cdiv(b.N, 16 * FA_WAVES);
      hipLaunchKernelGGL(fast_accum_kernel, dim3(static_cast<unsigned>(gxp * gy)), dim3(64 * FA_WAVES),
                         0, static_cast<hipStream_t>(stream), b, static_cast<int>(gx),
                         static_cast<int>(gy));
    }
  }
  return check_launch("fp8_fast_accum_gemm");
}
