// bf16 projections of a decode step: up to 16 rows against an (N, K) weight,
//
//   out[m, n] = bf16( sum_k X[m, k] W[n, k] [+ bias[n]] )   (fp32 sums)
//   [+ residual[m, n], rounded again]
//   or, gated:  bf16( act(bf16(X W1^T)) * bf16(X W2^T) )
//
// the out_proj, qkv / o projections and MLP of the model at decode batch sizes
// (model.py:77-153, mixers.py:801-803; library GEMMs and elementwise operators
// in the reference).
//
// The weight stream is the whole cost, and a call is short (5-40 us), so what
// counts is how soon its loads are in flight and how many.  A workgroup owns 16
// W rows and its eight waves split K: each reads its part of those rows straight
// into registers (v_mfma_f32_16x16x32_bf16, the weight as operand A), four k
// steps ahead in 42 VGPRs, so that four workgroups share a CU and one's start
// and end pass under the others' streams.  The partial sums meet in LDS.  The
// gated form streams both weights and writes the product: one launch for two
// GEMMs, the activation and the multiply.
//
// Measured with the weights streaming from HBM (us at M = 1 / 8 / 16, against
// the library's GEMM): 4096 x 4096 8.5 / 9.6 / 11.5 (15.6), 11264 x 4096 20.2 /
// 24.7 / 29.7 (26.4), 4096 x 11264 18.7 / 20.0 / 26.7 (20.6 / 19.5 / 20.0), 1920 x
// 1920 4.5 / 5.1 / 5.9 (8.0); gated 2 x 11264 x 4096 34.5 / 37.0 / 42.0 (52.4 and
// 5 for the multiply).  The rows of X cost as L2 reads, so the plain form takes
// M > 8 only for small weights, and fewer than 8 at K > 5120 (linear.py has the
// rule and its figures).  Sixteen k steps ahead 9.3 / 11.9 /
// 13.5 at 4096 x 4096, two row groups a workgroup 13 / 15 / 17, sixteen waves 9.1
// / 10.4 / 12.3, loads of X for the M rows alone 11.0 / 11.8 / 12.8.
#include <type_traits>

#include "common.h"

namespace evo2 {

typedef __attribute__((ext_vector_type(4))) float sl_f4;
typedef __bf16 sl_b8 __attribute__((ext_vector_type(8)));

constexpr int SL_ROWS = 16;   // X rows
constexpr int SL_WAVES = 8;   // waves per workgroup: parts of K
constexpr int SL_CH = 2;      // k-steps of 32 per chunk, two chunks in flight

struct StreamArgs {
  const bf16_t *x; int64_t sx;    // (M, K)
  const bf16_t *w[2]; int64_t sw; // (N, K) each
  const bf16_t *bias;             // (N,) or null
  const bf16_t *res; int64_t sr;  // (M, N) added after rounding, or null
  bf16_t *out; int64_t so;        // (M, N)
  int M, N, K;
  int gelu;                       // gated: exact GELU on the first product
};

template <bool GATED>
__global__ __launch_bounds__(64 * SL_WAVES) void bf16_stream_kernel(StreamArgs p) {
  constexpr int NWT = GATED ? 2 : 1;
  __shared__ float part[NWT][SL_WAVES][256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;  // operand row, octet of k
  const int n0 = blockIdx.x * 16;
  const int units = p.K / 32, per = (units + SL_WAVES - 1) / SL_WAVES;
  const int u0 = wave * per, u1 = min(u0 + per, units);  // this wave's k-steps
  const bf16_t *wr[NWT];
#pragma unroll
  for (int t = 0; t < NWT; ++t)
    wr[t] = p.w[t] + (int64_t)min(n0 + r, p.N - 1) * p.sw + 8 * g;
  const bf16_t *xr = p.x + (int64_t)min(r, p.M - 1) * p.sx + 8 * g;
  uint4 wf[2][NWT][SL_CH], xf[2][SL_CH];
  auto load = [&](auto buf, int u) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int j = 0; j < SL_CH; ++j) {
      const int k = 32 * min(u + j, units - 1);  // (past the part: loaded, not used)
#pragma unroll
      for (int t = 0; t < NWT; ++t) wf[B][t][j] = *reinterpret_cast<const uint4 *>(wr[t] + k);
      xf[B][j] = *reinterpret_cast<const uint4 *>(xr + k);
    }
  };
  sl_f4 acc[NWT];
#pragma unroll
  for (int t = 0; t < NWT; ++t) acc[t] = sl_f4{0.f, 0.f, 0.f, 0.f};
  auto use = [&](auto buf, int u) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int j = 0; j < SL_CH; ++j) {
      if (u + j >= u1) break;  // uniform
#pragma unroll
      for (int t = 0; t < NWT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sl_b8, wf[B][t][j]),
                                                         __builtin_bit_cast(sl_b8, xf[B][j]), acc[t], 0, 0, 0);
    }
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  load(B0{}, u0);
  load(B1{}, u0 + SL_CH);
  for (int u = u0; u < u1; u += 2 * SL_CH) {
    use(B0{}, u);
    if (u + 2 * SL_CH < u1) load(B0{}, u + 2 * SL_CH);
    use(B1{}, u + SL_CH);
    if (u + 3 * SL_CH < u1) load(B1{}, u + 3 * SL_CH);
  }
  // lane (r, g) holds X row r, W rows n0 + 4 g + i in acc[.][i]
#pragma unroll
  for (int t = 0; t < NWT; ++t)
    *reinterpret_cast<sl_f4 *>(&part[t][wave][4 * lane]) = acc[t];
  __syncthreads();
  if (tid >= 256) return;
  const int m = (tid >> 2) & 15, n = n0 + 4 * (tid >> 6) + (tid & 3);
  if (m >= p.M || n >= p.N) return;
  float v[NWT];
#pragma unroll
  for (int t = 0; t < NWT; ++t) {
    v[t] = 0.0f;
#pragma unroll
    for (int w = 0; w < SL_WAVES; ++w) v[t] += part[t][w][tid];
  }
  float o = v[0];
  if constexpr (GATED) {
    float a = rbf(v[0]);
    if (p.gelu) a = rbf(0.5f * a * (1.0f + erff(a * 0.70710678118654752440f)));
    o = a * rbf(v[1]);
  } else {
    if (p.bias) o += bf2f(p.bias[n]);
    if (p.res) o = rbf(o) + bf2f(p.res[(int64_t)m * p.sr + n]);
  }
  p.out[(int64_t)m * p.so + n] = f2bf(o);
}

}  // namespace evo2

using namespace evo2;

static int stream_check(const char *who, int64_t M, int64_t N, int64_t K, const void *x, int64_t sx,
                        const void *w, const void *w2, int64_t sw, const void *out) {
  if (M < 0 || N <= 0 || K <= 0 || N > 0x7fffff00 || K > 0x7fffff00)
    return fail(EVO2_ERR_INVALID, "%s: bad sizes M=%lld N=%lld K=%lld", who, (long long)M, (long long)N,
                (long long)K);
  if (M > SL_ROWS || K % 32)
    return fail(EVO2_ERR_UNSUPPORTED, "%s: M=%lld must be at most %d and K=%lld a multiple of 32", who,
                (long long)M, SL_ROWS, (long long)K);
  if (M > 0 && (!x || !w || !w2 || !out)) return fail(EVO2_ERR_INVALID, "%s: null pointer argument", who);
  if (sx % 8 || sw % 8 || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16 ||
      reinterpret_cast<uintptr_t>(w2) % 16)
    return fail(EVO2_ERR_UNSUPPORTED, "%s: operand rows must be 16-byte aligned", who);
  return EVO2_OK;
}

extern "C" int evo2_bf16_stream_linear(const void *x, int64_t sx, const void *w, int64_t sw, const void *bias,
                                       const void *residual, int64_t sr, void *out, int64_t so, int64_t M,
                                       int64_t N, int64_t K, void *stream) {
  const int rc = stream_check("bf16_stream_linear", M, N, K, x, sx, w, w, sw, out);
  if (rc || M == 0) return rc;
  StreamArgs a{static_cast<const bf16_t *>(x), sx,
               {static_cast<const bf16_t *>(w), static_cast<const bf16_t *>(w)}, sw,
               static_cast<const bf16_t *>(bias), static_cast<const bf16_t *>(residual), sr,
               static_cast<bf16_t *>(out), so, static_cast<int>(M), static_cast<int>(N),
               static_cast<int>(K), 0};
  hipLaunchKernelGGL(bf16_stream_kernel<false>, dim3(static_cast<unsigned>(cdiv(N, 16))), dim3(64 * SL_WAVES), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch("bf16_stream_linear");
}

extern "C" int evo2_bf16_stream_gated(const void *x, int64_t sx, const void *w1, const void *w2, int64_t sw,
                                      int32_t gelu, void *out, int64_t so, int64_t M, int64_t N, int64_t K,
                                      void *stream) {
  const int rc = stream_check("bf16_stream_gated", M, N, K, x, sx, w1, w2, sw, out);
  if (rc || M == 0) return rc;
  StreamArgs a{static_cast<const bf16_t *>(x), sx,
               {static_cast<const bf16_t *>(w1), static_cast<const bf16_t *>(w2)}, sw, nullptr, nullptr, 0,
               static_cast<bf16_t *>(out), so, static_cast<int>(M), static_cast<int>(N),
               static_cast<int>(K), gelu};
  hipLaunchKernelGGL(bf16_stream_kernel<true>, dim3(static_cast<unsigned>(cdiv(N, 16))), dim3(64 * SL_WAVES), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch("bf16_stream_gated");
}
