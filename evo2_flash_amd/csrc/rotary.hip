// The step between an attention layer's qkv projection and its attention, for
// the whole-model harness (model.py:104-153): neox rotary of q and k with
// linear position scaling, and the write of k and v into 16-position KV pages
// (keys (pages, heads, head_dim, 16), values (pages, heads, 16, head_dim)).
//
//   angle(t, i) = (t / factor) * inv_freq[i],  i < head_dim / 2
//   (x[i], x[i + hd/2]) -> (x[i] cos - x[i + hd/2] sin, x[i + hd/2] cos + x[i] sin)
//
// in fp32, each product and sum rounded by itself (no FMA: the bits of the
// separate fp32 operators, rotary_neox in model.py), then to bf16 once.  As
// separate elementwise operators this was some 35 launches and ~14 passes over q, k and v: 2.3 ms of a 6.0 ms
// attention layer over a 16384-token prompt (32 heads of 128), 100 us of a
// 299 us decode layer at batch 8.
#include "common.h"

#pragma clang fp contract(off)

namespace evo2 {

struct RotaryArgs {
  const bf16_t *qkv; int64_t sqkv;   // rows (q | k | v), each heads * hd; row stride
  const float *inv_freq;             // (hd / 2,)
  float factor;
  bf16_t *q;                         // rotated queries
  bf16_t *k, *vt;                    // prefill: keys (N, heads, L, hd), values (N, heads, hd, Lv)
  bf16_t *kp; int64_t kp0, kp1, kp2; // key pages + strides (page, head, dim)
  bf16_t *vp; int64_t vp0, vp1, vp2; // value pages + strides (page, head, position)
  int64_t num_pages;
  const int32_t *table; int64_t st;  // block table, row stride
  const int64_t *positions;          // decode: (B,)
  int max_pages;                     // decode: block table columns
  int L, Lv, heads, hd;
};

// Prefill: a workgroup takes 64 positions (four pages) of one sequence and
// RP_HEADS heads in turn, so the angles' sines and cosines are computed once
// for them.  64 positions make every row of the transposed values a whole
// 128-byte line; k and v are transposed through LDS (rows of 65 dwords: the
// eight octets of positions and eight dim pairs a wave reads at once fall on
// 64 different banks).  Bound by memory: it reads q, k, v once and writes q
// once, k and v twice: 16384 positions x 32 heads, 1.07 GB in 235 us (4.6 TB/s;
// a plain copy 4.9).
constexpr int RP_T = 64;      // positions per workgroup
constexpr int RP_HD = 128;    // head dim
constexpr int RP_HEADS = 4;   // heads per workgroup
constexpr int RP_ROW = 65;    // dwords per staged row

__device__ __forceinline__ void unpack8(uint4 w, float (&f)[8]) {
  f[0] = lo_bf(w.x); f[1] = hi_bf(w.x); f[2] = lo_bf(w.y); f[3] = hi_bf(w.y);
  f[4] = lo_bf(w.z); f[5] = hi_bf(w.z); f[6] = lo_bf(w.w); f[7] = hi_bf(w.w);
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  return make_uint4(pack_bf(f[0], f[1]), pack_bf(f[2], f[3]), pack_bf(f[4], f[5]), pack_bf(f[6], f[7]));
}

__global__ __launch_bounds__(256) void rotary_prefill_kernel(RotaryArgs p) {
  __shared__ float2 cs[RP_T][RP_HD / 2];          // cos, sin
  __shared__ uint32_t tile[RP_T * RP_ROW];        // one head's k, then v, by position
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * RP_T;
  const int n = blockIdx.z;
  const int64_t h3 = static_cast<int64_t>(p.heads) * RP_HD;  // elements of q in a row
  const int nt = min(RP_T, p.L - t0);  // positions of the prompt here (none: values' padding only)
  for (int i = tid; i < RP_T * (RP_HD / 2); i += 256) {
    const int t = i / (RP_HD / 2), f = i % (RP_HD / 2);
    float s, c;
    sincosf((static_cast<float>(t0 + t) / p.factor) * p.inv_freq[f], &s, &c);
    cs[t][f] = make_float2(c, s);
  }
  __syncthreads();
  const bf16_t *rows = p.qkv + (static_cast<int64_t>(n) * p.L + t0) * p.sqkv;
  const int h0 = blockIdx.y * RP_HEADS;
  const int h1 = min(h0 + RP_HEADS, p.heads);
  // dim pairs and position octets of the transposed writes
  auto gather = [&](int dp, int o, uint4 &lo, uint4 &hi) __attribute__((always_inline)) {
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = tile[(8 * o + j) * RP_ROW + dp];
    lo = make_uint4((w[0] & 0xffffu) | (w[1] << 16), (w[2] & 0xffffu) | (w[3] << 16),
                    (w[4] & 0xffffu) | (w[5] << 16), (w[6] & 0xffffu) | (w[7] << 16));
    hi = make_uint4((w[0] >> 16) | (w[1] & 0xffff0000u), (w[2] >> 16) | (w[3] & 0xffff0000u),
                    (w[4] >> 16) | (w[5] & 0xffff0000u), (w[6] >> 16) | (w[7] & 0xffff0000u));
  };
  auto page_of = [&](int pg) __attribute__((always_inline)) -> int64_t {
    const int64_t page = p.table[n * p.st + t0 / 16 + pg];
    return page >= 0 && page < p.num_pages ? page : -1;  // no write outside the cache
  };
  const int npg = nt > 0 ? (nt + 15) / 16 : 0;  // pages with a position of the prompt (the last one zero-padded)
  for (int h = h0; h < h1; ++h) {
    const int64_t plane = static_cast<int64_t>(n) * p.heads + h;
    // rotated q to its plane, rotated k to its plane and the tile; item: (t,
    // 8-dim chunk of the first half)
#pragma unroll
    for (int it = 0; it < RP_T * 8 / 256; ++it) {
      const int i = it * 256 + tid;
      const int t = i >> 3, c = (i & 7) * 8;
      uint4 ka = make_uint4(0, 0, 0, 0), kb = ka;
      if (t < nt) {
        const bf16_t *r = rows + t * p.sqkv + h * RP_HD + c;
        const uint4 qa4 = *reinterpret_cast<const uint4 *>(r), qb4 = *reinterpret_cast<const uint4 *>(r + 64);
        const uint4 ka4 = *reinterpret_cast<const uint4 *>(r + h3), kb4 = *reinterpret_cast<const uint4 *>(r + h3 + 64);
        float a[8], b[8], x[8], y[8];
        unpack8(qa4, a);
        unpack8(qb4, b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float2 w = cs[t][c + e];
          x[e] = a[e] * w.x - b[e] * w.y;
          y[e] = b[e] * w.x + a[e] * w.y;
        }
        const int64_t o = (plane * p.L + t0 + t) * RP_HD + c;
        *reinterpret_cast<uint4 *>(p.q + o) = pack8(x);
        *reinterpret_cast<uint4 *>(p.q + o + 64) = pack8(y);
        unpack8(ka4, a);
        unpack8(kb4, b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float2 w = cs[t][c + e];
          x[e] = a[e] * w.x - b[e] * w.y;
          y[e] = b[e] * w.x + a[e] * w.y;
        }
        ka = pack8(x);
        kb = pack8(y);
        *reinterpret_cast<uint4 *>(p.k + o) = ka;
        *reinterpret_cast<uint4 *>(p.k + o + 64) = kb;
      }
      uint32_t *d = tile + t * RP_ROW + c / 2;
      d[0] = ka.x; d[1] = ka.y; d[2] = ka.z; d[3] = ka.w;
      d[32] = kb.x; d[33] = kb.y; d[34] = kb.z; d[35] = kb.w;
    }
    __syncthreads();
    // key pages: a wave writes one page of the head (lane: half of 16
    // positions, dim pair)
    {
      const int pg = tid >> 6, half = tid & 1;
      const int64_t page = pg < npg ? page_of(pg) : -1;
      if (page >= 0) {
        bf16_t *o = p.kp + page * p.kp0 + h * p.kp1 + 8 * half;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          const int dp = it * 32 + ((tid & 63) >> 1);
          uint4 lo, hi;
          gather(dp, 2 * pg + half, lo, hi);
          *reinterpret_cast<uint4 *>(o + (2 * dp) * p.kp2) = lo;
          *reinterpret_cast<uint4 *>(o + (2 * dp + 1) * p.kp2) = hi;
        }
      }
    }
    __syncthreads();
    // values: to their page and the tile
#pragma unroll
    for (int it = 0; it < RP_T * 16 / 256; ++it) {
      const int i = it * 256 + tid;
      const int t = i >> 4, c = (i & 15) * 8;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (t < nt) v = *reinterpret_cast<const uint4 *>(rows + t * p.sqkv + 2 * h3 + h * RP_HD + c);
      const int pg = t >> 4;
      const int64_t page = pg < npg ? page_of(pg) : -1;
      if (page >= 0)
        *reinterpret_cast<uint4 *>(p.vp + page * p.vp0 + h * p.vp1 + (t & 15) * p.vp2 + c) = v;
      uint32_t *d = tile + t * RP_ROW + c / 2;
      d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
    }
    __syncthreads();
    // the transposed values: eight lanes write a dim's 64 positions; zeros
    // from the prompt's end to Lv
    bf16_t *vt = p.vt + plane * RP_HD * p.Lv + t0;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int i = it * 256 + tid;
      const int o = i & 7, dp = i >> 3;
      if (t0 + 8 * o < p.Lv) {
        uint4 lo, hi;
        gather(dp, o, lo, hi);
        bf16_t *w = vt + static_cast<int64_t>(2 * dp) * p.Lv + 8 * o;
        *reinterpret_cast<uint4 *>(w) = lo;
        *reinterpret_cast<uint4 *>(w + p.Lv) = hi;
      }
    }
    __syncthreads();  // the tile is free for the next head's keys
  }
}

// Decode: one token per sequence.  A workgroup takes one sequence and
// RD_HEADS heads; latency only (a few KB a sequence), so it is one launch for
// rotary and both page writes: 5.6 us at batch 8.
constexpr int RD_HEADS = 8;

__global__ __launch_bounds__(256) void rotary_decode_kernel(RotaryArgs p) {
  const int b = blockIdx.y, tid = threadIdx.x;
  const int h0 = blockIdx.x * RD_HEADS, nh = min(RD_HEADS, p.heads - h0);
  const int half = p.hd / 2;
  const int64_t pos = p.positions[b];
  const int64_t col = pos >> 4;
  int64_t page = pos >= 0 && col < p.max_pages ? p.table[b * p.st + col] : -1;
  if (page >= p.num_pages) page = -1;  // no write outside the cache
  const int off = static_cast<int>(pos & 15);
  const int64_t hs = static_cast<int64_t>(p.heads) * p.hd;
  const bf16_t *row = p.qkv + b * p.sqkv;
  const float scaled = static_cast<float>(pos) / p.factor;
  for (int i = tid; i < nh * half; i += 256) {
    const int h = h0 + i / half, f = i % half;
    const bf16_t *r = row + h * p.hd + f;
    float s, c;
    sincosf(scaled * p.inv_freq[f], &s, &c);
    const float q1 = bf2f(r[0]), q2 = bf2f(r[half]), k1 = bf2f(r[hs]), k2 = bf2f(r[hs + half]);
    bf16_t *qo = p.q + b * hs + h * p.hd + f;
    qo[0] = f2bf(q1 * c - q2 * s);
    qo[half] = f2bf(q2 * c + q1 * s);
    if (page >= 0) {
      bf16_t *ko = p.kp + page * p.kp0 + h * p.kp1 + off;
      ko[f * p.kp2] = f2bf(k1 * c - k2 * s);
      ko[(f + half) * p.kp2] = f2bf(k2 * c + k1 * s);
      bf16_t *vo = p.vp + page * p.vp0 + h * p.vp1 + off * p.vp2 + f;
      vo[0] = r[2 * hs];
      vo[half] = r[2 * hs + half];
    }
  }
}

}  // namespace evo2

using namespace evo2;

extern "C" int evo2_rotary_prefill(const void *qkv, int64_t sqkv, const float *inv_freq, float factor,
                                   void *q, void *k, void *vt, int64_t Lv, void *k_pages,
                                   int64_t kp0, int64_t kp1, int64_t kp2, void *v_pages, int64_t vp0,
                                   int64_t vp1, int64_t vp2, int64_t num_pages, const int32_t *table,
                                   int64_t st, int64_t max_pages, int64_t N, int64_t heads,
                                   int64_t head_dim, int64_t L, void *stream) {
  if (N < 0 || heads <= 0 || L < 0 || N > 65535 || cdiv(heads, RP_HEADS) > 65535 || L > 0x7fffff00 ||
      Lv < L || Lv > 0x7fffff00 || num_pages < 0)
    return fail(EVO2_ERR_INVALID, "rotary_prefill: bad sizes N=%lld heads=%lld L=%lld Lv=%lld", (long long)N,
                (long long)heads, (long long)L, (long long)Lv);
  if (head_dim != RP_HD)
    return fail(EVO2_ERR_UNSUPPORTED, "rotary_prefill: head_dim %lld (128 only)", (long long)head_dim);
  if (N == 0 || L == 0) return EVO2_OK;
  if (!qkv || !inv_freq || !q || !k || !vt || !k_pages || !v_pages || !table)
    return fail(EVO2_ERR_INVALID, "rotary_prefill: null pointer argument");
  if (cdiv(L, 16) > max_pages)
    return fail(EVO2_ERR_INVALID, "rotary_prefill: %lld positions exceed the block table's %lld pages",
                (long long)L, (long long)max_pages);
  if (Lv > cdiv(L, 128) * 128 || Lv % 8)
    return fail(EVO2_ERR_INVALID, "rotary_prefill: Lv=%lld must be a multiple of 8 within the last 128 positions",
                (long long)Lv);
  const uintptr_t align = reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(q) |
                          reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(vt) |
                          reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages);
  if (align % 16 || sqkv % 8 || kp0 % 8 || kp1 % 8 || kp2 % 8 || vp0 % 8 || vp1 % 8 || vp2 % 8)
    return fail(EVO2_ERR_UNSUPPORTED, "rotary_prefill: rows must be 16-byte aligned");
  RotaryArgs a{static_cast<const bf16_t *>(qkv), sqkv, inv_freq, factor, static_cast<bf16_t *>(q),
               static_cast<bf16_t *>(k), static_cast<bf16_t *>(vt), static_cast<bf16_t *>(k_pages), kp0, kp1,
               kp2, static_cast<bf16_t *>(v_pages), vp0, vp1, vp2, num_pages, table, st, nullptr,
               static_cast<int>(max_pages), static_cast<int>(L), static_cast<int>(Lv),
               static_cast<int>(heads), RP_HD};
  hipLaunchKernelGGL(rotary_prefill_kernel,
                     dim3(static_cast<unsigned>(cdiv(Lv, RP_T)), static_cast<unsigned>(cdiv(heads, RP_HEADS)),
                          static_cast<unsigned>(N)),
                     dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return check_launch("rotary_prefill");
}

extern "C" int evo2_rotary_decode(const void *qkv, int64_t sqkv, const float *inv_freq, float factor,
                                  void *q, void *k_pages, int64_t kp0, int64_t kp1, int64_t kp2,
                                  void *v_pages, int64_t vp0, int64_t vp1, int64_t vp2,
                                  int64_t num_pages, const int32_t *table, int64_t st, int64_t max_pages,
                                  const int64_t *positions, int64_t B, int64_t heads, int64_t head_dim,
                                  void *stream) {
  if (B < 0 || heads <= 0 || head_dim <= 0 || head_dim % 2 || B > 65535 || heads > 0x7fffff ||
      head_dim > 0xffff || num_pages < 0 || max_pages > 0x7fffffff)
    return fail(EVO2_ERR_INVALID, "rotary_decode: bad sizes B=%lld heads=%lld head_dim=%lld", (long long)B,
                (long long)heads, (long long)head_dim);
  if (B == 0) return EVO2_OK;
  if (!qkv || !inv_freq || !q || !k_pages || !v_pages || !table || !positions)
    return fail(EVO2_ERR_INVALID, "rotary_decode: null pointer argument");
  RotaryArgs a{static_cast<const bf16_t *>(qkv), sqkv, inv_freq, factor, static_cast<bf16_t *>(q), nullptr,
               nullptr, static_cast<bf16_t *>(k_pages), kp0, kp1, kp2, static_cast<bf16_t *>(v_pages), vp0,
               vp1, vp2, num_pages, table, st, positions, static_cast<int>(max_pages), 1, 1,
               static_cast<int>(heads), static_cast<int>(head_dim)};
  hipLaunchKernelGGL(rotary_decode_kernel,
                     dim3(static_cast<unsigned>(cdiv(heads, RD_HEADS)), static_cast<unsigned>(B)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch("rotary_decode");
}
