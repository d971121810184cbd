// Row kernels of the prompt forward (prefill) between its GEMMs, for gfx950.
//
// The prompt forward has to leave the bits of Transformers' Qwen3 modules run
// with torch's GPU kernels (engine/engine.py:343-351), so each kernel here
// restates a chain of torch elementwise and reduction kernels: fp32 arithmetic,
// bf16 rounding wherever a module stores a bf16 tensor, and the fp32 sums of the
// mean of squares in the order torch's row reduction leaves them in (row_sq_order
// below). The wrappers compare that order with torch once per device and row
// width; where it differs, the torch operations run instead.
//
// All three are bound by memory: they read and write each bf16 element once,
// where the torch chain writes an fp32 copy, its squares and every rounded
// intermediate (a norm is 8 kernels and 34 bytes per element, here one kernel
// and 4, or 8 with the residual add). At 8192 tokens of the Qwen3-4B widths: residual
// add + norm 28.4 us (5.9 TB/s), q/k norm + RoPE + cache 47.7 us (4.2 TB/s), SwiGLU
// 75.2 us (6.4 TB/s); all of a layer's torch kernels around the GEMMs and SDPA took
// about 1,100 us there, these take 180. Four layers of prefill: 512 tokens 2,175 ->
// 1,319 us, 4 x 2048 tokens 11,980 -> 8,456 us.
#include "ko_common.h"

using namespace ko;

namespace {

// a * b and a + b rounded separately: torch's square, sums and products are
// different kernels, so nothing may be fused into an fma.
__device__ __forceinline__ float mul_r(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float add_r(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// The order of the sums of a row's squares over W lanes (64 for rows of 256 to
// 8064 elements, 32 for heads of 128): lane l takes the quads l, l + W, ... of
// the row, keeps the four positions of a quad in four sums, adds those in
// order, and the lanes are then added pairwise, neighbours first.
__device__ __forceinline__ void row_sq(float (&a)[4], const uint2& v) {
  const float e0 = bf16lo(v.x), e1 = bf16hi(v.x), e2 = bf16lo(v.y), e3 = bf16hi(v.y);
  a[0] = add_r(a[0], mul_r(e0, e0));
  a[1] = add_r(a[1], mul_r(e1, e1));
  a[2] = add_r(a[2], mul_r(e2, e2));
  a[3] = add_r(a[3], mul_r(e3, e3));
}
template <int W>
__device__ __forceinline__ float row_sq_order(const float (&a)[4]) {
  float v = add_r(add_r(add_r(a[0], a[1]), a[2]), a[3]);
  // After each step all lanes of a group hold the group's sum, so a mirror
  // reaches the neighbouring group as an xor would.
  v = add_r(v, dpp_f<0xb1>(v));    // quad_perm [1, 0, 3, 2]
  v = add_r(v, dpp_f<0x4e>(v));    // quad_perm [2, 3, 0, 1]
  v = add_r(v, dpp_f<0x141>(v));   // row_half_mirror
  v = add_r(v, dpp_f<0x140>(v));   // row_mirror
  v = sum_xor16(v);
  if constexpr (W == 64) v = sum_xor32(v);
  return v;
}

// torch.rsqrt's bits, which are the correctly rounded ones (v_rsq_f32 alone is one
// ulp off for 11 % of the mantissas): a third-order step in fp64 on v_rsq_f32. Equal to
// torch.rsqrt for every mantissa at both exponent parities.
__device__ __forceinline__ float rsqrt_torch(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const double yd = (double)y, e = 1.0 - (double)x * yd * yd;
  const float z = (float)(yd + yd * e * (0.5 + 0.375 * e));
  return y == 0.f || __builtin_isinf(y) ? y : z;  // x infinite or zero
}

__device__ __forceinline__ uint2 ldg8(const void* p) {
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  typedef const __attribute__((address_space(1))) u32x2 g_u32x2;
  const u32x2 v = *(g_u32x2*)p;
  return make_uint2(v.x, v.y);
}
// bf16(w * bf16(x * rstd)) on a packed pair
__device__ __forceinline__ uint32_t scale2(uint32_t x, uint32_t w, float rstd) {
  const uint32_t t = pack_bf16x2(bf16lo(x) * rstd, bf16hi(x) * rstd);
  return pack_bf16x2(bf16lo(w) * bf16lo(t), bf16hi(w) * bf16hi(t));
}
__device__ __forceinline__ uint32_t add2(uint32_t x, uint32_t y) {
  return pack_bf16x2(bf16lo(x) + bf16lo(y), bf16hi(x) + bf16hi(y));
}

// ---- residual add + RMSNorm of one row per wavefront ------------------------
// NC: quads per lane (n <= 256 * NC). A wavefront's loads are all issued before
// the first sum; a row of 2560 is 10 loads of 512 bytes.
template <int NC, bool ADD>
__global__ __launch_bounds__(256) void prefill_norm_kernel(uint16_t* __restrict__ res,
                                                           const uint16_t* __restrict__ delta,
                                                           const uint16_t* __restrict__ wt,
                                                           uint16_t* __restrict__ out, int rows,
                                                           int n, float inv_n, float eps) {
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  uint16_t* rp = res + row * n;
  uint2 x[NC], d[ADD ? NC : 1], w[NC];
  const uint2 zero = make_uint2(0, 0);
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = 4 * (64 * j + lane);
    x[j] = c < n ? ldg8(rp + c) : zero;
    if constexpr (ADD) d[j] = c < n ? ldg8(delta + row * n + c) : zero;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = 4 * (64 * j + lane);
    w[j] = c < n ? ldg8(wt + c) : zero;
  }
  float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = 4 * (64 * j + lane);
    if constexpr (ADD) {
      x[j] = make_uint2(add2(x[j].x, d[j].x), add2(x[j].y, d[j].y));
      if (c < n) *reinterpret_cast<uint2*>(rp + c) = x[j];
    }
    if (c < n) row_sq(a, x[j]);
  }
  const float var = mul_r(row_sq_order<64>(a), inv_n);
  const float rstd = rsqrt_torch(add_r(var, eps));
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = 4 * (64 * j + lane);
    if (c < n)
      *reinterpret_cast<uint2*>(out + row * n + c) =
          make_uint2(scale2(x[j].x, w[j].x, rstd), scale2(x[j].y, w[j].y, rstd));
  }
}

// ---- q/k RMSNorm + RoPE and the prompt's K/V into the cache ------------------
// A head takes 32 lanes (lane r of the half: elements 4r .. 4r + 3), so a
// wavefront works on two heads at a time, HT pairs of one token with their loads
// issued together; the rotate_half partner (element +- 64) is 16 lanes away.
// One wavefront per item = token * tasks + task (a task: 2 * HT heads), 4 items a workgroup:
// cos and sin are read once per task.
constexpr int PD = 128;  // head dim
constexpr int HT = 4;    // pairs of heads per wavefront

__global__ __launch_bounds__(256) void prefill_qkv_kernel(
    uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ qw, const uint16_t* __restrict__ kw,
    const uint16_t* __restrict__ cosb, const uint16_t* __restrict__ sinb,
    uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, int M, int S, int tasks, long long cb,
    long long ch, float eps, int nq, int nkv) {
  const int lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int m = item / tasks, task = item - m * tasks;
  if (m >= M) return;
  const int b = m / S, s = m - b * S;
  const int nh = nq + 2 * nkv, h0 = task * 2 * HT + half;
  uint2 x[HT], w[HT];
#pragma unroll
  for (int i = 0; i < HT; ++i) {
    const int h = min(h0 + 2 * i, nh - 1);
    const uint16_t* src = h < nq ? q + ((long long)m * nq + h) * PD
                          : h < nq + nkv ? k + ((long long)m * nkv + (h - nq)) * PD
                                         : v + ((long long)m * nkv + (h - nq - nkv)) * PD;
    x[i] = ldg8(src + 4 * r);
    w[i] = ldg8((h < nq ? qw : kw) + 4 * r);
  }
  const uint2 cv = ldg8(cosb + (long long)s * PD + 4 * r);
  const uint2 sv = ldg8(sinb + (long long)s * PD + 4 * r);
#pragma unroll
  for (int i = 0; i < HT; ++i) {
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    row_sq(a, x[i]);
    const float var = mul_r(row_sq_order<32>(a), 1.0f / PD);
    const float rstd = rsqrt_torch(add_r(var, eps));
    const uint2 xn = make_uint2(scale2(x[i].x, w[i].x, rstd), scale2(x[i].y, w[i].y, rstd));
    // the partner's four elements (lane r ^ 16): rows {0, 0, 2, 2} and {1, 1, 3, 3}
    const auto p0 = __builtin_amdgcn_permlane16_swap(xn.x, xn.x, false, false);
    const auto p1 = __builtin_amdgcn_permlane16_swap(xn.y, xn.y, false, false);
    const bool low = r < 16;  // rotate_half: the first half takes -x[d + 64]
    const uint32_t neg = low ? 0x80008000u : 0u;
    const uint32_t o0 = (low ? (uint32_t)p0[1] : (uint32_t)p0[0]) ^ neg;
    const uint32_t o1 = (low ? (uint32_t)p1[1] : (uint32_t)p1[0]) ^ neg;
    // bf16(bf16(xn * cos) + bf16(rot * sin))
    const uint32_t a0 = pack_bf16x2(bf16lo(xn.x) * bf16lo(cv.x), bf16hi(xn.x) * bf16hi(cv.x));
    const uint32_t a1 = pack_bf16x2(bf16lo(xn.y) * bf16lo(cv.y), bf16hi(xn.y) * bf16hi(cv.y));
    const uint32_t b0 = pack_bf16x2(bf16lo(o0) * bf16lo(sv.x), bf16hi(o0) * bf16hi(sv.x));
    const uint32_t b1 = pack_bf16x2(bf16lo(o1) * bf16lo(sv.y), bf16hi(o1) * bf16hi(sv.y));
    const uint2 y = make_uint2(add2(a0, b0), add2(a1, b1));
    const int h = h0 + 2 * i;
    if (h >= nh) continue;
    uint16_t* dst;
    if (h < nq) dst = q + ((long long)m * nq + h) * PD;
    else if (h < nq + nkv) dst = kc + b * cb + (h - nq) * ch + (long long)s * PD;
    else dst = vc + b * cb + (h - nq - nkv) * ch + (long long)s * PD;
    *reinterpret_cast<uint2*>(dst + 4 * r) = h < nq + nkv ? y : x[i];
  }
}

// ---- SwiGLU of separate gate and up tensors ----------------------------------
__device__ __forceinline__ uint32_t silu2(uint32_t g, uint32_t u) {
  const float g0 = bf16lo(g), g1 = bf16hi(g);
  const uint32_t t = pack_bf16x2(g0 / (1.0f + expf(-g0)), g1 / (1.0f + expf(-g1)));
  return pack_bf16x2(bf16lo(t) * bf16lo(u), bf16hi(t) * bf16hi(u));
}
// out may be gate (each thread reads its chunk before it writes it): no __restrict__ there.
__global__ __launch_bounds__(256) void silu_mul2_kernel(const uint16_t* gate,
                                                        const uint16_t* __restrict__ up,
                                                        uint16_t* out, long long nc) {
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= nc) return;
  const uint4 g = ldg16(gate + 8 * c), u = ldg16(up + 8 * c);
  *reinterpret_cast<uint4*>(out + 8 * c) =
      make_uint4(silu2(g.x, u.x), silu2(g.y, u.y), silu2(g.z, u.z), silu2(g.w, u.w));
}

bool al(const void* p, unsigned a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace

extern "C" {

int ko_prefill_norm(void* res, const void* delta, const void* weight, void* out, int rows, int n,
                    float eps, void* stream) {
  if (!res || !weight || !out || rows < 1) return KO_EINVAL;
  if (n < 256 || n > 8064 || (n & 3)) return KO_ENOTSUP;
  if (!al(res, 8) || !al(weight, 8) || !al(out, 8) || (delta && !al(delta, 8))) return KO_EINVAL;
  // one wavefront per workgroup while that fills the 256 CUs less than 8 deep
  const int wpb = rows <= 2048 ? 1 : 4;
  const dim3 grid((rows + wpb - 1) / wpb), block(64 * wpb);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float inv = 1.0f / (float)n;
  uint16_t* r = static_cast<uint16_t*>(res);
  const uint16_t* d = static_cast<const uint16_t*>(delta);
  const uint16_t* w = static_cast<const uint16_t*>(weight);
  uint16_t* o = static_cast<uint16_t*>(out);
#define KO_PN(NC)                                                                              \
  if (d) hipLaunchKernelGGL((prefill_norm_kernel<NC, true>), grid, block, 0, s, r, d, w, o,    \
                            rows, n, inv, eps);                                                \
  else hipLaunchKernelGGL((prefill_norm_kernel<NC, false>), grid, block, 0, s, r, d, w, o,     \
                          rows, n, inv, eps)
  if (n <= 2560) {
    KO_PN(10);
  } else {
    KO_PN(32);
  }
#undef KO_PN
  return KO_LAUNCH_STATUS();
}

int ko_prefill_qkv(void* q, const void* k, const void* v, const void* q_w, const void* k_w,
                   const void* cos, const void* sin, void* k_cache, void* v_cache, int B, int S,
                   long long cache_b_stride, long long cache_h_stride, float eps, int nq, int nkv,
                   int d, int max_pos, void* stream) {
  if (!q || !k || !v || !q_w || !k_w || !cos || !sin || !k_cache || !v_cache) return KO_EINVAL;
  if (d != PD) return KO_ENOTSUP;
  if (B < 1 || S < 1 || nq < 1 || nkv < 1 || S > max_pos || cache_b_stride < 0 ||
      cache_h_stride < 0 || (cache_b_stride & 3) || (cache_h_stride & 3))
    return KO_EINVAL;
  if (!al(q, 8) || !al(k, 8) || !al(v, 8) || !al(q_w, 8) || !al(k_w, 8) || !al(cos, 8) ||
      !al(sin, 8) || !al(k_cache, 8) || !al(v_cache, 8))
    return KO_EINVAL;
  const int tasks = (nq + 2 * nkv + 2 * HT - 1) / (2 * HT);
  const long long items = (long long)B * S * tasks;
  if (items > 0x7fffff00LL) return KO_ERANGE;
  hipLaunchKernelGGL(prefill_qkv_kernel, dim3((unsigned)((items + 3) / 4)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<uint16_t*>(q),
                     static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v),
                     static_cast<const uint16_t*>(q_w), static_cast<const uint16_t*>(k_w),
                     static_cast<const uint16_t*>(cos), static_cast<const uint16_t*>(sin),
                     static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), B * S, S,
                     tasks, cache_b_stride, cache_h_stride, eps, nq, nkv);
  return KO_LAUNCH_STATUS();
}

int ko_silu_mul2(const void* gate, const void* up, void* out, long long n, void* stream) {
  if (!gate || !up || !out || n < 8 || (n & 7)) return KO_EINVAL;
  if (!al(gate, 16) || !al(up, 16) || !al(out, 16)) return KO_EINVAL;
  const long long nc = n >> 3, blocks = (nc + 255) / 256;
  if (blocks > 0x7fffffffLL) return KO_ERANGE;
  hipLaunchKernelGGL(silu_mul2_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(gate),
                     static_cast<const uint16_t*>(up), static_cast<uint16_t*>(out), nc);
  return KO_LAUNCH_STATUS();
}

}  // extern "C"
