// Skinny GEMM, layout 5: up to 64 rows of x per weight pass on MFMA tiles
// (v_mfma_f32_16x16x32_bf16 on the tiled weight copy); the semantics are those of
// gemv.hip's entry points (engine/kernels/gemv.py:30-106).
//
// Bound by the weight stream and, from 16 rows on, by how fast a CU takes in x: layouts 2
// and 4 read x again for every one or two column tiles, in a pattern that touches 16
// half lines per load, and normalise it in every workgroup. Here
//   - a workgroup owns several column tiles at once. At the layer projections' widths that
//     is at most one workgroup per CU, so x passes through each CU once; the LM head's 9,496
//     tiles are 1,583 workgroups of 6, which read all of x each (at 64 rows 320 KiB, 520 MB
//     from the L2s beside 778 MB of weights: 208 us, against 288 in layout 2's two passes);
//   - the projections behind a norm read x normalised beforehand (row_finish_kernel), in
//     the MFMA operand order, 1 KiB contiguous per load (16 / 64 rows, 6144 x 2560:
//     8.5 / 17.2 us with x in rows, 7.6 / 12.0 us in this order);
//   - the residual projections, whose 160 column tiles cannot fill 256 CUs, also cut K
//     into slices with plain stores of the fp32 sums; row_finish_kernel adds them,
//     the residual, and leaves the next projection's normalised x.
// Measured against layouts 2 and 4 with their norms (us, cold weights; the residual
// projections with their row_finish): 32 rows qkv 14.3 -> 9.2, o 10.5 -> 8.9, gate/up 24.3
// -> 20.5, down 19.5 -> 14.0; 64 rows 27.7 -> 12.0, 15.5 -> 10.5, 47.5 -> 24.7, 31.9 ->
// 17.2; a norm of its own costs 2.8-3.6.
#include "gemv_launch.h"

using namespace ko;

namespace {

constexpr int RW = 8;  // wavefronts per workgroup

__device__ __forceinline__ void arg_better(float ov, int oi, float& v, int& i) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

// Element (m, k) of x in the operand order of a call with mt row tiles: for K step k / 32
// and row tile m / 16 a 1 KiB block, lane l = m % 16 + 16 (k % 32 / 8) at 8 l.
__device__ __forceinline__ long long xt_index(int m, int k, int mt) {
  return ((long long)(k >> 5) * mt + (m >> 4)) * 512 + ((m & 15) + 16 * ((k & 31) >> 3)) * 8 +
         (k & 7);
}

// Workgroup (group, slice): TN column tiles (with their up tiles for SWIGLU) over the
// slice's `steps` K steps of 32, at most NS a wavefront. A wavefront multiplies every
// weight block of a step with all MT row tiles of x. SUMS: the slice's fp32 sums to
// part[slice][row][column], else the epilogue.
// XT: x in the operand order, padded to 16 MT rows; the steps are dealt out one at a time,
// and x and weights run through one ring of PD steps in registers (as many as they hold
// beside MT * NB accumulators). Else x in rows: a wavefront has consecutive steps, loads
// their x as runs of each row, turns it through its own LDS (as layout 2) and keeps it;
// only the weights run through the ring (64 / 32 rows, against x read from rows in operand
// order in the ring: o 13.1 -> 10.5 / 10.1 -> 8.9 us, down 20.2 -> 17.2 / 15.1 -> 14.0).
template <int EPI, bool XT, bool SUMS, int MT, int TN, int NS, int PD>
__global__ __launch_bounds__(64 * RW, 1) void gemm_rows_kernel(GemvArgs a, int nslices, int steps,
                                                               float* __restrict__ part) {
  constexpr int NW = EPI == EPI_SWIGLU ? 2 : 1, NB = TN * NW;
  constexpr int MR = NB * MT <= 12 ? MT : 12 / NB;  // row tiles summed per round (96 KiB)
  static_assert(MR >= 1 && PD <= NS, "one row tile of sums fits the LDS");
  // a wavefront's own region: its x on the way to the operand order, later its sums
  constexpr int XR = XT ? 0 : 68 * NS, CR = MR * NB * 64, CPR = 4 * NS;
  __shared__ uint4 s_w[RW][XR > CR ? XR : CR];
  __shared__ float2 s_best[EPI == EPI_ARGMAX ? MT * 16 : 1][TN];
  const int t = threadIdx.x, wv = t >> 6, lane = t & 63, col = lane & 15, g = lane >> 4;
  const int N = a.N, K = a.K, mr = a.mrows, T = (N + 15) / 16, KS = K / 32;
  const int group = blockIdx.x / nslices, slice = blockIdx.x - group * nslices;
  const int s0 = slice * steps, tile0 = group * TN;
  // step j of this wavefront: first + stride * j, while below `steps`
  const int first = XT ? wv : wv * NS;
  constexpr int STRIDE = XT ? RW : 1;

  const uint16_t* wp[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
    wp[n] = a.w + ((long long)min(tile0 + n / NW, T - 1) + (n % NW) * T) * KS * 512 + 8 * lane;
  uint4 xb[XT ? PD : NS][MT], wb[PD][NB];
  auto issue = [&](int j, int slot) {
    const int st = s0 + min(first + STRIDE * j, steps - 1);  // past the end: loaded, not used
    if constexpr (XT) {
#pragma unroll
      for (int u = 0; u < MT; ++u)
        xb[slot][u] = ldg16(a.x + ((long long)st * MT + u) * 512 + 8 * lane);
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) wb[slot][n] = ldg16_stream(wp[n] + (long long)st * 512);
  };
  if constexpr (!XT) {
    // rows past mrows and steps past the slice: a valid chunk, whose result is not used
    const int kmax = 4 * max(min(steps - first, NS), 1) - 1;
    const uint16_t* xs = a.x + (s0 + min(first, steps - 1)) * 32;
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int ch = 64 * i + lane, row = ch / CPR, kc = min(ch - row * CPR, kmax);
        if (64 * i < (mr - 16 * u) * CPR)  // uniform
          xb[i][u] = ldg16(xs + (long long)min(16 * u + row, mr - 1) * K + 8 * kc);
      }
    __builtin_amdgcn_sched_barrier(0);  // x ahead of the weights: loads return in order
  }
#pragma unroll
  for (int j = 0; j < PD; ++j) issue(j, j);
  __builtin_amdgcn_sched_barrier(0);  // the whole ring is in flight before the first product
  if constexpr (!XT) {
#pragma unroll
    for (int u = 0; u < MT; ++u) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int ch = 64 * i + lane, row = ch / CPR, kc = ch - row * CPR;
        if (64 * i < (mr - 16 * u) * CPR) s_w[wv][68 * (kc >> 2) + 17 * (kc & 3) + row] = xb[i][u];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int j = 0; j < NS; ++j) xb[j][u] = s_w[wv][68 * j + 17 * g + col];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }

  f32x4 c[MT][NB];
#pragma unroll
  for (int u = 0; u < MT; ++u)
#pragma unroll
    for (int n = 0; n < NB; ++n) c[u][n] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int slot = j % PD;
    if (first + STRIDE * j < steps) {  // uniform per wavefront
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int u = 0; u < MT; ++u)
          c[u][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, xb[XT ? slot : j][u]),
              __builtin_bit_cast(bf16x8, wb[slot][n]),
              c[u][n], 0, 0, 0);
    }
    if (j + PD < NS) issue(j + PD, slot);
  }

  // The wavefronts' sums through LDS in the accumulators' own order (16 bytes per lane,
  // no bank conflicts), MR row tiles a round; a wavefront finishes whole tiles: lane
  // (col, g) holds rows 4g .. 4g + 3 of column col.
#pragma unroll
  for (int u0 = 0; u0 < MT; u0 += MR) {
    if (u0) __syncthreads();
#pragma unroll
    for (int u = u0; u < u0 + MR && u < MT; ++u)
#pragma unroll
      for (int n = 0; n < NB; ++n)
        s_w[wv][((u - u0) * NB + n) * 64 + lane] = __builtin_bit_cast(uint4, c[u][n]);
    __syncthreads();
    const int ru = min(MR, MT - u0);
    for (int task = wv; task < ru * TN; task += RW) {
      const int u = task / TN, q = task - u * TN;
      float tot[4] = {0.f, 0.f, 0.f, 0.f}, tot2[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        const f32x4 v = __builtin_bit_cast(f32x4, s_w[w][(u * NB + q * NW) * 64 + lane]);
        tot[0] += v[0], tot[1] += v[1], tot[2] += v[2], tot[3] += v[3];
        if constexpr (NW == 2) {
          const f32x4 v2 = __builtin_bit_cast(f32x4, s_w[w][(u * NB + q * NW + 1) * 64 + lane]);
          tot2[0] += v2[0], tot2[1] += v2[1], tot2[2] += v2[2], tot2[3] += v2[3];
        }
      }
      const int n = (tile0 + q) * 16 + col;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (u0 + u) + 4 * g + i;
        const bool ok = row < mr && n < N;
        if constexpr (SUMS) {
          if (ok) part[((long long)slice * mr + row) * N + n] = tot[i];
        } else {
          if (ok) epilogue<EPI>(a, row, n, tot[i], tot2[i]);
          if constexpr (EPI == EPI_ARGMAX) {
            float bv = ok ? round_bf16(tot[i]) : -INFINITY;
            int bi = ok ? n : 0x7fffffff;
#define KO_ARG_STEP(CTRL) \
  arg_better(dpp_f<CTRL>(bv), __builtin_amdgcn_update_dpp(0, bi, CTRL, 0xf, 0xf, false), bv, bi);
            KO_ARG_STEP(0x128)
            KO_ARG_STEP(0x124)
            KO_ARG_STEP(0x122)
            KO_ARG_STEP(0x121)
#undef KO_ARG_STEP
            if (col == 0) s_best[row][q] = make_float2(bv, __int_as_float(bi));
          }
        }
      }
    }
  }
  if constexpr (EPI == EPI_ARGMAX) {
    __syncthreads();
    if (t < mr) {
      float2 b = s_best[t][0];
      float bv = b.x;
      int bi = __float_as_int(b.y);
#pragma unroll
      for (int q = 1; q < TN; ++q) arg_better(s_best[t][q].x, __float_as_int(s_best[t][q].y), bv, bi);
      a.part[(long long)t * a.nparts + blockIdx.x] = make_float2(bv, __int_as_float(bi));
    }
  }
}

// One workgroup per row, four columns per thread and round. S > 0: the residual add of the
// S slices' sums in slice order, h <- bf16(h + bf16(sum)), and ss_out[m] += sum(h^2) when
// given. Then, with xn, the next projection's input bf16(nw * bf16(h * rstd)) in the
// operand order of mt row tiles (rstd from ss when given, S = 0). Bound by the launch
// and one memory round trip: 2.8 us at 16 rows of 2560 for the norm alone.
template <int S>
__global__ __launch_bounds__(1024) void row_finish_kernel(const float* __restrict__ part,
                                                          uint16_t* __restrict__ h,
                                                          const uint16_t* __restrict__ nw,
                                                          uint16_t* __restrict__ xn,
                                                          const float* __restrict__ ss,
                                                          float* __restrict__ ss_out, int M,
                                                          int N, int mt, float eps) {
  __shared__ float red[16];
  const int m = blockIdx.x, nc = N >> 2;
  uint16_t* hrow = h + (long long)m * N;
  const bool wide = (reinterpret_cast<uintptr_t>(hrow) & 7) == 0;
  constexpr int R = 2;  // rounds: N <= 8192
  uint2 hv[R], wv[R];
  float sq = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int c = threadIdx.x + r * blockDim.x;
    hv[r] = wv[r] = make_uint2(0, 0);
    if (c < nc) {
      float4 p[S > 0 ? S : 1];
#pragma unroll
      for (int s = 0; s < S; ++s)
        p[s] = *reinterpret_cast<const float4*>(part + ((long long)s * M + m) * N + 4 * c);
      if (wide) {
        hv[r] = *reinterpret_cast<const uint2*>(hrow + 4 * c);
      } else {
        const uint16_t* e = hrow + 4 * c;
        hv[r] = make_uint2(e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16);
      }
      if (xn) wv[r] = *reinterpret_cast<const uint2*>(nw + 4 * c);
      if constexpr (S > 0) {
        float4 v = p[0];
#pragma unroll
        for (int s = 1; s < S; ++s) v.x += p[s].x, v.y += p[s].y, v.z += p[s].z, v.w += p[s].w;
        const uint32_t y0 = pack_bf16x2(v.x, v.y), y1 = pack_bf16x2(v.z, v.w);
        hv[r].x = pack_bf16x2(bf16lo(hv[r].x) + bf16lo(y0), bf16hi(hv[r].x) + bf16hi(y0));
        hv[r].y = pack_bf16x2(bf16lo(hv[r].y) + bf16lo(y1), bf16hi(hv[r].y) + bf16hi(y1));
        if (wide) {
          *reinterpret_cast<uint2*>(hrow + 4 * c) = hv[r];
        } else {
          uint16_t* e = hrow + 4 * c;
          e[0] = (uint16_t)hv[r].x, e[1] = (uint16_t)(hv[r].x >> 16);
          e[2] = (uint16_t)hv[r].y, e[3] = (uint16_t)(hv[r].y >> 16);
        }
      }
      const float e0 = bf16lo(hv[r].x), e1 = bf16hi(hv[r].x), e2 = bf16lo(hv[r].y),
                  e3 = bf16hi(hv[r].y);
      sq += e0 * e0 + e1 * e1 + e2 * e2 + e3 * e3;
    }
  }
  if (!xn && !ss_out) return;
  float tot;
  if (S == 0 && ss) {
    tot = ss[m];
  } else {
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    tot = 0.f;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) tot += red[i];
  }
  if (ss_out && threadIdx.x == 0) atomicAdd(ss_out + m, tot);
  if (!xn) return;
  const float rstd = rsqrtf(tot / (float)N + eps);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int c = threadIdx.x + r * blockDim.x;
    if (c < nc)
      *reinterpret_cast<uint2*>(xn + xt_index(m, 4 * c, mt)) =
          make_uint2(norm2(hv[r].x, wv[r].x, rstd), norm2(hv[r].y, wv[r].y, rstd));
  }
}

template <int S>
int finish(const float* part, uint16_t* h, const uint16_t* nw, uint16_t* xn, const float* ss,
           float* ss_out, int M, int N, float eps, hipStream_t s) {
  const int nt = ((N >> 2) + 63) / 64 * 64;
  hipLaunchKernelGGL((row_finish_kernel<S>), dim3(M), dim3(nt < 1024 ? nt : 1024), 0, s, part, h,
                     nw, xn, ss, ss_out, M, N, (M + 15) / 16, eps);
  return KO_LAUNCH_STATUS();
}

template <int EPI, bool XT, bool SUMS, int MT, int TN, int NS, int PD>
void go(const GemvArgs& a, int slices, float* part, hipStream_t s) {
  const int T = (a.N + 15) / 16;
  hipLaunchKernelGGL((gemm_rows_kernel<EPI, XT, SUMS, MT, TN, NS, PD>),
                     dim3((T + TN - 1) / TN * slices), dim3(64 * RW), 0, s, a, slices,
                     a.K / 32 / slices, part);
}
// P1..P4: the ring's depth with 1..4 row tiles
template <int EPI, bool XT, bool SUMS, int TN, int NS, int P1, int P2, int P3, int P4>
int go_mt(const GemvArgs& a, int slices, float* part, hipStream_t s) {
  switch ((a.mrows + 15) / 16) {
    case 1: go<EPI, XT, SUMS, 1, TN, NS, P1>(a, slices, part, s); break;
    case 2: go<EPI, XT, SUMS, 2, TN, NS, P2>(a, slices, part, s); break;
    case 3: go<EPI, XT, SUMS, 3, TN, NS, P3>(a, slices, part, s); break;
    default: go<EPI, XT, SUMS, 4, TN, NS, P4>(a, slices, part, s); break;
  }
  return KO_LAUNCH_STATUS();
}

}  // namespace

namespace ko {

int launch_layout5(GemvArgs a, int epi, bool norm, int tn, int slices, const RowsChain& chain,
                   float* part, hipStream_t s) {
  if (epi == EPI_RESID) {
    int st = a.K == 4096 ? go_mt<EPI_RESID, false, true, 3, 4, 4, 4, 4, 4>(a, slices, part, s)
                         : go_mt<EPI_RESID, false, true, 3, 10, 8, 6, 4, 2>(a, slices, part, s);
    if (st) return st;
    return finish<4>(part, a.h, chain.next_nw, chain.next_xn, nullptr, a.ss_out, a.mrows, a.N,
                     a.eps, s);
  }
  // x in the operand order: given by the caller's previous projection, or normed here
  uint16_t* xn = reinterpret_cast<uint16_t*>(part);
  if (chain.xn) {
    a.x = chain.xn;
  } else {
    int st = finish<0>(nullptr, const_cast<uint16_t*>(a.x), a.nw, xn, a.ss, nullptr, a.mrows, a.K,
                       a.eps, s);
    if (st) return st;
    a.x = xn;
  }
  switch (epi) {
    case EPI_F32: return go_mt<EPI_F32, true, false, 2, 10, 10, 8, 6, 5>(a, 1, nullptr, s);
    case EPI_BF16: return go_mt<EPI_BF16, true, false, 2, 10, 10, 8, 6, 5>(a, 1, nullptr, s);
    case EPI_SWIGLU: return go_mt<EPI_SWIGLU, true, false, 3, 10, 5, 4, 3, 3>(a, 1, nullptr, s);
    default:
      if (tn == 4) return go_mt<EPI_ARGMAX, true, false, 4, 10, 5, 5, 4, 4>(a, 1, nullptr, s);
      return go_mt<EPI_ARGMAX, true, false, 6, 10, 5, 4, 3, 3>(a, 1, nullptr, s);
  }
}

}  // namespace ko
