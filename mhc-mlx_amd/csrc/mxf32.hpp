// MHCRewire post-combine on fp32 MFMA (v_mfma_f32_16x16x4_f32) for any C,
// alignment and dtypes (mix32.hip takes C a multiple of 64):
//   forward   out = Mf X + p Y                   (Mf_ij = p_i M_ij a_j)
//   backward  dx = Mf^T G,  dy = p G,  S = G X^T,  Yd_i = sum_c G_ic Y_ic
//
// Nothing couples the channels of a token, so a column is a (token, channel)
// pair and a slab is 64 consecutive columns: at C = 32 (MHCRewire's 32 streams
// of a 1024-wide Linear) a slab spans two tokens, where a slab of one token
// would be half padding.  The lane layout within a slab is lf32_fwd.hip's:
// lane (q, r) holds streams krow(m, q) at four columns, the B operand of the
// stream contractions; S takes its operands from the wave's LDS, where G and X
// are written as rows (see lf32_bwd.hpp).  Yd is a lane sum: Y needs no other
// layout.  Waves walk the slabs; the next slab's loads are issued before this
// one's output rows.
//
// 8192 x 32 x 32, bf16 x and y, fp32 out and dout, against the VALU kernels
// before it (one thread per channel, rows of Mf broadcast from LDS), calls
// replayed over two inputs in turn: forward 32 -> 16 us (4.1 TB/s), VJP call
// with its reduction 96 -> 36 us; 8192 x 16 x 128 fp32 36 -> 33 us (6.1 TB/s)
// and 87 -> 64 us; 8192 x 24 x 40 bf16 26 -> 16 us and 536 -> 35 us; 4096 x 64 x
// 32 bf16 60 -> 19 us and 289 -> 76 us.
#pragma once

#include <type_traits>

#include "mhc_device.hpp"
#include "mhc_host.hpp"
#include "mhc_lf32.hpp"
#include "mhc_mxf32.hpp"
#include "mhc_plan.hpp"

namespace mhc {

namespace {

constexpr int kMxfWaves = 4;
constexpr int kMxfPitch = kLfSlab + 4;

// column / C for a column below 2^31
MHC_DEV uint32_t mxf_token(uint32_t col, const MxfArgs& A) { return __umulhi(col << 1, A.cmul) >> A.csh; }

// The lane's columns of a slab: element offset of each from the row of stream 0 of the slab's first token, kLfOut past
// the last column.
template <bool VEC>
struct MxfPos {
  uint32_t e[VEC ? 1 : 4];
  int64_t base;  // element offset of that token (wave-uniform)
  uint32_t left; // elements from there to the tensor's end, capped so that their bytes stay below 2^31
  MHC_DEV void set(const MxfArgs& A, int64_t slab, int r) {
    const uint32_t c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(slab * kLfSlab));
    const uint32_t t0 = mxf_token(c0, A);
    constexpr int64_t kMost = (1 << 29) - 1;
    const int64_t nC = (int64_t)A.n * A.C;
    base = t0 * nC;
    const int64_t rest = A.T * nC - base;
    left = rest < kMost ? (uint32_t)rest : (uint32_t)kMost;
#pragma unroll
    for (int v = 0; v < (VEC ? 1 : 4); ++v) {
      const uint32_t col = c0 + (uint32_t)lf_chan<VEC>(r, v);
      const uint32_t t = mxf_token(col, A);
      e[v] = col < A.cols ? (t - t0) * (uint32_t)nC + (col - t * (uint32_t)A.C) : kLfOut;
    }
  }
  // byte offsets in stream `row` (outside for rows past n)
  MHC_DEV LfOff<VEC> row(int i, int n, int C, int elem) const {
    LfOff<VEC> f;
#pragma unroll
    for (int v = 0; v < (VEC ? 1 : 4); ++v)
      f.o[v] = i < n && e[v] != kLfOut ? (e[v] + (uint32_t)(i * C)) * (uint32_t)elem : kLfOut;
    return f;
  }
};

template <typename T, bool VEC>
MHC_DEV __amdgpu_buffer_rsrc_t mxf_rsrc(const T* p, const MxfPos<VEC>& at) {
  return lf_rsrc(p + at.base, p != nullptr ? at.left * (uint32_t)sizeof(T) : 0u);
}

MHC_DEV float mxf_act(const float* h, int i, int n, int mode, float scale) {
  if (mode == MHC_H_NONE) return i < n ? 1.0f : 0.0f;
  return lf_act(h[i < n ? i : 0], i, n, mode == MHC_H_RAW, scale);
}

template <typename XT, typename YT, typename OT, int NB, int MODE>
__global__ __launch_bounds__(64 * kMxfWaves) void mxf_fwd_kernel(MxfArgs A) {
  constexpr bool VEC = MODE != kLfElem;
  constexpr bool BIG = NB > 2;
  constexpr int NK = 4 * NB;
  constexpr int AUX = lf_aux(MODE);
  __shared__ __align__(16) float4 s_m[BIG ? NB * NB * 64 : 1];
  __shared__ float s_p[BIG ? 16 * NB : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane >> 4, r = lane & 15;
  const int n = A.n, C = A.C;
  auto krow = [&](int m) { return NB == 1 ? 4 * m + q : q * NK + m; };
  const float av = mxf_act(A.hpre, lane, n, A.h_mode, 1.0f), pv = mxf_act(A.hpost, lane, n, A.h_mode, 2.0f);

  float am[BIG ? 1 : NB][NK], p[BIG ? 1 : NB][4];
  if constexpr (BIG) {
    for (int k0 = 0; k0 < NB * NB * 64; k0 += 64 * kMxfWaves) {
      const int k = k0 + (int)threadIdx.x;  // NB * NB waves' worth in steps of four: the last step may be partial
      const int l = k & 63, g = (k >> 6) % NB, i = 16 * ((k >> 6) / NB) + (l & 15), j = (l >> 4) * NK + 4 * g;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = lf_lane(pv, i) * lf_entry(A.M, i, j + e, n) * lf_lane(av, j + e);
      if (k < NB * NB * 64) s_m[k] = make_float4(v[0], v[1], v[2], v[3]);
    }
    if (wave == 0 && lane < 16 * NB) s_p[lane] = pv;
    __syncthreads();
  } else {
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      const float pi = lf_lane(pv, 16 * I + r);
#pragma unroll
      for (int m = 0; m < NK; ++m) am[I][m] = pi * lf_entry(A.M, 16 * I + r, krow(m), n) * lf_lane(av, krow(m));
#pragma unroll
      for (int k = 0; k < 4; ++k) p[I][k] = lf_lane(pv, 16 * I + 4 * q + k);
    }
  }

  const XT* X = (const XT*)A.x;
  const YT* Y = (const YT*)A.y;
  OT* O = (OT*)A.out;
  const int64_t slabs = ((int64_t)A.cols + kLfSlab - 1) / kLfSlab;
  const int64_t stride = (int64_t)gridDim.x * kMxfWaves;
  LfQuad<XT, VEC> x[NK];
  LfQuad<YT, VEC> y[BIG ? 1 : NB][4];
  auto load = [&](const MxfPos<VEC>& at) {
    const auto rx = mxf_rsrc(X, at);
#pragma unroll
    for (int m = 0; m < NK; ++m) x[m].template load<AUX>(rx, at.row(krow(m), n, C, sizeof(XT)), 0);
    if constexpr (!BIG) {
      const auto ry = mxf_rsrc(Y, at);
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int k = 0; k < 4; ++k) y[I][k].template load<AUX>(ry, at.row(16 * I + 4 * q + k, n, C, sizeof(YT)), 0);
    }
  };
  MxfPos<VEC> at;
  int64_t s = (int64_t)blockIdx.x * kMxfWaves + wave;
  if (s >= slabs) return;
  at.set(A, s, r);
  if constexpr (BIG) {
    for (; s < slabs; s += stride) {
      at.set(A, s, r);
      load(at);
      const auto ry = mxf_rsrc(Y, at);
      const auto ro = mxf_rsrc(O, at);
#pragma unroll 1
      for (int I = 0; I < NB; ++I) {
        LfQuad<YT, VEC> yb[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) yb[k].template load<AUX>(ry, at.row(16 * I + 4 * q + k, n, C, sizeof(YT)), 0);
        f32x4 d[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) d[v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < NB; ++g) {
          const float4 m4 = s_m[(I * NB + g) * 64 + lane];
          const float mm[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v) d[v] = lf_mfma(mm[e], x[4 * g + e].get(v), d[v]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float pk = s_p[16 * I + 4 * q + k];
          float o[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = fmaf(pk, yb[k].get(v), d[v][k]);
          lf_store<OT, VEC, AUX>(ro, at.row(16 * I + 4 * q + k, n, C, sizeof(OT)), 0, o);
        }
      }
    }
  } else {
    load(at);
    // (entering the loop with these loads pending would make every iteration's waits as strict as the first's)
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    for (;;) {
      f32x4 d[NB][4];
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int v = 0; v < 4; ++v) d[I][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < NK; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int I = 0; I < NB; ++I) d[I][v] = lf_mfma(am[I][m], x[m].get(v), d[I][v]);
      // y joins last: begun with it, every product of the mix would be rounded against this larger term
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int k = 0; k < 4; ++k) d[I][v][k] = fmaf(p[I][k], y[I][k].get(v), d[I][v][k]);
      const MxfPos<VEC> now = at;
      const bool more = s + stride < slabs;
      if (more) {
        at.set(A, s + stride, r);
        load(at);
      }
      issue_fence();
      const auto ro = mxf_rsrc(O, now);
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float o[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = d[I][v][k];
          lf_store<OT, VEC, AUX>(ro, now.row(16 * I + 4 * q + k, n, C, sizeof(OT)), 0, o);
        }
      if (!more) break;
      s += stride;
    }
  }
}

constexpr int mxf_wave_floats(int nb) { return 2 * 16 * nb * kMxfPitch; }

template <typename XT, typename YT, typename GT, int NB, int MODE>
__global__ __launch_bounds__(64 * kMxfWaves) __attribute__((amdgpu_waves_per_eu(NB > 2 ? 1 : 2)))
void mxf_bwd_kernel(MxfArgs A) {
  constexpr bool VEC = MODE != kLfElem;
  constexpr bool BIG = NB > 2;
  constexpr int NK = 4 * NB;
  constexpr int AUX = lf_aux(MODE);
  extern __shared__ __align__(16) float mxf_smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane >> 4, r = lane & 15;
  const int n = A.n, C = A.C;
  float* sx = mxf_smem + wave * mxf_wave_floats(NB);  // [16 NB][68]
  float* sg = sx + 16 * NB * kMxfPitch;
  float4* s_mt = reinterpret_cast<float4*>(mxf_smem + kMxfWaves * mxf_wave_floats(NB));  // BIG
  auto krow = [&](int m) { return NB == 1 ? 4 * m + q : q * NK + m; };
  const float av = mxf_act(A.hpre, lane, n, A.h_mode, 1.0f), pv = mxf_act(A.hpost, lane, n, A.h_mode, 2.0f);

  // Mf^T: column 16 J + r of Mf at streams krow(m); p of streams krow(m)
  float amt[BIG ? 1 : NB][NK], p[NK];
#pragma unroll
  for (int m = 0; m < NK; ++m) p[m] = lf_lane(pv, krow(m));
  if constexpr (BIG) {
    for (int k0 = 0; k0 < NB * NB * 64; k0 += 64 * kMxfWaves) {
      const int k = k0 + (int)threadIdx.x;
      const int l = k & 63, g = (k >> 6) % NB, j = 16 * ((k >> 6) / NB) + (l & 15), i = (l >> 4) * NK + 4 * g;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = lf_lane(pv, i + e) * lf_entry(A.M, i + e, j, n) * lf_lane(av, j);
      if (k < NB * NB * 64) s_mt[k] = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      const float aj = lf_lane(av, 16 * J + r);
#pragma unroll
      for (int m = 0; m < NK; ++m) amt[J][m] = p[m] * lf_entry(A.M, krow(m), 16 * J + r, n) * aj;
    }
  }

  const XT* X = (const XT*)A.x;
  const YT* Y = (const YT*)A.y;
  const GT* G = (const GT*)A.g;
  XT* DX = (XT*)A.out;
  YT* DY = (YT*)A.dy;
  f32x4 sm[NB][NB];
  float yd[NK];
#pragma unroll
  for (int m = 0; m < NK; ++m) yd[m] = 0.0f;
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int J = 0; J < NB; ++J) sm[I][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int64_t slabs = ((int64_t)A.cols + kLfSlab - 1) / kLfSlab;
  const int64_t stride = (int64_t)gridDim.x * kMxfWaves;
  LfQuad<XT, VEC> x[NK];
  LfQuad<GT, VEC> g[NK];
  LfQuad<YT, VEC> y[NK];
  auto load = [&](const MxfPos<VEC>& at) {
    const auto rx = mxf_rsrc(X, at);
    const auto rg = mxf_rsrc(G, at);
    const auto ry = mxf_rsrc(Y, at);
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      g[m].template load<AUX>(rg, at.row(krow(m), n, C, sizeof(GT)), 0);
      x[m].template load<AUX>(rx, at.row(krow(m), n, C, sizeof(XT)), 0);
      y[m].template load<AUX>(ry, at.row(krow(m), n, C, sizeof(YT)), 0);
    }
  };
  // Yd, dy and the slab's rows into LDS
  auto take = [&](const MxfPos<VEC>& at) {
    const auto rdy = mxf_rsrc(DY, at);
    issue_fence();  // the previous slab's reads stay ahead of these writes
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        yd[m] = fmaf(g[m].get(v), y[m].get(v), yd[m]);
        o[v] = p[m] * g[m].get(v);
      }
      lf_store<YT, VEC, AUX>(rdy, at.row(krow(m), n, C, sizeof(YT)), 0, o);
      float* px = sx + krow(m) * kMxfPitch;
      float* pg = sg + krow(m) * kMxfPitch;
      if constexpr (VEC) {
        *reinterpret_cast<float4*>(px + 4 * r) = make_float4(x[m].get(0), x[m].get(1), x[m].get(2), x[m].get(3));
        *reinterpret_cast<float4*>(pg + 4 * r) = make_float4(g[m].get(0), g[m].get(1), g[m].get(2), g[m].get(3));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          px[lf_chan<VEC>(r, v)] = x[m].get(v);
          pg[lf_chan<VEC>(r, v)] = g[m].get(v);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < NK; ++m) asm volatile("" : "+v"(yd[m]));  // formed here, not where the sums end
    issue_fence();
  };
  // (a row block of G at a time, a slab's products in chains of 16: see lf32_bwd.hpp)
  auto sums = [&] {
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      f32x4 part[2][NB];
#pragma unroll
      for (int J = 0; J < NB; ++J) part[0][J] = part[1][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        const int c = 16 * k + 4 * q;
        const f32x4 gv = *reinterpret_cast<const f32x4*>(sg + (16 * I + r) * kMxfPitch + c);
        f32x4 xv[NB];
#pragma unroll
        for (int J = 0; J < NB; ++J) xv[J] = *reinterpret_cast<const f32x4*>(sx + (16 * J + r) * kMxfPitch + c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int J = 0; J < NB; ++J) part[e & 1][J] = lf_mfma(gv[e], xv[J][e], part[e & 1][J]);
        if (k == 1) {
#pragma unroll
          for (int J = 0; J < NB; ++J) {
            sm[I][J] += part[0][J] + part[1][J];
            part[0][J] = part[1][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
        }
      }
#pragma unroll
      for (int J = 0; J < NB; ++J) sm[I][J] += part[0][J] + part[1][J];
    }
  };

  int64_t s = (int64_t)blockIdx.x * kMxfWaves + wave;
  MxfPos<VEC> at;
  if (s < slabs) {
    at.set(A, s, r);
    if constexpr (!BIG) {
      load(at);
      __builtin_amdgcn_s_waitcnt(kWaitVm0);
    }
  }
  while (s < slabs) {
    const bool more = s + stride < slabs;
    if constexpr (BIG) {
      load(at);
      take(at);
      sums();
      const auto ro = mxf_rsrc(DX, at);
#pragma unroll 1
      for (int J = 0; J < NB; ++J) {
        f32x4 d[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) d[v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const float4 m4 = s_mt[(J * NB + k) * 64 + lane];
          const float mm[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v) d[v] = lf_mfma(mm[e], g[4 * k + e].get(v), d[v]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float o[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = d[v][k];
          lf_store<XT, VEC, AUX>(ro, at.row(16 * J + 4 * q + k, n, C, sizeof(XT)), 0, o);
        }
      }
      if (more) at.set(A, s + stride, r);
    } else {
      take(at);
      f32x4 d[NB][4];
#pragma unroll
      for (int J = 0; J < NB; ++J)
#pragma unroll
        for (int v = 0; v < 4; ++v) d[J][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < NK; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int J = 0; J < NB; ++J) d[J][v] = lf_mfma(amt[J][m], g[m].get(v), d[J][v]);
      const MxfPos<VEC> now = at;
      if (more) {
        at.set(A, s + stride, r);
        load(at);
      }
      issue_fence();
      sums();
      const auto ro = mxf_rsrc(DX, now);
#pragma unroll
      for (int J = 0; J < NB; ++J)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float o[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = d[J][v][k];
          lf_store<XT, VEC, AUX>(ro, now.row(16 * J + 4 * q + k, n, C, sizeof(XT)), 0, o);
        }
    }
    s += stride;
  }

  // ---- the workgroup's partial row [S n*n | Yd n | 0 ..]; the waves' sums are added in wave order
  issue_fence();
  constexpr int NM = 256 * NB * NB;
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int k = 0; k < 4; ++k) sx[(16 * I + 4 * q + k) * (16 * NB) + 16 * J + r] = sm[I][J][k];
#pragma unroll
  for (int m = 0; m < NK; ++m) {
    const float v = group_sum<16>(yd[m]);
    if (r == 0) sx[NM + krow(m)] = v;
  }
  __syncthreads();
  float* prow = A.part + (int64_t)blockIdx.x * A.P;
  const int nn = n * n;
  for (int k = threadIdx.x; k < A.P; k += blockDim.x) {
    const int from = k < nn ? (k / n) * (16 * NB) + k % n : NM + k - nn;
    float v = 0.0f;
    if (k < nn + n)
      for (int w = 0; w < kMxfWaves; ++w) v += mxf_smem[w * mxf_wave_floats(NB) + from];
    prow[k] = v;
  }
}

template <int NB, typename F>
int mxf_by_mode(int mode, F&& f) {
  if (mode == kLfLine) return f(std::integral_constant<int, NB>{}, std::integral_constant<int, kLfLine>{});
  if (mode == kLfVec) return f(std::integral_constant<int, NB>{}, std::integral_constant<int, kLfVec>{});
  return f(std::integral_constant<int, NB>{}, std::integral_constant<int, kLfElem>{});
}

template <typename F>
int mxf_by_shape(int n, int mode, F&& f) {
  if (n <= 16) return mxf_by_mode<1>(mode, f);
  if (n <= 32) return mxf_by_mode<2>(mode, f);
  if (n <= 48) return mxf_by_mode<3>(mode, f);
  return mxf_by_mode<4>(mode, f);
}

// resident workgroups, at most one wave per slab
inline int64_t mxf_blocks(const MxfArgs& A, const void* kfn, size_t smem, Knob k, int64_t most) {
  const int occ = occupancy_blocks(kfn, 64 * kMxfWaves, smem);
  if (occ <= 0) return 0;
  const int pref = knob(k, 0);
  int64_t blocks = (int64_t)device_cu_count() * (pref > 0 ? pref : occ);
  blocks = std::min(blocks, ceil_div(ceil_div((int64_t)A.cols, kLfSlab), kMxfWaves));
  return std::max<int64_t>(1, std::min(blocks, most));
}

template <typename XT, typename YT, typename OT>
int mxf_fwd_typed(const MxfArgs& A, hipStream_t s) {
  const int mode = std::min(lf_mode(A.C, sizeof(XT), sizeof(OT), aligned(A.x, 4 * sizeof(XT)) && aligned(A.out, 4 * sizeof(OT))),
                            lf_mode(A.C, sizeof(XT), sizeof(YT), aligned(A.y, 4 * sizeof(YT))));
  return mxf_by_shape(A.n, mode, [&](auto nb, auto md) {
    constexpr int NB = decltype(nb)::value, MODE = decltype(md)::value;
    const int64_t blocks = mxf_blocks(A, (const void*)mxf_fwd_kernel<XT, YT, OT, NB, MODE>, 0, kKnobMixFwdGrid, kMaxGrid);
    if (blocks == 0) return 1;
    hipLaunchKernelGGL((mxf_fwd_kernel<XT, YT, OT, NB, MODE>), dim3((unsigned)blocks), dim3(64 * kMxfWaves), 0, s, A);
    MHC_CHECK_LAUNCH("mxf_fwd_kernel");
    return (int)MHC_OK;
  });
}

template <typename XT, typename YT, typename GT>
int mxf_bwd_typed(const MxfArgs& A, int64_t gmax, hipStream_t s, int64_t* np) {
  const int mode = std::min(lf_mode(A.C, sizeof(XT), sizeof(GT), aligned(A.x, 4 * sizeof(XT)) && aligned(A.out, 4 * sizeof(XT)) &&
                                                                     aligned(A.g, 4 * sizeof(GT))),
                            lf_mode(A.C, sizeof(XT), sizeof(YT), aligned(A.y, 4 * sizeof(YT)) && aligned(A.dy, 4 * sizeof(YT))));
  return mxf_by_shape(A.n, mode, [&](auto nb, auto md) {
    constexpr int NB = decltype(nb)::value, MODE = decltype(md)::value;
    const size_t smem = (size_t)(kMxfWaves * mxf_wave_floats(NB) + (NB > 2 ? NB * NB * 256 : 0)) * sizeof(float);
    const void* kfn = (const void*)mxf_bwd_kernel<XT, YT, GT, NB, MODE>;
    const int64_t blocks = mxf_blocks(A, kfn, smem, kKnobMixBwdGrid, gmax);
    if (blocks == 0) return 1;
    hipLaunchKernelGGL((mxf_bwd_kernel<XT, YT, GT, NB, MODE>), dim3((unsigned)blocks), dim3(64 * kMxfWaves), smem, s, A);
    MHC_CHECK_LAUNCH("mxf_bwd_kernel");
    *np = blocks;
    return (int)MHC_OK;
  });
}

// y and out / dout of x's dtype or fp32
template <typename XT>
int mxf_fwd_types(const MxfArgs& A, bool y_f32, bool o_f32, hipStream_t s) {
  if constexpr (std::is_same<XT, float>::value) {
    return mxf_fwd_typed<float, float, float>(A, s);
  } else {
    if (y_f32) return o_f32 ? mxf_fwd_typed<XT, float, float>(A, s) : mxf_fwd_typed<XT, float, XT>(A, s);
    return o_f32 ? mxf_fwd_typed<XT, XT, float>(A, s) : mxf_fwd_typed<XT, XT, XT>(A, s);
  }
}

template <typename XT>
int mxf_bwd_types(const MxfArgs& A, bool y_f32, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  if constexpr (std::is_same<XT, float>::value) {
    return mxf_bwd_typed<float, float, float>(A, gmax, s, np);
  } else {
    if (y_f32) return g_f32 ? mxf_bwd_typed<XT, float, float>(A, gmax, s, np) : mxf_bwd_typed<XT, float, XT>(A, gmax, s, np);
    return g_f32 ? mxf_bwd_typed<XT, XT, float>(A, gmax, s, np) : mxf_bwd_typed<XT, XT, XT>(A, gmax, s, np);
  }
}

}  // namespace

}  // namespace mhc
