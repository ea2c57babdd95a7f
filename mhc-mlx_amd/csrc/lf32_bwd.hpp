// Backward of the layer on fp32 MFMA (v_mfma_f32_16x16x4_f32), 8 < n <= 64,
// any C, fp32 or 16-bit x, dout of x's dtype or fp32.  Per token, with
// y = a^T x, d = p^T g, inv and kf the token's RMS scalars:
//   dy = d inv w - kf y,   dx = M^T g + a dy,   dw += d y inv,
//   dM += g x^T,   dA_i = sum dy x_i,   dP_i = sum g_i y inv w.
//
// Two contractions of n^2 FMAs per channel, over streams (M^T g) and over
// channels (g x^T); on the VALU against LDS broadcasts they held the kernel to
// 4-27% of HBM.  On the fp32 matrix cores they take about 40% of the time
// that reading x and g and writing dx takes at n = 32 in fp32, so the kernel
// is laid out to touch each of them once.
//
// A slab is 64 channels of every stream.  The wave loads it in the stream
// layout of the forward (lane (q, r): streams krow(m, q), four channels):
// y, d, and M^T g with g as the B operand.  The channel contraction needs
// the other layout (lane (q, r): streams 16 I + r, channels 16 k + 4q ..+3 as
// A and B operands), so the wave writes x and g as fp32 rows into its own LDS
// (pitch 68: 4 banks between rows, no conflicts in either direction) and
// reads them back as 16-byte pieces.
//
// No sum needs the token after the RMS barrier:
//   dA_i = inv sum d w x_i - kf sum y x_i,   dP_i = inv sum y w g_i
// are formed as lane partials from the same LDS reads that feed g x^T and
// scaled per token, so x is read once.
//
// SPW > 0 (layer-wide, n <= 32): M^T g of the wave's SPW slabs is held across
// the barrier and the next token's x and g are loaded meanwhile.  SPW = 0: the
// wave walks any number of slabs, y and d in LDS, and reads g again after the
// barrier (from the caches).  Per-token parameters take SPW = 0, with one wave
// per workgroup where there are tokens enough to fill the chip (the token's
// dM, dA and dP are then the wave's own), else up to four.  Above
// n = 32 (BIG) M^T's operands come from LDS, one 16-row block at a time.
//
// Backward kernel, against the VALU kernels before it, calls replayed over two
// inputs in turn: 4096 x 32 x 512 fp32 1360 -> 152 us (5.3 TB/s), 4096 x 16 x
// 1024 fp32 385 -> 141 us (5.7 TB/s), 2048 x 64 x 512 fp32 4138 -> 321 us (one
// wave per SIMD: dM alone is 64 registers), 1024 x 32 x 4096 fp32 3233 -> 430 us
// (g read twice), per token 4096 x 32 x 512 fp32 1367 -> 186 us and 2500 x 10 x
// 4000 fp32 750 -> 369 us, 3001 x 16 x 1100 fp16 346 -> 90 us and 20000 x 24 x
// 100 bf16 1990 -> 128 us (16-bit rows: bound by the VALU's conversions and LDS).
#pragma once

#include <type_traits>

#include "mhc_device.hpp"
#include "mhc_generic.hpp"
#include "mhc_host.hpp"
#include "mhc_lf32.hpp"
#include "mhc_plan.hpp"

namespace mhc {

namespace {

constexpr int kLfPitch = kLfSlab + 4;
constexpr int kLfPtWaves = 4;  // waves per token at most with per-token parameters
// floats of one wave's LDS: x rows, g rows, and y, d w, y w of a slab
constexpr int lf_wave_floats(int nb) { return 2 * 16 * nb * kLfPitch + 3 * kLfSlab; }
// floats of M^T's operands (BIG)
constexpr int lf_mat_floats(int nb) { return nb > 2 ? nb * nb * 256 + 16 * nb : 0; }

template <typename XT, typename GT, int NB, int SPW, int MODE, bool PT>
__global__ __launch_bounds__(PT ? 64 * kLfPtWaves : (NB > 2 ? 256 : 64 * kLfMaxWaves)) void lf32_bwd_kernel(GenArgs A) {
  constexpr bool VEC = MODE != kLfElem;
  constexpr int NK = 4 * NB;
  constexpr int NJ = SPW > 0 ? SPW : 1;
  constexpr bool BIG = NB > 2;
  static_assert(SPW == 0 || (!BIG && !PT), "slabs held in registers: layer-wide, n <= 32");
  extern __shared__ __align__(16) float lf_smem[];
  __shared__ float s_red[2][2][kLfMaxWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = __builtin_amdgcn_readfirstlane(blockDim.x >> 6);
  const int q = lane >> 4, r = lane & 15;
  const int n = A.n, C = A.C, nn = n * n, S = (C + kLfSlab - 1) / kLfSlab;
  const uint32_t rowx = (uint32_t)C * sizeof(XT), rowg = (uint32_t)C * sizeof(GT);
  const uint32_t xbytes = (uint32_t)n * rowx, gbytes = (uint32_t)n * rowg;
  const int64_t tile = (int64_t)n * C;
  const XT* X = (const XT*)A.x;
  const GT* G = (const GT*)A.g;
  XT* DX = (XT*)A.out;
  const bool raw = A.h_mode == MHC_H_RAW;
  auto krow = [&](int m) { return NB == 1 ? 4 * m + q : q * NK + m; };
  const uint32_t xstep = NB == 1 ? 4u * rowx : rowx, gstep = NB == 1 ? 4u * rowg : rowg;

  // ---- LDS
  float* sx = lf_smem + wave * lf_wave_floats(NB);  // [16 NB][68]
  float* sg = sx + 16 * NB * kLfPitch;
  float* sc = sg + 16 * NB * kLfPitch;              // y, d w, y w of the slab: [3][64]
  float* s_mat = lf_smem + nw * lf_wave_floats(NB);
  const float4* s_mt = reinterpret_cast<const float4*>(s_mat);  // BIG: [row block][steps 4g..][lane]
  float* s_a = s_mat + NB * NB * 256;                           // BIG: a [16 NB]
  float* s_y = s_mat + lf_mat_floats(NB);                       // SPW = 0: y, d and dw of the token
  float* s_d = s_y + S * kLfSlab;
  float* s_dw = s_d + S * kLfSlab;

  // ---- parameters
  float a[NK], p[NK], ad[BIG ? 1 : NB][4], amt[BIG ? 1 : NB][NK];
  float av, pv;  // a and p of stream `lane`
  auto load_params = [&](int64_t t) {
    const float* M = A.M + t * A.M_ts;
    av = lf_act(A.hpre[t * A.h_ts + (lane < n ? lane : 0)], lane, n, raw, 1.0f);
    pv = lf_act(A.hpost[t * A.h_ts + (lane < n ? lane : 0)], lane, n, raw, 2.0f);
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      a[m] = lf_lane(av, krow(m));
      p[m] = lf_lane(pv, krow(m));
    }
    if constexpr (BIG) {
      __syncthreads();
      for (int k = threadIdx.x; k < NB * NB * 64; k += blockDim.x) {
        const int l = k & 63, g = (k >> 6) % NB, j = 16 * ((k >> 6) / NB) + (l & 15), i = (l >> 4) * NK + 4 * g;
        reinterpret_cast<float4*>(s_mat)[k] = make_float4(lf_entry(M, i, j, n), lf_entry(M, i + 1, j, n),
                                                          lf_entry(M, i + 2, j, n), lf_entry(M, i + 3, j, n));
      }
      if (wave == 0 && lane < 16 * NB) s_a[lane] = av;
      __syncthreads();
    }
  };
  // M^T's operands and a of the output rows (n <= 32; per token they are loaded after the pass over x and g)
  auto load_mat = [&](int64_t t) {
    const float* M = A.M + t * A.M_ts;
#pragma unroll
    for (int J = 0; J < (BIG ? 0 : NB); ++J) {
#pragma unroll
      for (int m = 0; m < NK; ++m) amt[J][m] = lf_entry(M, krow(m), 16 * J + r, n);
#pragma unroll
      for (int k = 0; k < 4; ++k) ad[J][k] = lf_lane(av, 16 * J + 4 * q + k);
    }
  };
  if constexpr (!PT) {
    load_params(0);
    load_mat(0);
  }

  // ---- sums of the wave: dM blocks (rows 16 I + 4q + k, column 16 J + r); dA, dP of streams 16 I + r over the lane's
  // channels; the token's parts of them before the RMS scalars are known
  f32x4 dm[NB][NB];
  float da[NB], dp[NB], ux[NB], vx[NB], ug[NB];
#pragma unroll
  for (int I = 0; I < NB; ++I) {
    da[I] = dp[I] = 0.0f;
#pragma unroll
    for (int J = 0; J < NB; ++J) dm[I][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }

  LfQuad<XT, VEC> x[NJ][NK];
  LfQuad<GT, VEC> g[NJ][NK];
  auto load_w = [&](int s, float (&w)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = s * kLfSlab + lf_chan<VEC>(r, v);
      w[v] = A.w[c < C ? c : 0];
    }
  };
  auto load_x = [&](int j, __amdgpu_buffer_rsrc_t rs, const LfOff<VEC>& off) {
    const LfOff<VEC> f = off.fresh();
#pragma unroll
    for (int m = 0; m < NK; ++m) x[j][m].template load<lf_aux(MODE)>(rs, f, (uint32_t)m * xstep);
  };
  auto load_g = [&](auto aux, int j, __amdgpu_buffer_rsrc_t rs, const LfOff<VEC>& off) {
    const LfOff<VEC> f = off.fresh();
#pragma unroll
    for (int m = 0; m < NK; ++m) g[j][m].template load<decltype(aux)::value>(rs, f, (uint32_t)m * gstep);
  };
  constexpr std::integral_constant<int, 0> kKeep{};
  constexpr std::integral_constant<int, lf_aux(MODE)> kOnce{};

  // y and d of the slab, its rows into LDS, and the token's two sums
  auto take = [&](int j, const float (&w)[4], float (&y)[4], float (&d)[4], float& ss, float& sr) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float ys = 0.0f, ds = 0.0f;
#pragma unroll
      for (int m = 0; m < NK; ++m) {
        ys = fmaf(a[m], x[j][m].get(v), ys);
        ds = fmaf(p[m], g[j][m].get(v), ds);
      }
      y[v] = lf_sum_q(ys);
      d[v] = lf_sum_q(ds);
      ss = fmaf(y[v], y[v], ss);
      sr = fmaf(d[v] * y[v], w[v], sr);
    }
    issue_fence();  // the previous slab's reads stay ahead of these writes
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      float* px = sx + krow(m) * kLfPitch;
      float* pg = sg + krow(m) * kLfPitch;
      if constexpr (VEC) {
        *reinterpret_cast<float4*>(px + 4 * r) = make_float4(x[j][m].get(0), x[j][m].get(1), x[j][m].get(2), x[j][m].get(3));
        *reinterpret_cast<float4*>(pg + 4 * r) = make_float4(g[j][m].get(0), g[j][m].get(1), g[j][m].get(2), g[j][m].get(3));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          px[lf_chan<VEC>(r, v)] = x[j][m].get(v);
          pg[lf_chan<VEC>(r, v)] = g[j][m].get(v);
        }
      }
    }
    if (q == 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int c = lf_chan<VEC>(r, v);
        sc[c] = y[v];
        sc[kLfSlab + c] = d[v] * w[v];
        sc[2 * kLfSlab + c] = y[v] * w[v];
      }
    }
    issue_fence();
  };
  // dM and the dot products over the slab in LDS, one row block of g at a time (so that the partial sums are few).  A
  // slab's products are summed in four chains of 16, and only their sum joins the wave's: one chain over all of a wave's
  // slabs would round every product against the whole sum (dH_res at 30000 x 9 x 400 bf16 1.8e-6 off the exact sum), one
  // over a slab against the slab's (dM at 130 x 64 x 512 fp32 1.7e-7 off float64, here 1.2e-7, on the VALU kernel 1.1e-7;
  // at n = 32, with two chains, 1.8e-7, 1.4e-7 and 1.2e-7).  Prefetched slabs leave registers for two chains of 32, with
  // SPW = 1 at n <= 16 for one, added at half a slab and at its end (a second one would cost a wave per SIMD), and three
  // slabs of mixed types for the one of 64 (C > 1024, where the VALU kernel's dM is 2.7e-7 off).  Against one chain:
  // 4096 x 32 x 512 fp32 149 -> 151 us, 2048 x 64 x 512 299 -> 318, 2048 x 48 x 512 172 -> 181.
  constexpr bool kHalf = NB == 1 && SPW == 1;
  constexpr int kChains = SPW == 0 ? 4 : (kHalf || (NB == 1 && SPW == 3 && sizeof(XT) != sizeof(GT)) ? 1 : 2);
  auto sums = [&] {
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      f32x4 part[kChains][NB];
#pragma unroll
      for (int h = 0; h < kChains; ++h)
#pragma unroll
        for (int J = 0; J < NB; ++J) part[h][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        __builtin_amdgcn_sched_barrier(0);  // the four steps' operands at once would take 80-112 registers
        const int c = 16 * k + 4 * q;
        const f32x4 gv = *reinterpret_cast<const f32x4*>(sg + (16 * I + r) * kLfPitch + c);
        f32x4 xv[NB];
#pragma unroll
        for (int J = 0; J < NB; ++J) xv[J] = *reinterpret_cast<const f32x4*>(sx + (16 * J + r) * kLfPitch + c);
        const f32x4 yv = *reinterpret_cast<const f32x4*>(sc + c);
        const f32x4 dw = *reinterpret_cast<const f32x4*>(sc + kLfSlab + c);
        const f32x4 yw = *reinterpret_cast<const f32x4*>(sc + 2 * kLfSlab + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int J = 0; J < NB; ++J) part[e % kChains][J] = lf_mfma(gv[e], xv[J][e], part[e % kChains][J]);
          ug[I] = fmaf(gv[e], yw[e], ug[I]);
          if (I == 0) {
#pragma unroll
            for (int J = 0; J < NB; ++J) {
              ux[J] = fmaf(xv[J][e], dw[e], ux[J]);
              vx[J] = fmaf(xv[J][e], yv[e], vx[J]);
            }
          }
        }
        // the dot products stay here: moved to their use after the barrier they would hold every operand until then
#pragma unroll
        for (int J = 0; J < NB; ++J) asm volatile("" : "+v"(ux[J]), "+v"(vx[J]), "+v"(ug[J]));
        if (kHalf && k == 1) {
          dm[0][0] += part[0][0];
          part[0][0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
#pragma unroll
      for (int J = 0; J < NB; ++J) {
        if constexpr (kChains == 4) dm[I][J] += (part[0][J] + part[1][J]) + (part[2][J] + part[3][J]);
        else if constexpr (kChains == 2) dm[I][J] += part[0][J] + part[1][J];
        else dm[I][J] += part[0][J];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // M^T g of g[j] (n <= 32)
  auto mix = [&](int j, f32x4 (&dd)[NB][4]) {
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) dd[J][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < NK; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float b = g[j][m].get(v);
#pragma unroll
        for (int J = 0; J < NB; ++J) dd[J][v] = lf_mfma(amt[J][m], b, dd[J][v]);
      }
  };
  auto store_rows = [&](const f32x4 (&dd)[4], const float (&a4)[4], const float (&dy)[4], int J,
                        __amdgpu_buffer_rsrc_t ro, const LfOff<VEC>& off) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = fmaf(a4[k], dy[v], dd[v][k]);
      lf_store<XT, VEC, lf_aux(MODE)>(ro, off.fresh(), (uint32_t)(16 * J + k) * rowx, o);
    }
  };
  // the token's RMS scalars from the waves' sums (one barrier; the buffers alternate), and its dA, dP
  float inv, kf;
  auto rms = [&](float ss, float sr, int it) {
    ss = group_sum<16>(ss);
    sr = group_sum<16>(sr);
    if (lane == 0) {
      s_red[it & 1][0][wave] = ss;
      s_red[it & 1][1][wave] = sr;
    }
    lds_barrier();
    float tss = 0.0f, tsr = 0.0f;
    for (int k = 0; k < nw; ++k) {
      tss += s_red[it & 1][0][k];
      tsr += s_red[it & 1][1][k];
    }
    inv = 1.0f / sqrtf(tss / (float)C + A.eps);
    kf = (inv * inv * inv / (float)C) * tsr;
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      da[I] += inv * ux[I] - kf * vx[I];
      dp[I] += inv * ug[I];
    }
  };

  // the wave's dM, dA and dP into its LDS, and their sum over the waves (entry k of [dM n*n | dA n | dP n])
  constexpr int NM = 256 * NB * NB;
  auto spill_sums = [&] {
    issue_fence();  // the wave's rows in LDS are done with
#pragma unroll
    for (int I = 0; I < NB; ++I) {
#pragma unroll
      for (int J = 0; J < NB; ++J)
#pragma unroll
        for (int k = 0; k < 4; ++k) sx[(16 * I + 4 * q + k) * (16 * NB) + 16 * J + r] = dm[I][J][k];
      const float va = lf_sum_q(da[I]), vp = lf_sum_q(dp[I]);
      if (q == 0) {
        sx[NM + 16 * I + r] = va;
        sx[NM + 16 * NB + 16 * I + r] = vp;
      }
    }
  };
  auto wave_total = [&](int k) {
    const int at = k < nn ? (k / n) * (16 * NB) + k % n : (k < nn + n ? NM + k - nn : NM + 16 * NB + k - nn - n);
    float v = 0.0f;
    for (int wv = 0; wv < nw; ++wv) v += lf_smem[wv * lf_wave_floats(NB) + at];
    return v;
  };

  int it = 0;
  float dwr[NJ][4];
  if constexpr (SPW > 0) {
    LfOff<VEC> ix[NJ], ig[NJ], io[NJ];
    float w[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int s = wave + j * nw;
      ix[j].set((uint32_t)krow(0) * rowx, s, r, C, sizeof(XT));
      ig[j].set((uint32_t)krow(0) * rowg, s, r, C, sizeof(GT));
      io[j].set((uint32_t)(4 * q) * rowx, s, r, C, sizeof(XT));
      load_w(s, w[j]);
#pragma unroll
      for (int v = 0; v < 4; ++v) dwr[j][v] = 0.0f;
    }
    auto load = [&](int j, int64_t t) {
      const int64_t at = (t < A.T ? t : 0) * tile;
      load_x(j, lf_rsrc(X + at, t < A.T ? xbytes : 0u), ix[j]);
      load_g(kOnce, j, lf_rsrc(G + at, t < A.T ? gbytes : 0u), ig[j]);
    };
#pragma unroll
    for (int j = 0; j < NJ; ++j) load(j, blockIdx.x);
    // (entering the loop with these loads pending would make every iteration's waits as strict as the first's)
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    for (int64_t t = blockIdx.x; t < A.T; t += gridDim.x, ++it) {
      float y[NJ][4], d[NJ][4], ss = 0.0f, sr = 0.0f;
      f32x4 dd[NJ][NB][4];
#pragma unroll
      for (int I = 0; I < NB; ++I) ux[I] = vx[I] = ug[I] = 0.0f;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        take(j, w[j], y[j], d[j], ss, sr);
        mix(j, dd[j]);
        load(j, t + gridDim.x);
        issue_fence();
        sums();
      }
      rms(ss, sr, it);
      const auto ro = lf_rsrc(DX + t * tile, xbytes);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        float dy[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          dy[v] = d[j][v] * inv * w[j][v] - kf * y[j][v];
          dwr[j][v] = fmaf(d[j][v], y[j][v] * inv, dwr[j][v]);
        }
#pragma unroll
        for (int J = 0; J < NB; ++J) store_rows(dd[j][J], ad[J], dy, J, ro, io[j]);
      }
    }
  } else {
    for (int c = threadIdx.x; c < S * kLfSlab; c += blockDim.x) s_dw[c] = 0.0f;
    __syncthreads();
    for (int64_t t = blockIdx.x; t < A.T; t += gridDim.x, ++it) {
      if constexpr (PT) {
        load_params(t);
#pragma unroll
        for (int I = 0; I < NB; ++I) {
          da[I] = dp[I] = 0.0f;
#pragma unroll
          for (int J = 0; J < NB; ++J) dm[I][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      const auto rx = lf_rsrc(X + t * tile, xbytes);
      const auto rg = lf_rsrc(G + t * tile, gbytes);
      const auto ro = lf_rsrc(DX + t * tile, xbytes);
      auto load_gs = [&](auto aux, int s) {
        LfOff<VEC> off;
        off.set((uint32_t)krow(0) * rowg, s, r, C, sizeof(GT));
        load_g(aux, 0, rg, off);
      };
      auto load_xs = [&](int s) {
        LfOff<VEC> off;
        off.set((uint32_t)krow(0) * rowx, s, r, C, sizeof(XT));
        load_x(0, rx, off);
      };
      float ss = 0.0f, sr = 0.0f;
#pragma unroll
      for (int I = 0; I < NB; ++I) ux[I] = vx[I] = ug[I] = 0.0f;
      load_xs(wave);
      load_gs(kKeep, wave);
      for (int s = wave; s < S; s += nw) {
        float y[4], d[4], w[4];
        load_w(s, w);
        take(0, w, y, d, ss, sr);
        if (s + nw < S) {
          load_xs(s + nw);
          load_gs(kKeep, s + nw);
        }
        if (q == 0) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            s_y[s * kLfSlab + lf_chan<VEC>(r, v)] = y[v];
            s_d[s * kLfSlab + lf_chan<VEC>(r, v)] = d[v];
          }
        }
        issue_fence();
        sums();
      }
      load_gs(kOnce, wave);
      if constexpr (PT) load_mat(t);
      rms(ss, sr, it);
      if constexpr (PT) {
        // the waves' parts through their slab rows (done with until the next token), added in wave order
        spill_sums();
        lds_barrier();
        for (int k = threadIdx.x; k < nn + 2 * n; k += blockDim.x) {
          float v = wave_total(k);
          if (k < nn) {
            A.dM_tok[t * nn + k] = v;
          } else {
            const bool post = k >= nn + n;
            const int i = k - nn - (post ? n : 0);
            if (raw) {
              const float sg = sigmoidf_((post ? A.hpost : A.hpre)[t * A.h_ts + i]);
              v *= (post ? 2.0f : 1.0f) * sg * (1.0f - sg);
            }
            (post ? A.dpost_tok : A.dpre_tok)[t * n + i] = v;
          }
        }
        lds_barrier();
      }
      for (int s = wave; s < S; s += nw) {
        float dy[4], w[4];
        load_w(s, w);
#pragma unroll
        for (int v = 0; v < 4; ++v) {  // the wave's own values
          const int c = s * kLfSlab + lf_chan<VEC>(r, v);
          const float y = s_y[c], d = s_d[c];
          dy[v] = d * inv * w[v] - kf * y;
          if (q == 0) s_dw[c] = fmaf(d, y * inv, s_dw[c]);
        }
        LfOff<VEC> io;
        io.set((uint32_t)(4 * q) * rowx, s, r, C, sizeof(XT));
        if constexpr (BIG) {
#pragma unroll 1
          for (int J = 0; J < NB; ++J) {
            f32x4 dd[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) dd[v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < NB; ++k) {
              const float4 m4 = s_mt[(J * NB + k) * 64 + lane];
              const float mm[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
              for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) dd[v] = lf_mfma(mm[e], g[0][4 * k + e].get(v), dd[v]);
            }
            float a4[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) a4[k] = s_a[16 * J + 4 * q + k];
            store_rows(dd, a4, dy, J, ro, io);
          }
          if (s + nw < S) load_gs(kOnce, s + nw);
        } else {
          f32x4 dd[NB][4];
          mix(0, dd);
          if (s + nw < S) load_gs(kOnce, s + nw);
          issue_fence();
#pragma unroll
          for (int J = 0; J < NB; ++J) store_rows(dd[J], ad[J], dy, J, ro, io);
        }
      }
    }
  }

  // ---- the workgroup's partial row [dw C | 0 .. Cp | dM | dA | dP]; the waves' sums are added in wave order
  float* prow = A.part + (int64_t)blockIdx.x * A.P;
  if constexpr (SPW > 0) {
    if (q == 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int c = (wave + j * nw) * kLfSlab + lf_chan<VEC>(r, v);
          if (c < C) prow[c] = dwr[j][v];
        }
    }
    for (int c = C + (int)threadIdx.x; c < A.Cp; c += blockDim.x) prow[c] = 0.0f;
  } else {
    __syncthreads();
    for (int c = threadIdx.x; c < A.Cp; c += blockDim.x) prow[c] = c < C ? s_dw[c] : 0.0f;
  }
  if constexpr (!PT) {
    spill_sums();
    __syncthreads();
    for (int k = threadIdx.x; k < nn + 2 * n; k += blockDim.x) prow[A.Cp + k] = wave_total(k);
  }
}

// bytes of a workgroup's LDS; `loop`: SPW = 0
inline size_t lf_bwd_smem(int nb, int waves, int S, bool loop) {
  return ((size_t)waves * lf_wave_floats(nb) + lf_mat_floats(nb) + (loop ? (size_t)3 * S * kLfSlab : 0)) * sizeof(float);
}

template <typename XT, typename GT, int NB, int SPW, int MODE, bool PT>
int lf_bwd_launch(const GenArgs& A, int waves, int64_t gmax, hipStream_t s, int64_t* num_partials) {
  const int S = (int)ceil_div(A.C, kLfSlab);
  const size_t smem = lf_bwd_smem(NB, waves, S, SPW == 0);
  const void* kfn = (const void*)lf32_bwd_kernel<XT, GT, NB, SPW, MODE, PT>;
  const int occ = occupancy_blocks(kfn, waves * 64, smem);
  if (occ <= 0) return 1;
  int64_t blocks = std::min<int64_t>(gmax, (int64_t)device_cu_count() * occ);
  const int grid_pref = knob(kKnobBwdGrid, 0);
  if (grid_pref > 0) blocks = std::min<int64_t>(gmax, grid_pref);
  blocks = std::max<int64_t>(1, std::min<int64_t>(A.T, blocks));
  hipLaunchKernelGGL((lf32_bwd_kernel<XT, GT, NB, SPW, MODE, PT>), dim3((unsigned)blocks), dim3(waves * 64), smem, s, A);
  MHC_CHECK_LAUNCH("lf32_bwd_kernel");
  *num_partials = blocks;
  return MHC_OK;
}

constexpr size_t kLfLds = 160 * 1024 - 1024;  // of a CU, less the static part

// The largest wave count of SPW = 0 whose LDS fits (0: the row does not fit at all).
template <int NB>
int lf_bwd_waves(int C, int most) {
  const size_t rest = ((size_t)lf_mat_floats(NB) + (size_t)3 * ceil_div(C, kLfSlab) * kLfSlab) * sizeof(float);
  for (int w = most; w > 0; --w)
    if (rest + (size_t)w * lf_wave_floats(NB) * sizeof(float) <= kLfLds) return w;
  return 0;
}

template <typename XT, typename GT, int NB, int MODE>
int lf_bwd_split(const GenArgs& A, int64_t gmax, hipStream_t s, int64_t* np) {
  const int S = (int)ceil_div(A.C, kLfSlab);
  if (A.M_ts != 0) {
    // waves per token: the fewest with which eight waves can be resident on a CU (a workgroup's y, d and dw take 12 C
    // bytes of LDS beside its waves' rows) and the tokens fill eight on every CU; else the most resident ones
    int waves = 0;
    int64_t best = 0;
    for (int w = 1; w <= std::min(S, kLfPtWaves) && best < 8; ++w) {
      const int64_t resident = w * (int64_t)(kLfLds / lf_bwd_smem(NB, w, S, true));
      const int64_t filled = std::min(resident, ceil_div(A.T * w, (int64_t)device_cu_count()));
      if (filled > best) {
        best = filled;
        waves = w;
      }
    }
    if (waves == 0) return 1;
    return lf_bwd_launch<XT, GT, NB, 0, MODE, true>(A, waves, gmax, s, np);
  }
  if constexpr (NB <= 2) {
    if (S <= kLfMaxWaves) return lf_bwd_launch<XT, GT, NB, 1, MODE, false>(A, S, gmax, s, np);
  }
  if constexpr (NB == 1) {
    if (S <= 2 * kLfMaxWaves) return lf_bwd_launch<XT, GT, NB, 2, MODE, false>(A, (int)ceil_div(S, 2), gmax, s, np);
    if constexpr (MODE != kLfElem && sizeof(XT) == 2) {
      if (S <= 3 * kLfMaxWaves) return lf_bwd_launch<XT, GT, NB, 3, MODE, false>(A, (int)ceil_div(S, 3), gmax, s, np);
    }
  }
  const int waves = lf_bwd_waves<NB>(A.C, std::min(NB > 2 ? 4 : kLfMaxWaves, S));
  if (waves == 0) return 1;
  return lf_bwd_launch<XT, GT, NB, 0, MODE, false>(A, waves, gmax, s, np);
}

}  // namespace

template <typename XT, typename GT>
int lf_bwd_types(const GenArgs& A, int64_t gmax, hipStream_t s, int64_t* np) {
  const int mode = lf_mode(A.C, sizeof(XT), sizeof(GT), aligned(A.x, 4 * sizeof(XT)) &&
                           aligned(A.out, 4 * sizeof(XT)) && aligned(A.g, 4 * sizeof(GT)));
  auto by_nb = [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    if (mode == kLfLine) return lf_bwd_split<XT, GT, NB, kLfLine>(A, gmax, s, np);
    if (mode == kLfVec) return lf_bwd_split<XT, GT, NB, kLfVec>(A, gmax, s, np);
    return lf_bwd_split<XT, GT, NB, kLfElem>(A, gmax, s, np);
  };
  if (A.n <= 16) return by_nb(std::integral_constant<int, 1>{});
  if (A.n <= 32) return by_nb(std::integral_constant<int, 2>{});
  if (A.n <= 48) return by_nb(std::integral_constant<int, 3>{});
  return by_nb(std::integral_constant<int, 4>{});
}

}  // namespace mhc
