// Forward of the layer on fp32 MFMA (v_mfma_f32_16x16x4_f32), 8 < n <= 64,
// any C, fp32 or 16-bit x, layer-wide or per-token parameters:
//   out_i = sum_j M_ij x_j + p_i y inv w,  y = sum_j a_j x_j.
//
// At n = 32 the mix is 1024 FMAs per channel: on the VALU, against rows of M
// broadcast from LDS, it ran at 13-60% of what HBM allows.  The fp32 matrix
// cores take fp32 operands, so the products are the fp32 ones whatever the
// storage type, and at n = 32 they need about 60% of the channel's HBM time
// (fp32 in and out).  So the kernel is laid out for HBM: a slab is 64
// channels of every stream, each read once.  Forward kernel, against the VALU
// kernels before it: 4096 x 32 x 512 fp32 244 -> 98 us (5.5 TB/s), 2048 x 64 x
// 512 fp32 436 -> 112 us, 1024 x 32 x 4096 fp32 480 -> 263 us (two passes),
// 20000 x 24 x 100 bf16 455 -> 60 us, 3001 x 16 x 1100 fp16 81 -> 62 us (3.4
// TB/s: bound by instruction issue, 16-bit rows in 8-byte pieces), 4096 x 12 x
// 2001 bf16 (one element at a time) 215 -> 150 us.
//
// Lane (q = lane >> 4, r = lane & 15) holds streams krow(m, q), m < 4 NB, at
// four channels of the slab: the MFMA's B operand for channel v is "the four
// streams of step m, column r".  A is M's row 16 I + r at those streams.  D
// holds output rows 16 I + 4q + k of the same channels, so rows are loaded
// and stored in the same 16-byte pieces with no exchange between lanes.  y
// needs the lane's streams (VALU) and one sum over q.
//
// SPW > 0: the token's x is held in registers (SPW slabs per wave, at most
// eight waves), read once, the next token's loads issued as soon as the
// MFMAs have consumed it, before this token's stores.  SPW = 0, longer
// tokens: two passes over the wave's slabs, y in LDS between them, the second
// read from the caches.
//
// Above n = 32 (BIG) M's operands and D of a whole slab would take 128
// registers beside x's 64: M sits in LDS, one float4 (four steps) per lane and
// row block, and the mix runs one 16-row block at a time after the RMS
// barrier, its rows stored before the next block is formed.
#include <type_traits>

#include "mhc_device.hpp"
#include "mhc_generic.hpp"
#include "mhc_host.hpp"
#include "mhc_lf32.hpp"
#include "mhc_plan.hpp"

namespace mhc {

namespace {

template <typename XT, typename OT, int NB, int SPW, int MODE, bool PT>
__global__ __launch_bounds__(64 * kLfMaxWaves) void lf32_fwd_kernel(GenFwdArgs A) {
  constexpr bool VEC = MODE != kLfElem;
  constexpr int NK = 4 * NB;
  constexpr int NJ = SPW > 0 ? SPW : 1;
  constexpr bool BIG = NB > 2;
  static_assert(!BIG || SPW <= 1, "one slab per wave above n = 32");
  extern __shared__ __align__(16) float lf_smem[];  // SPW = 0: y of the token, by slab
  __shared__ float s_red[2][kLfMaxWaves];
  __shared__ __align__(16) float4 s_m[BIG ? NB * NB * 64 : 1];  // BIG: M's operands, [row block][steps 4g..][lane]
  __shared__ float s_p[BIG ? 16 * NB : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = __builtin_amdgcn_readfirstlane(blockDim.x >> 6);
  const int q = lane >> 4, r = lane & 15;
  const int n = A.n, C = A.C, S = (C + kLfSlab - 1) / kLfSlab;
  const uint32_t rowx = (uint32_t)C * sizeof(XT), rowo = (uint32_t)C * sizeof(OT);
  const uint32_t xbytes = (uint32_t)n * rowx, obytes = (uint32_t)n * rowo;
  const int64_t tile = (int64_t)n * C;
  const XT* X = (const XT*)A.x;
  OT* O = (OT*)A.out;
  const bool raw = A.h_mode == MHC_H_RAW;
  // stream of step m in lane group q (above n = 16 a lane's steps are consecutive streams)
  auto krow = [&](int m) { return NB == 1 ? 4 * m + q : q * NK + m; };
  const uint32_t kstep = NB == 1 ? 4u * rowx : rowx;

  float am[BIG ? 1 : NB][NK], a[NK], p[BIG ? 1 : NB][4];
  // token t's parameters as they lie (per token, n <= 32, they are loaded one token ahead), and what the lane needs
  float ha, hp;
  auto load_params = [&](int64_t t) {
    ha = A.hpre[t * A.h_ts + (lane < n ? lane : 0)];
    hp = A.hpost[t * A.h_ts + (lane < n ? lane : 0)];
    if constexpr (!BIG) {
      const float* M = A.M + t * A.M_ts;
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int m = 0; m < NK; ++m) am[I][m] = lf_entry(M, 16 * I + r, krow(m), n);
    }
  };
  auto activate = [&] {
    const float av = lf_act(ha, lane, n, raw, 1.0f), pv = lf_act(hp, lane, n, raw, 2.0f);
#pragma unroll
    for (int m = 0; m < NK; ++m) a[m] = lf_lane(av, krow(m));
    if constexpr (BIG) {
      if (wave == 0 && lane < 16 * NB) s_p[lane] = pv;
    } else {
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int k = 0; k < 4; ++k) p[I][k] = lf_lane(pv, 16 * I + 4 * q + k);
    }
  };
  auto stage_params = [&](int64_t t) {  // BIG
    const float* M = A.M + t * A.M_ts;
    load_params(t);
    __syncthreads();  // the previous token's rows are formed
    for (int k = threadIdx.x; k < NB * NB * 64; k += blockDim.x) {
      const int l = k & 63, g = (k >> 6) % NB, row = 16 * ((k >> 6) / NB) + (l & 15), col = (l >> 4) * NK + 4 * g;
      s_m[k] = make_float4(lf_entry(M, row, col, n), lf_entry(M, row, col + 1, n), lf_entry(M, row, col + 2, n),
                           lf_entry(M, row, col + 3, n));
    }
    activate();
    __syncthreads();
  };
  if constexpr (BIG) {
    if constexpr (!PT) stage_params(0);
  } else {
    load_params(PT ? (int64_t)blockIdx.x : 0);
    if constexpr (!PT) activate();
  }

  LfQuad<XT, VEC> x[NJ][NK];
  // y of the four channels of x[j] on every lane group
  auto agg = [&](int j, float (&y)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float s = 0.0f;
#pragma unroll
      for (int m = 0; m < NK; ++m) s = fmaf(a[m], x[j][m].get(v), s);
      y[v] = lf_sum_q(s);
    }
  };
  // all row blocks of the mix over x[j] (n <= 32)
  auto mix = [&](int j, f32x4 (&d)[NB][4]) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int v = 0; v < 4; ++v) d[I][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < NK; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float b = x[j][m].get(v);
#pragma unroll
        for (int I = 0; I < NB; ++I) d[I][v] = lf_mfma(am[I][m], b, d[I][v]);
      }
  };
  auto load_w = [&](int s, float (&w)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = s * kLfSlab + lf_chan<VEC>(r, v);
      w[v] = A.w[c < C ? c : 0];
    }
  };
  // rows 16 I + 4q .. + 3 of the slab: d + p y inv w
  auto store_rows = [&](const f32x4 (&d)[4], const float (&p4)[4], const float (&yn)[4], int I,
                        __amdgpu_buffer_rsrc_t ro, const LfOff<VEC>& off) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = fmaf(yn[v], p4[k], d[v][k]);
      lf_store<OT, VEC, lf_aux(MODE)>(ro, off.fresh(), (uint32_t)(16 * I + k) * rowo, o);
    }
  };
  // BIG: the mix of x[0] and its stores, one row block at a time
  auto mix_store = [&](const float (&yn)[4], __amdgpu_buffer_rsrc_t ro, const LfOff<VEC>& off) {
#pragma unroll 1
    for (int I = 0; I < NB; ++I) {
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
          for (int v = 0; v < 4; ++v) d[v] = lf_mfma(mm[e], x[0][4 * g + e].get(v), d[v]);
      }
      float p4[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) p4[k] = s_p[16 * I + 4 * q + k];
      store_rows(d, p4, yn, I, ro, off);
    }
  };
  // the token's RMS factor from the waves' sums of y^2 (one barrier; the buffers alternate)
  auto rms = [&](float ss, int it, int64_t t) {
    ss = group_sum<16>(ss);
    if (lane == 0) s_red[it & 1][wave] = ss;
    lds_barrier();
    float tot = 0.0f;
    for (int k = 0; k < nw; ++k) tot += s_red[it & 1][k];
    const float inv = 1.0f / sqrtf(tot / (float)C + A.eps);
    if (A.inv_rms != nullptr && threadIdx.x == 0) A.inv_rms[t] = inv;
    return inv;
  };
  auto load = [&](auto aux, int j, __amdgpu_buffer_rsrc_t rx, const LfOff<VEC>& off) {
    const LfOff<VEC> f = off.fresh();
#pragma unroll
    for (int m = 0; m < NK; ++m) x[j][m].template load<decltype(aux)::value>(rx, f, (uint32_t)m * kstep);
  };
  constexpr std::integral_constant<int, 0> kKeep{};   // cached: read again
  constexpr std::integral_constant<int, lf_aux(MODE)> kOnce{};

  int it = 0;
  if constexpr (SPW > 0) {
    LfOff<VEC> ix[NJ], io[NJ];
    float w[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int s = wave + j * nw;
      ix[j].set((uint32_t)krow(0) * rowx, s, r, C, sizeof(XT));
      io[j].set((uint32_t)(4 * q) * rowo, s, r, C, sizeof(OT));
      load_w(s, w[j]);
    }
    // a wave's loads of token t (none when t is past the end: an empty resource)
    auto load_token = [&](int64_t t) {
      const auto rx = lf_rsrc(X + (t < A.T ? t : 0) * tile, t < A.T ? xbytes : 0u);
#pragma unroll
      for (int j = 0; j < NJ; ++j) load(kOnce, j, rx, ix[j]);
    };
    if constexpr (!BIG) load_token(blockIdx.x);
    // (entering the loop with these loads pending would make every iteration's waits as strict as the first's)
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    for (int64_t t = blockIdx.x; t < A.T; t += gridDim.x, ++it) {
      if constexpr (BIG) load_token(t);
      if constexpr (PT && BIG) stage_params(t);
      if constexpr (PT && !BIG) activate();
      const auto ro = lf_rsrc(O + t * tile, obytes);
      float y[NJ][4], ss = 0.0f;
      if constexpr (BIG) {
        agg(0, y[0]);
#pragma unroll
        for (int v = 0; v < 4; ++v) ss = fmaf(y[0][v], y[0][v], ss);
        const float inv = rms(ss, it, t);
        float yn[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) yn[v] = (y[0][v] * inv) * w[0][v];
        mix_store(yn, ro, io[0]);
      } else {
        f32x4 d[NJ][NB][4];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          agg(j, y[j]);
#pragma unroll
          for (int v = 0; v < 4; ++v) ss = fmaf(y[j][v], y[j][v], ss);
          mix(j, d[j]);
        }
        load_token(t + gridDim.x);
        if constexpr (PT) load_params(t + gridDim.x < A.T ? t + gridDim.x : t);
        issue_fence();
        const float inv = rms(ss, it, t);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          float yn[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) yn[v] = (y[j][v] * inv) * w[j][v];
#pragma unroll
          for (int I = 0; I < NB; ++I) store_rows(d[j][I], p[I], yn, I, ro, io[j]);
        }
      }
    }
  } else {
    for (int64_t t = blockIdx.x; t < A.T; t += gridDim.x, ++it) {
      if constexpr (PT && BIG) stage_params(t);
      if constexpr (PT && !BIG) {
        if (it != 0) load_params(t);
        activate();
      }
      const auto rx = lf_rsrc(X + t * tile, xbytes);
      const auto ro = lf_rsrc(O + t * tile, obytes);
      auto load_slab = [&](auto aux, int s) {
        LfOff<VEC> off;
        off.set((uint32_t)krow(0) * rowx, s, r, C, sizeof(XT));
        load(aux, 0, rx, off);
      };
      float ss = 0.0f;
      load_slab(kKeep, wave);
      for (int s = wave; s < S; s += nw) {
        float y[4];
        agg(0, y);
        if (s + nw < S) load_slab(kKeep, s + nw);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ss = fmaf(y[v], y[v], ss);
          if (q == 0) lf_smem[s * kLfSlab + lf_chan<VEC>(r, v)] = y[v];
        }
      }
      if constexpr (!BIG) load_slab(kOnce, wave);
      const float inv = rms(ss, it, t);
      for (int s = wave; s < S; s += nw) {
        if constexpr (BIG) load_slab(kOnce, s);
        float yn[4], w[4];
        load_w(s, w);
#pragma unroll
        for (int v = 0; v < 4; ++v)  // the wave's own values
          yn[v] = (lf_smem[s * kLfSlab + lf_chan<VEC>(r, v)] * inv) * w[v];
        LfOff<VEC> oo;
        oo.set((uint32_t)(4 * q) * rowo, s, r, C, sizeof(OT));
        if constexpr (BIG) {
          mix_store(yn, ro, oo);
        } else {
          f32x4 d[NB][4];
          mix(0, d);
          if (s + nw < S) load_slab(kOnce, s + nw);
          issue_fence();
#pragma unroll
          for (int I = 0; I < NB; ++I) store_rows(d[I], p[I], yn, I, ro, oo);
        }
      }
    }
  }
}

template <typename XT, typename OT, int NB, int SPW, int MODE, bool PT>
int lf_fwd_launch(const GenArgs& A, int waves, hipStream_t s) {
  const int S = (int)ceil_div(A.C, kLfSlab);
  const size_t smem = SPW > 0 ? 0 : (size_t)S * kLfSlab * sizeof(float);
  const void* kfn = (const void*)lf32_fwd_kernel<XT, OT, NB, SPW, MODE, PT>;
  const int occ = occupancy_blocks(kfn, waves * 64, smem);
  if (occ <= 0) return 1;
  const int per_cu = knob(kKnobFwdGrid, 0);
  int64_t blocks = (int64_t)device_cu_count() * (per_cu > 0 ? per_cu : occ);
  blocks = std::max<int64_t>(1, std::min<int64_t>(A.T, blocks));
  hipLaunchKernelGGL((lf32_fwd_kernel<XT, OT, NB, SPW, MODE, PT>), dim3((unsigned)blocks), dim3(waves * 64), smem, s,
                     GenFwdArgs(A));
  MHC_CHECK_LAUNCH("lf32_fwd_kernel");
  return MHC_OK;
}

constexpr int kLfFwdMaxC = 32768;  // y of a token in LDS: 128 KB

template <typename XT, typename OT, int NB, int MODE, bool PT>
int lf_fwd_split(const GenArgs& A, hipStream_t s) {
  const int S = (int)ceil_div(A.C, kLfSlab);
  // The fewest slabs per wave that fit in eight waves (64 fp32 values of x per lane at most, half of that with one
  // offset per channel), then the two-pass form.  At n <= 16 two at least where a wave would otherwise do too little:
  // per token, since every wave takes the token's M and activations again (15000 x 16 x 100 fp32 49.1 -> 45.5 us,
  // 8008 x 9 x 333 fp32 62 -> 50 us), and for 16-bit elements one at a time (6006 x 12 x 333 bf16 43.7 -> 34.7 us).
  const bool two = NB == 1 && S > 1 && (PT || (MODE == kLfElem && sizeof(XT) == 2));
  const int least = knob(kKnobFwdSpw, two ? 2 : 1);
  if (least <= 1 && S <= kLfMaxWaves) return lf_fwd_launch<XT, OT, NB, 1, MODE, PT>(A, S, s);
  if constexpr (NB == 1 || (NB == 2 && MODE != kLfElem)) {
    if (least <= 2 && S <= 2 * kLfMaxWaves) return lf_fwd_launch<XT, OT, NB, 2, MODE, PT>(A, (int)ceil_div(S, 2), s);
  }
  if constexpr (NB == 1 && MODE != kLfElem) {
    if (least <= 4 && S <= 4 * kLfMaxWaves) return lf_fwd_launch<XT, OT, NB, 4, MODE, PT>(A, (int)ceil_div(S, 4), s);
  }
  if (A.C > kLfFwdMaxC) return 1;
  return lf_fwd_launch<XT, OT, NB, 0, MODE, PT>(A, std::min(S, kLfMaxWaves), s);
}

template <typename XT, typename OT>
int lf_fwd_types(const GenArgs& A, hipStream_t s) {
  const int mode = lf_mode(A.C, sizeof(XT), sizeof(OT), aligned(A.x, 4 * sizeof(XT)) && aligned(A.out, 4 * sizeof(OT)));
  auto by_nb = [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    auto by_mode = [&](auto m) {
      constexpr int MODE = decltype(m)::value;
      return A.M_ts != 0 ? lf_fwd_split<XT, OT, NB, MODE, true>(A, s) : lf_fwd_split<XT, OT, NB, MODE, false>(A, s);
    };
    if (mode == kLfLine) return by_mode(std::integral_constant<int, kLfLine>{});
    if (mode == kLfVec) return by_mode(std::integral_constant<int, kLfVec>{});
    return by_mode(std::integral_constant<int, kLfElem>{});
  };
  if (A.n <= 16) return by_nb(std::integral_constant<int, 1>{});
  if (A.n <= 32) return by_nb(std::integral_constant<int, 2>{});
  if (A.n <= 48) return by_nb(std::integral_constant<int, 3>{});
  return by_nb(std::integral_constant<int, 4>{});
}

}  // namespace

int lf32_fused_fwd(const GenArgs& A, int xd, int od, hipStream_t s) {
  if (knob(kKnobFwdMfma, 1) == 0) return 1;
  // offsets inside a token are 32-bit, with the top bit for "outside"
  if ((int64_t)A.n * A.C * 4 >= (int64_t)1 << 31 || A.n > 64) return 1;
  // fp32 rows of 21 to 32 slabs at n <= 16, one element at a time (ragged or unaligned), are read twice here, and
  // fused_fwd_kernel, one pass on up to 1024 threads, is the faster one once the CUs have tokens enough (4000 x 12 x 1999
  // 190 against 228 us, 300 x 12 x 1999 22 against 18; 3000 x 16 x 1301 137 against 150, 1000 x 9 x 1301 27 against 22).
  // Vector rows, four slabs per wave, are not (4000 x 12 x 2000 157 against 150, 3000 x 16 x 2048 149 against 132, per token
  // 3000 x 9 x 1600 83 against 68).
  if (A.n <= 16 && xd == MHC_DTYPE_F32 && A.C > 1280 && A.C <= 2048 &&
      A.T > (A.C > 1536 ? 2 : 8) * (int64_t)device_cu_count() &&
      lf_mode(A.C, 4, 4, aligned(A.x, 16) && aligned(A.out, 16)) == kLfElem)
    return 1;
  if (xd == MHC_DTYPE_F32 && od == MHC_DTYPE_F32) return lf_fwd_types<float, float>(A, s);
  if (xd == MHC_DTYPE_BF16 && od == MHC_DTYPE_F32) return lf_fwd_types<__bf16, float>(A, s);
  if (xd == MHC_DTYPE_BF16 && od == MHC_DTYPE_BF16) return lf_fwd_types<__bf16, __bf16>(A, s);
  if (xd == MHC_DTYPE_F16 && od == MHC_DTYPE_F32) return lf_fwd_types<_Float16, float>(A, s);
  if (xd == MHC_DTYPE_F16 && od == MHC_DTYPE_F16) return lf_fwd_types<_Float16, _Float16>(A, s);
  return 1;
}

}  // namespace mhc
