// The layer at n <= 8 on the VALU for rows of any width and alignment: what
// fused_fwd_full_kernel and fused_bwd_lw_kernel (whole aligned chunks, whole
// workgroups) do not take, less what tile_fwd_first (fused_fwd.hip) keeps on
// fused_fwd_kernel, and in the backward two 16-bit operands element by element
// over more than 2048 channels of more than four streams (one offset per
// element of both does not fit the registers: bwd_tile_kernel).  At n <= 8 the
// mix is at most 64 FMAs per channel and HBM is the bound as long as every byte
// moves once, in wide accesses, with every lane at work, so:
//
// * A lane holds V channels of all n streams.  Token rows are addressed
//   through a buffer resource, which takes 16-byte pieces of rows that start
//   on any multiple of V elements and drops what lies past C or n; rows of
//   odd width go one element at a time, consecutive lanes on consecutive
//   elements.
// * A token takes G lanes (16, 32 or 64) while C <= G V, so that narrow
//   tokens fill the wave, then one wave with up to SPW chunks of 64 V
//   channels, then up to eight waves of a workgroup with one barrier for the
//   RMS sums; SPW = 0 walks any number of chunks, reading them a second time
//   (from the caches) after the barrier.
// * Per-token parameters are wave-uniform and come through scalar loads; one
//   lane per value evaluates the activations.  A token's n^2 + 2n gradient
//   sums are reduce-scattered across the wave (permlane swaps and DPP: 55
//   instructions for n = 4 where 24 butterfly sums take 240), after as many
//   channels per lane as the registers hold.
//
// Against the kernels that took these shapes before: forward 9990 x 4 x 1001
// bf16 103 -> 36 us (4.5 TB/s) and fp32 165 -> 63 us, 32768 x 2 x 96 bf16 30 ->
// 11 us, 2441 x 4 x 4096 fp32 per token 78 -> 57 us (5.6 TB/s); backward
// 9990 x 4 x 1001 bf16 164 -> 53 us, 4882 x 2 x 4096 bf16 108 -> 51 us, 32768 x
// 8 x 96 bf16 529 -> 41 us, 833 x 6 x 8000 bf16 213 -> 99 us (its 96 sums hold
// two waves per SIMD), per token 32768 x 8 x 96 bf16 637 -> 141 us and 8192 x 4 x
// 4096 bf16 179 -> 161 us (5.1 TB/s) repeated on the same tensors (185 us in a
// training step's trace, behind the forward and the Sinkhorn VJP).
#pragma once

#include <type_traits>

#include "mhc_device.hpp"
#include "mhc_generic.hpp"
#include "mhc_host.hpp"
#include "mhc_lf32.hpp"
#include "mhc_lv.hpp"
#include "mhc_plan.hpp"

namespace mhc {

namespace {

// Row access: one element at a time (kLvElem), four (kLvQuad) or eight
// (kLvOct, 16-bit rows) consecutive channels per lane; kLvNt adds the
// non-temporal hint for rows of whole 128-byte lines (see LfMode).
enum LvMode : int { kLvElem = 0, kLvQuad = 1, kLvOct = 2, kLvNt = 4 };
constexpr int lv_width(int mode) { return (mode & 3) == kLvOct ? 8 : 4; }
constexpr int lv_aux(int mode) { return mode & kLvNt ? 2 : 0; }
constexpr int kLvMaxWaves = 8;
constexpr uint32_t kLvNoRow = 0x40000000u;  // added to an offset: outside (tokens stay below 1 GiB)

template <int MODE>
struct LvAt {
  static constexpr bool kVec = (MODE & 3) != kLvElem;
  uint32_t e[kVec ? 1 : 4];  // element offset of the lane's channels in a row; kLfOut / 4 past C
  template <int G>
  MHC_DEV void set(int chunk, int l, int C) {
    constexpr int V = lv_width(MODE);
#pragma unroll
    for (int v = 0; v < (kVec ? 1 : 4); ++v) {
      const int c = chunk * G * V + (kVec ? l * V : l + G * v);
      e[v] = c < C ? (uint32_t)c : kLfOut / 4;
    }
  }
  // the same offsets, hidden: a row's addresses are formed where they are used, not once per row for the whole kernel
  MHC_DEV LvAt fresh() const {
    LvAt f = *this;
    if constexpr (!kVec) {
#pragma unroll
      for (int v = 0; v < 4; ++v) f.e[v] = lf_opaque(f.e[v]);
    }
    return f;
  }
};

// V channels of one row as packed words, loaded at `row` bytes.
template <typename T, int MODE>
MHC_DEV void lv_load(Vec<T, lv_width(MODE)>& d, __amdgpu_buffer_rsrc_t rs, const LvAt<MODE>& at, uint32_t row) {
  constexpr int V = lv_width(MODE), AUX = lv_aux(MODE), kBytes = V * (int)sizeof(T);
  if constexpr (LvAt<MODE>::kVec) {
    const uint32_t o = at.e[0] * (uint32_t)sizeof(T) + row;
    if constexpr (kBytes == 16) {
      const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, AUX);
      d.w[0] = u.x; d.w[1] = u.y; d.w[2] = u.z; d.w[3] = u.w;
    } else {
      static_assert(kBytes == 8, "four 16-bit elements");
      const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, AUX);
      d.w[0] = u.x; d.w[1] = u.y;
    }
  } else if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int v = 0; v < 4; ++v) d.w[v] = __builtin_amdgcn_raw_buffer_load_b32(rs, at.e[v] * 4u + row, 0, AUX);
  } else {
    uint32_t u[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) u[v] = __builtin_amdgcn_raw_buffer_load_b16(rs, at.e[v] * 2u + row, 0, AUX);
    d.w[0] = u[0] | (u[1] << 16);
    d.w[1] = u[2] | (u[3] << 16);
  }
}

template <typename T, int MODE>
MHC_DEV void lv_store(__amdgpu_buffer_rsrc_t rs, const LvAt<MODE>& at, uint32_t row,
                      const float (&v)[lv_width(MODE)]) {
  constexpr int V = lv_width(MODE), AUX = lv_aux(MODE), kBytes = V * (int)sizeof(T);
  if constexpr (LvAt<MODE>::kVec) {
    const uint32_t o = at.e[0] * (uint32_t)sizeof(T) + row;
    if constexpr (sizeof(T) == 4) {
      static_assert(kBytes == 16, "four fp32 elements");
      const u32x4 u = {__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                       __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3])};
      buf_store_b128<AUX>(u, rs, o, 0);
    } else if constexpr (kBytes == 16) {
      buf_store_b128<AUX>(u32x4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])},
                          rs, o, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])}, rs, o, 0, AUX);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (sizeof(T) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[k]), rs, at.e[k] * 4u + row, 0, AUX);
      else
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)bits16<T>(v[k]), rs, at.e[k] * 2u + row, 0, AUX);
    }
  }
}

// A token's (or the layer's) M, a and p, the same on every lane: M through
// scalar loads, the activations evaluated once each, a on lanes 0 .. n-1 and
// p on lanes 8 .. 8+n-1, then moved to scalar registers.  Zero past n.
template <int NMAX>
struct LvParams {
  float M[NMAX * NMAX], a[NMAX], p[NMAX];
  template <typename Args>
  MHC_DEV void load(const Args& A, int64_t t, int lane) {
    const int n = A.n;
    typedef const float __attribute__((address_space(4))) cfloat;
    cfloat* m = (cfloat*)(uintptr_t)(A.M + t * A.M_ts);
#pragma unroll
    for (int i = 0; i < NMAX; ++i)
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        const bool in = i < n && j < n;
        const float v = m[in ? i * n + j : 0];
        M[i * NMAX + j] = in ? v : 0.0f;
      }
    const int i = lane & 7;
    const bool post = lane & 8;
    const float h = (post ? A.hpost : A.hpre)[t * A.h_ts + (i < n ? i : 0)];
    const float act = lf_act(h, i, n, A.h_mode == MHC_H_RAW, post ? 2.0f : 1.0f);
#pragma unroll
    for (int k = 0; k < NMAX; ++k) {
      a[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, act), k));
      p[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, act), 8 + k));
    }
  }
};

// The waves of a workgroup and the tokens they take: `wpt` waves share a
// token, or (wpt = 1) every wave takes 64 / G tokens of its own.
template <int G>
struct LvWalk {
  int lane, wave, l, sub, part, wpt;
  int64_t t, stride;
  MHC_DEV LvWalk(int wpt_) : wpt(wpt_) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    l = lane & (G - 1);
    sub = lane / G;                  // the lane's token among the wave's
    part = wpt > 1 ? wave : 0;       // the wave's place in its token
    const int waves = __builtin_amdgcn_readfirstlane(blockDim.x >> 6);
    const int64_t own = wpt > 1 ? 1 : (int64_t)waves * (64 / G);
    t = (int64_t)blockIdx.x * own + (wpt > 1 ? 0 : (int64_t)wave * (64 / G));
    stride = (int64_t)gridDim.x * own;
  }
  // tokens of this step that exist (G = 64: 1)
  MHC_DEV uint32_t tokens(int64_t T) const {
    const int64_t left = T - t;
    return left < 64 / G ? (uint32_t)left : 64 / G;
  }
};

// sum over the G lanes of a token
template <int G>
MHC_DEV float lv_sum(float v) {
  v = group_sum<16>(v);
  if constexpr (G >= 32) v = xor_allreduce<16>(v, SumOp{});
  if constexpr (G >= 64) v = xor_allreduce<32>(v, SumOp{});
  return v;
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
template <int NMAX, typename XT, typename OT, int MODE, int SPW, int G, bool PT>
__global__ __launch_bounds__(64 * kLvMaxWaves) void lv_fwd_kernel(GenFwdArgs A, int wpt) {
  constexpr int V = lv_width(MODE);
  constexpr int NJ = SPW > 0 ? SPW : 1;
  static_assert(G == 64 || (!PT && SPW == 1), "several tokens per wave: layer-wide, one chunk");
  __shared__ float s_red[2][kLvMaxWaves];
  const LvWalk<G> W0(wpt);
  LvWalk<G> W = W0;
  const int n = A.n, C = A.C, S = (C + G * V - 1) / (G * V);
  const uint32_t rowx = (uint32_t)C * sizeof(XT), rowo = (uint32_t)C * sizeof(OT);
  const int64_t tile = (int64_t)n * C;
  const XT* X = (const XT*)A.x;
  OT* O = (OT*)A.out;
  const uint32_t subx = (uint32_t)W.sub * (uint32_t)n * rowx, subo = (uint32_t)W.sub * (uint32_t)n * rowo;
  LvParams<NMAX> P;
  if constexpr (!PT) P.load(A, 0, W.lane);

  Vec<XT, V> x[NJ][NMAX];
  LvAt<MODE> at[NJ];
  float w[NJ][V];
  auto place = [&](int j, int s) {
    at[j].template set<G>(s, W.l, C);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int c = s * G * V + (LvAt<MODE>::kVec ? W.l * V + v : W.l + G * v);
      w[j][v] = A.w[c < C ? c : 0];
    }
  };
  auto load = [&](int j, __amdgpu_buffer_rsrc_t rx) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i) lv_load<XT, MODE>(x[j][i], rx, at[j].fresh(), subx + (i < n ? (uint32_t)i * rowx : kLvNoRow));
  };
  auto agg = [&](int j, int v) {
    float y = 0.0f;
#pragma unroll
    for (int i = 0; i < NMAX; ++i) y = fmaf(P.a[i], x[j][i].get(v), y);
    return y;
  };
  auto finish = [&](int j, float inv, __amdgpu_buffer_rsrc_t ro) {
    float yn[V];
#pragma unroll
    for (int v = 0; v < V; ++v) yn[v] = (agg(j, v) * inv) * w[j][v];
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      float o[V];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        o[v] = 0.0f;
#pragma unroll
        for (int k = 0; k < NMAX; ++k) o[v] = fmaf(P.M[i * NMAX + k], x[j][k].get(v), o[v]);
        o[v] = fmaf(P.p[i], yn[v], o[v]);  // last: the largest term, and each sum is rounded at its own size
      }
      lv_store<OT, MODE>(ro, at[j].fresh(), subo + (i < n ? (uint32_t)i * rowo : kLvNoRow), o);
    }
  };

  if constexpr (SPW > 0) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) place(j, W.part + j * wpt);
  }
  int it = 0;
  for (; W.t < A.T; W.t += W.stride, ++it) {
    const uint32_t nt = W.tokens(A.T);
    const auto rx = lf_rsrc(X + W.t * tile, nt * (uint32_t)n * rowx);
    const auto ro = lf_rsrc(O + W.t * tile, nt * (uint32_t)n * rowo);
    float ss = 0.0f;
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) load(j, rx);
    }
    if constexpr (PT) P.load(A, W.t, W.lane);
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const float y = agg(j, v);
          ss = fmaf(y, y, ss);
        }
    } else {
      for (int s = W.part; s < S; s += wpt) {
        place(0, s);
        load(0, rx);
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const float y = agg(0, v);
          ss = fmaf(y, y, ss);
        }
      }
    }
    ss = lv_sum<G>(ss);
    if (wpt > 1) {
      if (W.lane == 0) s_red[it & 1][W.wave] = ss;
      lds_barrier();
      ss = 0.0f;
      for (int k = 0; k < wpt; ++k) ss += s_red[it & 1][k];
    }
    const float inv = 1.0f / sqrtf(ss / (float)C + A.eps);
    if (A.inv_rms != nullptr && W.l == 0 && W.part == 0 && (uint32_t)W.sub < nt) A.inv_rms[W.t + W.sub] = inv;
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) finish(j, inv, ro);
    } else {
      for (int s = W.part; s < S; s += wpt) {
        place(0, s);
        load(0, rx);
        finish(0, inv, ro);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Backward
// ---------------------------------------------------------------------------

// Sums of K values per lane over the wave's 64 lanes, scattered: a quad of
// lanes ends with at most `kLeft` of them.  Lane bits 5, 4 (permlane swaps)
// and 3, 2 (DPP) halve the values; bits 1, 0 are summed.  idx(r) is the value
// that slot r holds, -1 for padding.
template <int K>
struct LvScatter {
  static constexpr int H1 = (K + 1) / 2, H2 = (H1 + 1) / 2, H3 = (H2 + 1) / 2, H4 = (H3 + 1) / 2;
  static constexpr int kLeft = H4;
  float v[2 * H1];
  MHC_DEV static float dpp_pick(float lo, float hi, bool upper, float send_dpp) { return (upper ? hi : lo) + send_dpp; }
  MHC_DEV void run(int lane) {
#pragma unroll
    for (int r = 0; r < H1; ++r) {
      const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v[r]),
                                                      __builtin_bit_cast(unsigned, v[r + H1]), false, false);
      const unsigned lo = s[0], hi = s[1];
      v[r] = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
    }
    if constexpr (2 * H2 > H1) v[H1] = 0.0f;
#pragma unroll
    for (int r = 0; r < H2; ++r) {
      const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v[r]),
                                                      __builtin_bit_cast(unsigned, v[r + H2]), false, false);
      const unsigned lo = s[0], hi = s[1];
      v[r] = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
    }
    if constexpr (2 * H3 > H2) v[H2] = 0.0f;
    const bool b3 = lane & 8, b2 = lane & 4;
#pragma unroll
    for (int r = 0; r < H3; ++r) {
      const float lo = v[r], hi = v[r + H3];
      const float keep = b3 ? hi : lo, send = b3 ? lo : hi;
      v[r] = keep + dpp_mov<kDppRor8>(send);
    }
    if constexpr (2 * H4 > H3) v[H3] = 0.0f;
#pragma unroll
    for (int r = 0; r < H4; ++r) {
      const float lo = v[r], hi = v[r + H4];
      const float keep = b2 ? hi : lo, send = b2 ? lo : hi;
      // lane ^ 7: the other half's partner; the quad's sum below covers the flipped bits 1, 0
      float s = keep + dpp_mov<kDppHalfMirror>(send);
      s += dpp_mov<kDppXor1>(s);
      s += dpp_mov<kDppXor2>(s);
      v[r] = s;
    }
  }
  MHC_DEV static int idx(int lane, int r) {
    const int s3 = (lane & 4 ? H4 : 0) + r, s2 = (lane & 8 ? H3 : 0) + s3, s1 = (lane & 16 ? H2 : 0) + s2;
    const int k = (lane & 32 ? H1 : 0) + s1;
    return s3 < H3 && s2 < H2 && s1 < H1 && k < K ? k : -1;
  }
};

template <typename T>
MHC_DEV float lv_dot2(uint32_t g, uint32_t x, float acc);
template <>
MHC_DEV float lv_dot2<__bf16>(uint32_t g, uint32_t x, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, g), __builtin_bit_cast(bf16x2, x), acc, false);
}
template <>
MHC_DEV float lv_dot2<_Float16>(uint32_t g, uint32_t x, float acc) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, g), __builtin_bit_cast(f16x2, x), acc, false);
}
template <>
MHC_DEV float lv_dot2<float>(uint32_t, uint32_t, float acc) { return acc; }

template <int NMAX, typename XT, typename GT, int MODE, int SPW, int G, bool PT>
__global__ __launch_bounds__(64 * kLvMaxWaves) void lv_bwd_kernel(GenArgs A, int wpt) {
  constexpr int V = lv_width(MODE);
  constexpr int NJ = SPW > 0 ? SPW : 1;
  constexpr int K = NMAX * NMAX + 2 * NMAX;
  constexpr bool DOT = std::is_same<XT, GT>::value && sizeof(XT) == 2;
  static_assert(G == 64 || (!PT && SPW == 1), "several tokens per wave: layer-wide, one chunk");
  extern __shared__ float lv_smem[];  // SPW = 0: dw of the token's channels; else dw of the wave's lanes at the end
  __shared__ float s_red[2][2][kLvMaxWaves];
  __shared__ float s_acc[kLvMaxWaves][K];
  LvWalk<G> W(wpt);
  const int n = A.n, C = A.C, nn = n * n, S = (C + G * V - 1) / (G * V);
  const uint32_t rowx = (uint32_t)C * sizeof(XT), rowg = (uint32_t)C * sizeof(GT);
  const int64_t tile = (int64_t)n * C;
  const XT* X = (const XT*)A.x;
  const GT* Gd = (const GT*)A.g;
  XT* DX = (XT*)A.out;
  const bool raw = A.h_mode == MHC_H_RAW;
  const uint32_t subx = (uint32_t)W.sub * (uint32_t)n * rowx, subg = (uint32_t)W.sub * (uint32_t)n * rowg;
  LvParams<NMAX> P;
  if constexpr (!PT) P.load(A, 0, W.lane);

  LvScatter<K> acc;  // dM [NMAX * NMAX], dA, dP
  auto clear = [&] {
#pragma unroll
    for (int k = 0; k < 2 * LvScatter<K>::H1; ++k) acc.v[k] = 0.0f;
  };
  clear();
  Vec<XT, V> x[NJ][NMAX];
  Vec<GT, V> g[NJ][NMAX];
  LvAt<MODE> at[NJ];
  float w[NJ][V], dw[NJ][V];
  auto chan = [&](int s, int v) { return s * G * V + (LvAt<MODE>::kVec ? W.l * V + v : W.l + G * v); };
  auto place = [&](int j, int s) {
    at[j].template set<G>(s, W.l, C);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int c = chan(s, v);
      w[j][v] = A.w[c < C ? c : 0];
    }
  };
  auto load = [&](int j, __amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t rg) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      lv_load<XT, MODE>(x[j][i], rx, at[j].fresh(), subx + (i < n ? (uint32_t)i * rowx : kLvNoRow));
      lv_load<GT, MODE>(g[j][i], rg, at[j].fresh(), subg + (i < n ? (uint32_t)i * rowg : kLvNoRow));
    }
  };
  auto yd = [&](int j, int v, float& y, float& d) {
    y = d = 0.0f;
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      y = fmaf(P.a[i], x[j][i].get(v), y);
      d = fmaf(P.p[i], g[j][i].get(v), d);
    }
  };
  auto take = [&](int j, float& ss, float& sr) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float y, d;
      yd(j, v, y, d);
      ss = fmaf(y, y, ss);
      sr = fmaf(d * y, w[j][v], sr);
    }
  };
  float inv, kf;
  // dx, dw and the gradient sums of chunk j
  auto give = [&](int j, __amdgpu_buffer_rsrc_t ro, float (&dwv)[V]) {
    // 16-bit rows at n <= 4: all rows of a channel at a time, each element unpacked once; otherwise one row at a time,
    // so that only one row's values are live
    constexpr bool kRows = sizeof(GT) == 4 || NMAX > 4;
    float o[kRows ? 1 : NMAX][V], dy[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      // 16-bit x with fp32 gradients at n = 8: one channel's products at a time, or the unpacked rows of all spill
      if constexpr (NMAX > 4 && sizeof(XT) == 2 && sizeof(GT) == 4) __builtin_amdgcn_sched_barrier(0);
      float y, d;
      yd(j, v, y, d);
      const float yi = y * inv;
      dy[v] = d * inv * w[j][v] - kf * y;
      const float yn = yi * w[j][v];
      dwv[v] = fmaf(d, yi, dwv[v]);
      float gs[NMAX], xs[NMAX];
#pragma unroll
      for (int i = 0; i < NMAX; ++i) {
        gs[i] = g[j][i].get(v);
        xs[i] = x[j][i].get(v);
      }
      if constexpr (!kRows) {
#pragma unroll
        for (int k = 0; k < NMAX; ++k) {
          float s = 0.0f;
#pragma unroll
          for (int i = 0; i < NMAX; ++i) s = fmaf(P.M[i * NMAX + k], gs[i], s);
          o[k][v] = fmaf(P.a[k], dy[v], s);
        }
      }
#pragma unroll
      for (int i = 0; i < NMAX; ++i) {
        acc.v[NMAX * NMAX + i] = fmaf(dy[v], xs[i], acc.v[NMAX * NMAX + i]);
        acc.v[NMAX * NMAX + NMAX + i] = fmaf(gs[i], yn, acc.v[NMAX * NMAX + NMAX + i]);
      }
      if constexpr (!DOT) {
#pragma unroll
        for (int i = 0; i < NMAX; ++i)
#pragma unroll
          for (int k = 0; k < NMAX; ++k) acc.v[i * NMAX + k] = fmaf(gs[i], xs[k], acc.v[i * NMAX + k]);
      } else if (v & 1) {
#pragma unroll
        for (int i = 0; i < NMAX; ++i)
#pragma unroll
          for (int k = 0; k < NMAX; ++k)
            acc.v[i * NMAX + k] = lv_dot2<XT>(g[j][i].w[v >> 1], x[j][k].w[v >> 1], acc.v[i * NMAX + k]);
      }
    }
#pragma unroll
    for (int k = 0; k < NMAX; ++k) {
      if constexpr (kRows) {
        if constexpr (NMAX > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < V; ++v) {
          o[0][v] = 0.0f;
#pragma unroll
          for (int i = 0; i < NMAX; ++i) o[0][v] = fmaf(P.M[i * NMAX + k], g[j][i].get(v), o[0][v]);
          o[0][v] = fmaf(P.a[k], dy[v], o[0][v]);
        }
      }
      lv_store<XT, MODE>(ro, at[j].fresh(), subx + (k < n ? (uint32_t)k * rowx : kLvNoRow), o[kRows ? 0 : k]);
    }
  };

  if constexpr (SPW > 0) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      place(j, W.part + j * wpt);
#pragma unroll
      for (int v = 0; v < V; ++v) dw[j][v] = 0.0f;
    }
  } else {
    for (int c = threadIdx.x; c < S * G * V * (wpt > 1 ? 1 : (int)(blockDim.x >> 6)); c += blockDim.x) lv_smem[c] = 0.0f;
    __syncthreads();
  }
  float* s_dw = lv_smem + (SPW == 0 && wpt == 1 ? W.wave * S * G * V : 0);
  int it = 0;
  for (; W.t < A.T; W.t += W.stride, ++it) {
    const uint32_t nt = W.tokens(A.T);
    const auto rx = lf_rsrc(X + W.t * tile, nt * (uint32_t)n * rowx);
    const auto rg = lf_rsrc(Gd + W.t * tile, nt * (uint32_t)n * rowg);
    const auto ro = lf_rsrc(DX + W.t * tile, nt * (uint32_t)n * rowx);
    float ss = 0.0f, sr = 0.0f;
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) load(j, rx, rg);
    }
    if constexpr (PT) P.load(A, W.t, W.lane);
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) take(j, ss, sr);
    } else {
      for (int s = W.part; s < S; s += wpt) {
        place(0, s);
        load(0, rx, rg);
        take(0, ss, sr);
      }
    }
    ss = lv_sum<G>(ss);
    sr = lv_sum<G>(sr);
    if (wpt > 1) {
      if (W.lane == 0) {
        s_red[it & 1][0][W.wave] = ss;
        s_red[it & 1][1][W.wave] = sr;
      }
      lds_barrier();
      ss = sr = 0.0f;
      for (int k = 0; k < wpt; ++k) {
        ss += s_red[it & 1][0][k];
        sr += s_red[it & 1][1][k];
      }
    }
    inv = 1.0f / sqrtf(ss / (float)C + A.eps);
    kf = (inv * inv * inv / (float)C) * sr;
    if constexpr (SPW > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        // y and d are formed again here rather than held over the sums
#pragma unroll
        for (int i = 0; i < NMAX; ++i) {
#pragma unroll
          for (int k = 0; k < Vec<XT, V>::kWords; ++k) x[j][i].w[k] = lf_opaque(x[j][i].w[k]);
#pragma unroll
          for (int k = 0; k < Vec<GT, V>::kWords; ++k) g[j][i].w[k] = lf_opaque(g[j][i].w[k]);
        }
        // (a place past the last token stays out: its rows are zero, and with eps = 0 its inv is infinite and kf NaN)
        if (G == 64 || (uint32_t)W.sub < nt) give(j, ro, dw[j]);
      }
    } else {
      for (int s = W.part; s < S; s += wpt) {
        place(0, s);
        load(0, rx, rg);
        float d[V];
#pragma unroll
        for (int v = 0; v < V; ++v) d[v] = s_dw[chan(s, v)];  // the lane's own entries
        give(0, ro, d);
#pragma unroll
        for (int v = 0; v < V; ++v) s_dw[chan(s, v)] = d[v];
      }
    }
    if constexpr (PT) {
      // the token's sums: scattered over the wave, then the waves in order
      acc.run(W.lane);
      if ((W.lane & 3) == 0) {
#pragma unroll
        for (int r = 0; r < LvScatter<K>::kLeft; ++r) {
          const int k = LvScatter<K>::idx(W.lane, r);
          if (k >= 0) s_acc[W.wave][k] = acc.v[r];
        }
      }
      clear();
      if (wpt > 1) lds_barrier();  // (read before the next token's RMS barrier, written after it)
      else issue_fence();
      for (int k = wpt > 1 ? (int)threadIdx.x : W.lane; k < K; k += wpt > 1 ? (int)blockDim.x : 64) {
        float s = 0.0f;
        if (wpt > 1)
          for (int wv = 0; wv < wpt; ++wv) s += s_acc[wv][k];
        else
          s = s_acc[W.wave][k];
        if (k < NMAX * NMAX) {
          const int i = k / NMAX, j = k % NMAX;
          if (i < n && j < n) A.dM_tok[W.t * nn + i * n + j] = s;
        } else {
          const bool post = k >= NMAX * NMAX + NMAX;
          const int i = k - NMAX * NMAX - (post ? NMAX : 0);
          if (i < n) {
            if (raw) {
              const float h = (post ? A.hpost : A.hpre)[W.t * A.h_ts + i];
              const float sg = sigmoidf_(h);
              s *= (post ? 2.0f : 1.0f) * sg * (1.0f - sg);
            }
            (post ? A.dpost_tok : A.dpre_tok)[W.t * n + i] = s;
          }
        }
      }
    }
  }

  // ---- the workgroup's partial row [dw C | 0 .. Cp | dM | dA | dP]
  float* prow = A.part + (int64_t)blockIdx.x * A.P;
  const int waves = blockDim.x >> 6;
  __syncthreads();
  if constexpr (SPW > 0) {
    if (wpt > 1) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const int c = chan(W.part + j * wpt, v);
          if (c < C) prow[c] = dw[j][v];
        }
      for (int c = C + (int)threadIdx.x; c < A.Cp; c += blockDim.x) prow[c] = 0.0f;
    } else {
      // every wave's (and token place's) lanes hold the same channels: summed in order
      constexpr int kCh = G * V * NJ;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < V; ++v) lv_smem[(W.wave * (64 / G) + W.sub) * kCh + chan(j, v)] = dw[j][v];
      __syncthreads();
      for (int c = threadIdx.x; c < A.Cp; c += blockDim.x) {
        float s = 0.0f;
        if (c < C)
          for (int k = 0; k < waves * (64 / G); ++k) s += lv_smem[k * kCh + c];
        prow[c] = s;
      }
    }
  } else {
    const int copies = wpt > 1 ? 1 : waves;
    for (int c = threadIdx.x; c < A.Cp; c += blockDim.x) {
      float s = 0.0f;
      if (c < C)
        for (int k = 0; k < copies; ++k) s += lv_smem[k * S * G * V + c];
      prow[c] = s;
    }
  }
  if constexpr (!PT) {
    acc.run(W.lane);
    if ((W.lane & 3) == 0) {
#pragma unroll
      for (int r = 0; r < LvScatter<K>::kLeft; ++r) {
        const int k = LvScatter<K>::idx(W.lane, r);
        if (k >= 0) s_acc[W.wave][k] = acc.v[r];
      }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
      float s = 0.0f;
      for (int wv = 0; wv < waves; ++wv) s += s_acc[wv][k];
      int to = -1;
      if (k < NMAX * NMAX) {
        if (k / NMAX < n && k % NMAX < n) to = (k / NMAX) * n + k % NMAX;
      } else if (k < NMAX * NMAX + NMAX) {
        if (k - NMAX * NMAX < n) to = nn + k - NMAX * NMAX;
      } else if (k - NMAX * NMAX - NMAX < n) {
        to = nn + n + k - NMAX * NMAX - NMAX;
      }
      if (to >= 0) prow[A.Cp + to] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// The row mode of operands of t1 and t2 bytes; al4 / al8: all aligned to four / eight elements.
template <bool OCT>
int lv_mode(int C, int t1, int t2, bool al4, bool al8) {
  if (C % 4 != 0 || !al4) return kLvElem;
  const bool lines = (int64_t)C * t1 % 128 == 0 && (int64_t)C * t2 % 128 == 0;
  const int w = OCT && C % 8 == 0 && al8 ? kLvOct : kLvQuad;
  return lines ? w | kLvNt : w;
}

template <bool OCT, typename F>
int lv_by_mode(int mode, F&& f) {
  switch (mode) {
    case kLvElem: return f(std::integral_constant<int, kLvElem>{});
    case kLvQuad: return f(std::integral_constant<int, kLvQuad>{});
    case kLvQuad | kLvNt:
      if constexpr (!OCT) return f(std::integral_constant<int, kLvQuad | kLvNt>{});
      else return f(std::integral_constant<int, kLvQuad>{});
    default: break;
  }
  if constexpr (OCT) {
    if (mode == kLvOct) return f(std::integral_constant<int, kLvOct>{});
    return f(std::integral_constant<int, kLvOct | kLvNt>{});
  }
  return 1;
}

template <typename F>
int lv_by_n(int n, F&& f) {
  if (n <= 2) return f(std::integral_constant<int, 2>{});
  if (n <= 4) return f(std::integral_constant<int, 4>{});
  return f(std::integral_constant<int, 8>{});
}

// f(SPW, G, waves per token) for a row of C channels; MOST: the chunks that a wave's registers hold; `few`: few waves
// with many chunks each rather than many waves
template <int MODE, int MOST, typename F>
int lv_by_split(int C, bool few, bool sub, F&& f) {
  constexpr int V = lv_width(MODE);
  using I = std::integral_constant<int, 64>;
  if (sub && C <= 16 * V) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{}, 1);
  if (sub && C <= 32 * V) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 32>{}, 1);
  const int S = (int)ceil_div(C, 64 * V);
  int spw = 1;
  while (spw < MOST && (few ? spw < S : ceil_div(S, spw) > kLvMaxWaves)) spw *= 2;
  const int w = (int)ceil_div(S, spw);
  if (w <= kLvMaxWaves) {
    if (spw == 1) return f(std::integral_constant<int, 1>{}, I{}, w);
    if constexpr (MOST >= 2) {
      if (spw == 2) return f(std::integral_constant<int, 2>{}, I{}, w);
    }
    if constexpr (MOST >= 4) {
      if (spw == 4) return f(std::integral_constant<int, 4>{}, I{}, w);
    }
  }
  return f(std::integral_constant<int, 0>{}, I{}, std::min(S, kLvMaxWaves));
}

// chunks per wave that fit the registers
constexpr int lv_most(int mode, int nmax, bool bwd) {
  const bool quad = (mode & 3) == kLvQuad;
  return nmax <= 4 ? (quad ? 4 : 2) : (quad && !bwd ? 2 : 1);
}

// tokens per workgroup, threads
inline int64_t lv_tokens(int wpt, int G) { return wpt > 1 ? 1 : 4 * (64 / G); }
inline int lv_threads(int wpt) { return wpt > 1 ? 64 * wpt : 256; }

template <typename XT, typename OT>
int lv_fwd_typed(const GenArgs& A, hipStream_t s) {
  constexpr bool OCT = sizeof(XT) == 2 && sizeof(OT) == 2;
  const int mode = lv_mode<OCT>(A.C, sizeof(XT), sizeof(OT), aligned(A.x, 4 * sizeof(XT)) && aligned(A.out, 4 * sizeof(OT)),
                                aligned(A.x, 16) && aligned(A.out, 16));
  return lv_by_mode<OCT>(mode, [&](auto md) {
    constexpr int MODE = decltype(md)::value;
    return lv_by_n(A.n, [&](auto nm) {
      constexpr int NM = decltype(nm)::value;
      const bool pt = A.M_ts != 0;
      // (per token, few waves: every wave takes the token's parameters)
      return lv_by_split<MODE, lv_most(MODE, NM, false)>(A.C, pt, !pt, [&](auto sp, auto gr, int wpt) {
        constexpr int SPW = decltype(sp)::value, G = decltype(gr)::value;
        auto go = [&](auto ptc) {
          constexpr bool PT = decltype(ptc)::value;
          // (at n > 4 whole vectors of 16-bit rows go to fused_fwd_kernel per token and past 4096 channels)
          if constexpr (NM > 4 && (MODE & 3) == kLvOct && (PT || SPW == 0)) {
            return 1;
          } else {
            const int tpb = lv_threads(wpt);
            const int occ = occupancy_blocks((const void*)lv_fwd_kernel<NM, XT, OT, MODE, SPW, G, PT>, tpb, 0);
            if (occ <= 0) return 1;
            const int per_cu = knob(kKnobFwdGrid, 0);
            int64_t blocks = (int64_t)device_cu_count() * (per_cu > 0 ? per_cu : occ);
            blocks = std::max<int64_t>(1, std::min(blocks, ceil_div(A.T, lv_tokens(wpt, G))));
            hipLaunchKernelGGL((lv_fwd_kernel<NM, XT, OT, MODE, SPW, G, PT>), dim3((unsigned)blocks), dim3(tpb), 0, s,
                               GenFwdArgs(A), wpt);
            MHC_CHECK_LAUNCH("lv_fwd_kernel");
            return (int)MHC_OK;
          }
        };
        if constexpr (G == 64) {
          if (pt) return go(std::true_type{});
        }
        return go(std::false_type{});
      });
    });
  });
}

template <typename XT, typename GT>
int lv_bwd_typed(const GenArgs& A, int64_t gmax, hipStream_t s, int64_t* np) {
  constexpr bool OCT = sizeof(XT) == 2 && sizeof(GT) == 2;
  int mode = lv_mode<OCT>(A.C, sizeof(XT), sizeof(GT),
                                aligned(A.x, 4 * sizeof(XT)) && aligned(A.out, 4 * sizeof(XT)) && aligned(A.g, 4 * sizeof(GT)),
                                aligned(A.x, 16) && aligned(A.out, 16) && aligned(A.g, 16));
  if (A.n > 4 && (mode & 3) == kLvOct) mode = kLvQuad;  // (eight channels of eight streams and their sums do not fit)
  return lv_by_mode<OCT>(mode, [&](auto md) {
    constexpr int MODE = decltype(md)::value;
    return lv_by_n(A.n, [&](auto nm) {
      constexpr int NM = decltype(nm)::value;
      if constexpr (NM > 4 && (MODE & 3) == kLvOct) {
        return 1;
      } else {
      const bool pt = A.M_ts != 0;
      return lv_by_split<MODE, lv_most(MODE, NM, true)>(A.C, pt, !pt, [&](auto sp, auto gr, int wpt) {
        constexpr int G = decltype(gr)::value, V = lv_width(MODE);
        if constexpr (NM > 4 && MODE == kLvElem && decltype(sp)::value == 0 && OCT) {
          return 1;  // (one offset per element of two 16-bit operands over eight streams: too many registers)
        } else {
          auto go = [&](auto ptc) {
            constexpr bool PT = decltype(ptc)::value;
            // fp16 x, fp32 gradients, per-token parameters of n = 8: a lane's chunk does not stay in registers from the
            // dot products to the gradients, so it is read again
            constexpr bool kAgain = PT && NM > 4 && decltype(sp)::value == 1 && MODE != kLvElem && std::is_same<XT, _Float16>::value &&
                                    sizeof(GT) == 4;
            constexpr int SPW = kAgain ? 0 : decltype(sp)::value;
            const int tpb = lv_threads(wpt);
            const size_t chunk = (size_t)ceil_div(A.C, G * V) * G * V * sizeof(float);
            const size_t smem = SPW == 0 ? chunk * (wpt > 1 ? 1 : tpb / 64)
                                         : (wpt > 1 ? 0 : (size_t)(tpb / G) * G * V * SPW * sizeof(float));
            const int occ = occupancy_blocks((const void*)lv_bwd_kernel<NM, XT, GT, MODE, SPW, G, PT>, tpb, smem);
            if (occ <= 0) return 1;
            int64_t blocks = std::min<int64_t>(gmax, (int64_t)device_cu_count() * occ);
            const int grid_pref = knob(kKnobBwdGrid, 0);
            if (grid_pref > 0) blocks = std::min<int64_t>(gmax, grid_pref);
            blocks = std::max<int64_t>(1, std::min(blocks, ceil_div(A.T, lv_tokens(wpt, G))));
            hipLaunchKernelGGL((lv_bwd_kernel<NM, XT, GT, MODE, SPW, G, PT>), dim3((unsigned)blocks), dim3(tpb), smem, s,
                               A, wpt);
            MHC_CHECK_LAUNCH("lv_bwd_kernel");
            *np = blocks;
            return (int)MHC_OK;
          };
          if constexpr (G == 64) {
            if (pt) return go(std::true_type{});
          }
          return go(std::false_type{});
        }
      });
      }
    });
  });
}

}  // namespace

}  // namespace mhc
