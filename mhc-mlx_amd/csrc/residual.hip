// Fused residual add + stream aggregate (mhc_mlx/utils.py:4-24,
// kernels/residual_add_agg.metal:39-66 via metal.py:1673-1731):
//   out[t,i,c] = x[t,i,c] + res[t,i,c]
//   y_agg[t,c] = sum_i a_i (x[t,i,c] + res[t,i,c])      (fp32, from the unrounded sum)
// and its VJP (an extension: the reference kernel has no VJP):
//   d_val_i = dout_i + a_i dy                    dx = dres = d_val
//   dh_pre_i = sum_{t,c} dy (x_i + res_i)
//
// HBM-bound streaming.  Work item = (token, chunk of V channels) over all
// n streams (grid-stride beyond 2^24 blocks).  The streams are
// visited in groups of G: the group's x and res chunks are all issued before
// the first add, so every thread keeps 2G loads in flight.  The backward takes
// V = 8 channels per item and splits the streams over grid.y (one
// group of 4 per block row) and writes one partial row of dh_pre per block,
// finished by the fixed-order row reduction (deterministic, no atomics).
#include "mhc_device.hpp"
#include "mhc_host.hpp"
#include "mhc_plan.hpp"
#include "mhc_reduce.hpp"

namespace mhc {

namespace {

constexpr int kResThreads = 256;
constexpr int kResV = 8;
constexpr int kResSplit = 64;

struct ResArgs {
  const void* x;
  const void* res;
  const void* g;     // bwd: dout (may be null)
  const float* gy;   // bwd: d y_agg (may be null)
  void* out;         // fwd: out; bwd: dx
  void* out2;        // bwd: dres
  float* y_agg;      // fwd
  const float* hpre;
  float* part;       // bwd partial rows (may be null: no dh_pre)
  int64_t T;
  int n;
  int C;
  int nchunks;
  int h_mode;
  int vec;
  int P;
  int tpb;
};

MHC_DEV float act_pre(const ResArgs& A, int i) {
  const float h = A.hpre[i];
  return A.h_mode == MHC_H_RAW ? sigmoidf_(h) : h;
}

template <typename T>
MHC_DEV void load_c(Vec<T, kResV>& r, const T* p, bool vec, int valid) {
  if (vec && valid == kResV) r.load(p);
  else r.load_partial(p, valid);
}

template <typename T>
MHC_DEV void store_c(T* p, const float (&v)[kResV], bool vec, int valid) {
  if (vec && valid == kResV) store_vec<T, kResV, true>(p, v);
  else store_partial<T, kResV>(p, v, valid);
}

// V values to p (aligned to min(16, V elements)) as one store; NT: rows of whole 128-byte lines, past the caches.
template <typename T, int V, bool NT>
MHC_DEV void res_store(T* p, const float (&v)[V]) {
  if constexpr (NT) {
    store_vec<T, V, true>(p, v);
  } else if constexpr (V == 1) {
    store1<T>(p, v[0]);
  } else {
    constexpr int W = V * ElemTraits<T>::kBytes / 4;
    uint32_t w[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
      if constexpr (ElemTraits<T>::kBytes == 4) w[k] = __builtin_bit_cast(uint32_t, v[k]);
      else w[k] = pack2<T>(v[2 * k], v[2 * k + 1]);
    }
    uint32_t* b = reinterpret_cast<uint32_t*>(p);
    if constexpr (W == 2) {
      const u32x2 u = {w[0], w[1]};
      *reinterpret_cast<u32x2*>(b) = u;
    } else {
#pragma unroll
      for (int k = 0; k < W; k += 4) st16<false>(b + k, w[k], w[k + 1], w[k + 2], w[k + 3]);
    }
  }
}

// Bound by HBM.  A lane takes V channels of every stream, so that one instruction of a wave reads or writes one
// contiguous span: V = 8 when all rows are 16-bit, 4 when one is fp32 (eight channels of it are two 16-byte words,
// and each instruction then covers every other 16 bytes), both for rows that keep the vectors aligned; V = 1, K
// items a block apart, for the rest.  Against V = 8 for all, with ragged rows element by element: 8192 x 4 x 4096
// bf16 to fp32 231 -> 192 us (6.3 TB/s), fp32 323 -> 285, bf16 to bf16 158 -> 152; 3000 x 16 x 1100 fp16 to fp32
// 262 -> 92, 8000 x 4 x 1002 fp32 191 -> 79, 3001 x 7 x 1001 fp16 to fp32 111 -> 42.  K = 2 in groups of eight
// streams, where K = 4 takes 256 registers: the last 42 us against 59.
template <int G, typename XT, typename OT, int V, bool NT>
__global__ __launch_bounds__(kResThreads) void residual_add_agg_kernel(ResArgs A) {
  constexpr int K = V > 1 ? 1 : G > 4 ? 2 : 4;
  __shared__ float s_a[MHC_MAX_N];
  for (int i = threadIdx.x; i < A.n; i += blockDim.x) s_a[i] = act_pre(A, i);
  __syncthreads();
  const int n = A.n, C = A.C;
  const int64_t items = A.T * A.nchunks;
  const XT* X = (const XT*)A.x;
  const XT* R = (const XT*)A.res;
  OT* O = (OT*)A.out;
  const int tpb = A.tpb;  // (an argument arrives with the others; blockDim costs a load of its own)
  for (int64_t item0 = (int64_t)blockIdx.x * (tpb * K) + threadIdx.x; item0 < items;
       item0 += (int64_t)gridDim.x * (tpb * K)) {
    int64_t base[K], to[K];
    bool in[K];
    float agg[K][V];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t item = item0 + k * tpb;
      in[k] = item < items;
      const int64_t t = items <= UINT32_MAX ? (int64_t)((uint32_t)item / (uint32_t)A.nchunks) : item / A.nchunks;
      const int c0 = (int)(item - t * A.nchunks) * V;
      base[k] = t * n * C + c0;
      to[k] = t * C + c0;
#pragma unroll
      for (int v = 0; v < V; ++v) agg[k][v] = 0.0f;
    }
    for (int i0 = 0; i0 < n; i0 += G) {
      Vec<XT, V> xr[K][G], rr[K][G];
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int g = 0; g < G; ++g)
          if (in[k] && i0 + g < n) {
            xr[k][g].template load<NT>(X + base[k] + (int64_t)(i0 + g) * C);
            rr[k][g].template load<NT>(R + base[k] + (int64_t)(i0 + g) * C);
          }
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int g = 0; g < G; ++g)
          if (in[k] && i0 + g < n) {
            const float a = s_a[i0 + g];
            float o[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
              o[v] = xr[k][g].get(v) + rr[k][g].get(v);
              agg[k][v] = fmaf(o[v], a, agg[k][v]);
            }
            res_store<OT, V, NT>(O + base[k] + (int64_t)(i0 + g) * C, o);
          }
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (in[k]) res_store<float, V, NT>(A.y_agg + to[k], agg[k]);
  }
}

// grid.y = stream group (streams [blockIdx.y*G, +G)); block (bx, gy) writes
// columns [gy*G, gy*G+G) of partial row bx.
template <int G, typename XT, typename GT>
__global__ __launch_bounds__(kResThreads) void residual_add_agg_bwd_kernel(ResArgs A) {
  constexpr int V = kResV;
  __shared__ float s_stage[kResThreads / 64][G];
  const int n = A.n, C = A.C;
  const int i0 = blockIdx.y * G;
  float a[G];
#pragma unroll
  for (int g = 0; g < G; ++g) a[g] = (i0 + g < n) ? act_pre(A, i0 + g) : 0.0f;
  const int64_t items = A.T * A.nchunks;
  const XT* X = (const XT*)A.x;
  const XT* R = (const XT*)A.res;
  const GT* Gd = (const GT*)A.g;
  XT* DX = (XT*)A.out;
  XT* DR = (XT*)A.out2;
  const bool want_dh = A.part != nullptr && A.gy != nullptr;
  float acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = 0.0f;
  for (int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; item < items;
       item += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = item / A.nchunks;
    const int q = (int)(item - t * A.nchunks);
    const int c0 = q * V;
    const int valid = min(V, C - c0);
    const int64_t base = t * n * C + c0;
    Vec<float, V> gyr;
    if (A.gy) load_c<float>(gyr, A.gy + t * C + c0, A.vec, valid);
    else gyr.zero();
    Vec<GT, V> gr[G];
    Vec<XT, V> xr[G], rr[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (i0 + g < n) {
        const int64_t off = base + (int64_t)(i0 + g) * C;
        if (Gd) load_c<GT>(gr[g], Gd + off, A.vec, valid);
        else gr[g].zero();
        if (want_dh) {
          load_c<XT>(xr[g], X + off, A.vec, valid);
          load_c<XT>(rr[g], R + off, A.vec, valid);
        }
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (i0 + g < n) {
        const int64_t off = base + (int64_t)(i0 + g) * C;
        float d[V];
#pragma unroll
        for (int v = 0; v < V; ++v) d[v] = fmaf(a[g], gyr.get(v), gr[g].get(v));
        if (DX) store_c<XT>(DX + off, d, A.vec, valid);
        if (DR) store_c<XT>(DR + off, d, A.vec, valid);
        if (want_dh) {
#pragma unroll
          for (int v = 0; v < V; ++v) acc[g] = fmaf(gyr.get(v), xr[g].get(v) + rr[g].get(v), acc[g]);
        }
      }
    }
  }
  if (A.part == nullptr) return;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float s = wave_sum(acc[g]);
    if ((threadIdx.x & 63) == 0) s_stage[threadIdx.x >> 6][g] = s;
  }
  __syncthreads();
  float* prow = A.part + (int64_t)blockIdx.x * A.P;
  if (threadIdx.x < G && i0 + (int)threadIdx.x < n) {
    float s = 0.0f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += s_stage[w][threadIdx.x];
    prow[i0 + threadIdx.x] = s;
  }
  if (blockIdx.y == 0)
    for (int c = n + (int)threadIdx.x; c < A.P; c += blockDim.x) prow[c] = 0.0f;
}

__global__ __launch_bounds__(64) void residual_final_kernel(const float* __restrict__ part2, int S, int P,
                                                            int n, int h_mode,
                                                            const float* __restrict__ hpre,
                                                            float* __restrict__ dpre) {
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    float s = 0.0f;
    for (int k = 0; k < S; ++k) s += part2[(int64_t)k * P + j];
    if (h_mode == MHC_H_RAW) {
      const float a = sigmoidf_(hpre[j]);
      s *= a * (1.0f - a);
    }
    dpre[j] = s;
  }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------

int res_group(int n) { return n <= 4 ? 4 : 8; }
// The backward holds dout, x and res of a group in registers: groups of 4.
constexpr int kResBwdGroup = 4;

// One item per thread (the grid-stride loop then runs once) measured best on
// MI355X: 4% faster at 32768 x 4 x 4096 bf16 than the best of the persistent
// grids of 2-32 blocks per CU.  MHC_RES_GRID > 0 caps the grid
// at that many blocks per CU (tuning override).
int64_t res_fwd_grid(int64_t items, int tpb, int cus) {
  const int64_t g = ceil_div(items, tpb);
  const int per_cu = knob(kKnobResGrid, -1);
  if (per_cu < 0) return std::max<int64_t>(1, std::min<int64_t>(g, kMaxGrid));
  return std::max<int64_t>(1, std::min<int64_t>(g, (int64_t)cus * std::max(per_cu, 1)));
}

int64_t res_bwd_grid(int64_t T, int n, int C, int cus) {
  const int64_t groups = ceil_div(n, kResBwdGroup);
  const int64_t g = ceil_div(T * ceil_div(C, kResV), kResThreads);
  return std::max<int64_t>(1, std::min<int64_t>(g, (int64_t)cus * 8 / groups + 1));
}

bool res_vec_ok(int C, int V, std::initializer_list<std::pair<const void*, int>> ptrs) {
  if (C % V != 0) return false;
  for (auto& pr : ptrs) {
    if (pr.first == nullptr) continue;
    const int al = std::min(16, V * pr.second);
    if (!aligned(pr.first, al)) return false;
  }
  return true;
}

template <typename F>
int res_by_dtype(int code, F&& f) {
  switch (code) {
    case MHC_DTYPE_F32: return f((float*)nullptr);
    case MHC_DTYPE_BF16: return f((__bf16*)nullptr);
    case MHC_DTYPE_F16: return f((_Float16*)nullptr);
    default: return set_error(MHC_ERR_INVALID_ARG, "unknown dtype code %d", code);
  }
}

template <typename F>
int res_by_group(int n, F&& f) {
  if (res_group(n) == 4) return f(std::integral_constant<int, 4>{});
  return f(std::integral_constant<int, 8>{});
}

}  // namespace
}  // namespace mhc

using namespace mhc;

extern "C" int mhc_residual_add_agg_fwd(const void* x, const void* res, int dtype, const float* h_pre,
                                        int h_mode, void* out, int out_dtype, float* y_agg, int64_t T,
                                        int n, int C, void* stream) {
  clear_error();
  MHC_CHECK_ARG(n >= 1 && n <= MHC_MAX_N, "n=%d must be in [1, %d]", n, MHC_MAX_N);
  MHC_CHECK_ARG(C >= 1 && T >= 0, "invalid T=%lld / C=%d", (long long)T, C);
  MHC_CHECK_ARG(h_mode == MHC_H_ACTIVATED || h_mode == MHC_H_RAW, "invalid h_mode %d", h_mode);
  if (T == 0) return MHC_OK;
  MHC_CHECK_ARG(x && res && h_pre && out && y_agg, "null pointer argument");
  MHC_CHECK_ARG(dtype_bytes(dtype) && dtype_bytes(out_dtype), "unknown dtype code");
  ResArgs A{};
  A.x = x; A.res = res; A.out = out; A.y_agg = y_agg; A.hpre = h_pre; A.T = T; A.n = n; A.C = C;
  A.h_mode = h_mode;
  const int bx = dtype_bytes(dtype), bo = dtype_bytes(out_dtype);
  auto fits = [&](int v) { return res_vec_ok(C, v, {{x, bx}, {res, bx}, {out, bo}, {y_agg, 4}}); };
  const int V = bx == 2 && bo == 2 && fits(8) ? 8 : fits(4) ? 4 : 1;
  // Non-temporal for rows of whole 128-byte lines; other rows share lines with their neighbours (3000 x 16 x 1100 fp16
  // to fp32: 92 us cached, 95 with the hint).
  const bool nt = V > 1 && (int64_t)C * bx % 128 == 0 && (int64_t)C * bo % 128 == 0;
  A.nchunks = C / V;
  const int64_t lanes = ceil_div(T * A.nchunks, V > 1 ? 1 : res_group(n) > 4 ? 2 : 4);
  // One wave per workgroup where four leave half the CUs without work or a few with twice the work of the rest (200 x 9 x
  // 1536 fp32, 300 workgroups of four waves 8.3 us, 1200 of one 6.6; 400 x 48 x 768 39.6 and 31); elsewhere four (400 x 4 x
  // 1536, 600 workgroups, equal; 2000 x 2 x 768 bf16 5.0 against 6.3), and at n < 4, where a wave has few loads to wait for.
  const int cus = device_cu_count();
  const int64_t wide = ceil_div(lanes, kResThreads);
  const int tpb = n >= 4 && (2 * wide <= cus || (wide > cus && 4 * wide <= 5 * (int64_t)cus)) ? 64 : kResThreads;
  A.tpb = tpb;
  const int64_t blocks = res_fwd_grid(lanes, tpb, cus);
  hipStream_t s = (hipStream_t)stream;
  return res_by_group(n, [&](auto gc) {
    constexpr int G = decltype(gc)::value;
    return res_by_dtype(dtype, [&](auto* xp) {
      using XT = std::remove_pointer_t<decltype(xp)>;
      return res_by_dtype(out_dtype, [&](auto* op) {
        using OT = std::remove_pointer_t<decltype(op)>;
        auto go = [&](auto vc, auto ntc) {
          hipLaunchKernelGGL((residual_add_agg_kernel<G, XT, OT, decltype(vc)::value, decltype(ntc)::value>),
                             dim3((unsigned)blocks), dim3(tpb), 0, s, A);
          MHC_CHECK_LAUNCH("residual_add_agg_kernel");
          return (int)MHC_OK;
        };
        using std::integral_constant;
        if constexpr (sizeof(XT) == 2 && sizeof(OT) == 2) {
          if (V == 8) {
            return nt ? go(integral_constant<int, 8>{}, std::true_type{}) : go(integral_constant<int, 8>{}, std::false_type{});
          }
        }
        if (V == 4) {
          return nt ? go(integral_constant<int, 4>{}, std::true_type{}) : go(integral_constant<int, 4>{}, std::false_type{});
        }
        return go(integral_constant<int, 1>{}, std::false_type{});
      });
    });
  });
}

extern "C" size_t mhc_residual_add_agg_bwd_workspace_bytes(int64_t T, int n, int C) {
  if (T <= 0 || n < 1 || n > MHC_MAX_N || C < 1) return 0;
  const int64_t G = res_bwd_grid(T, n, C, device_cu_count());
  return (size_t)(G + kResSplit) * (size_t)round_up(n, 4) * sizeof(float);
}

extern "C" int mhc_residual_add_agg_bwd(const void* x, const void* res, int dtype, const void* dout,
                                        int dout_dtype, const float* dy_agg, const float* h_pre,
                                        int h_mode, void* dx, void* dres, float* dh_pre, void* workspace,
                                        size_t workspace_bytes, int64_t T, int n, int C, void* stream) {
  clear_error();
  MHC_CHECK_ARG(n >= 1 && n <= MHC_MAX_N, "n=%d must be in [1, %d]", n, MHC_MAX_N);
  MHC_CHECK_ARG(C >= 1 && T >= 0, "invalid T=%lld / C=%d", (long long)T, C);
  MHC_CHECK_ARG(h_mode == MHC_H_ACTIVATED || h_mode == MHC_H_RAW, "invalid h_mode %d", h_mode);
  MHC_CHECK_ARG(dtype_bytes(dtype), "unknown dtype code %d", dtype);
  MHC_CHECK_ARG(!dout || dout_dtype == MHC_DTYPE_F32 || dout_dtype == dtype,
                "dout_dtype must be fp32 or the inputs' dtype");
  MHC_CHECK_ARG(h_pre, "h_pre is required");
  const int cus = device_cu_count();
  if (T == 0) {
    // no tokens: dh_pre = 0 (a kernel write, not a memset, so the call stays capturable)
    if (dh_pre) {
      hipLaunchKernelGGL(residual_final_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, nullptr, 0, 4, n,
                         MHC_H_ACTIVATED, h_pre, dh_pre);
      MHC_CHECK_LAUNCH("residual_final_kernel");
    }
    return MHC_OK;
  }
  MHC_CHECK_ARG(!dh_pre || (x && res), "x and res are required for dh_pre");
  const int64_t G = res_bwd_grid(T, n, C, cus);
  const int P = round_up(n, 4);
  if (dh_pre) {
    const size_t need = (size_t)(G + kResSplit) * P * sizeof(float);
    MHC_CHECK_ARG(workspace && workspace_bytes >= need && aligned(workspace, 16),
                  "workspace of %zu bytes is smaller than the %zu bytes required", workspace_bytes, need);
  }
  ResArgs A{};
  A.x = x; A.res = res; A.g = dout; A.gy = dy_agg; A.out = dx; A.out2 = dres; A.hpre = h_pre;
  A.part = dh_pre ? (float*)workspace : nullptr;
  A.T = T; A.n = n; A.C = C; A.nchunks = (int)ceil_div(C, kResV); A.h_mode = h_mode; A.P = P;
  const int gdt = dout ? dout_dtype : dtype;
  A.vec = res_vec_ok(C, kResV, {{x, dtype_bytes(dtype)}, {res, dtype_bytes(dtype)}, {dout, dtype_bytes(gdt)},
                         {dy_agg, 4}, {dx, dtype_bytes(dtype)}, {dres, dtype_bytes(dtype)}});
  hipStream_t s = (hipStream_t)stream;
  const int groups = (int)ceil_div(n, kResBwdGroup);
  int rc = res_by_dtype(dtype, [&](auto* xp) {
    using XT = std::remove_pointer_t<decltype(xp)>;
    auto launch = [&](auto* gp) {
      using GT = std::remove_pointer_t<decltype(gp)>;
      hipLaunchKernelGGL((residual_add_agg_bwd_kernel<kResBwdGroup, XT, GT>),
                         dim3((unsigned)G, (unsigned)groups), dim3(kResThreads), 0, s, A);
      MHC_CHECK_LAUNCH("residual_add_agg_bwd_kernel");
      return MHC_OK;
    };
    if (gdt == MHC_DTYPE_F32) return launch((float*)nullptr);
    return launch((XT*)nullptr);
  });
  if (rc != MHC_OK || !dh_pre) return rc;
  float* part2 = (float*)workspace + (size_t)G * P;
  const int S = (int)std::min<int64_t>(kResSplit, G);
  const int rows = (int)ceil_div(G, S);
  const int S_used = (int)ceil_div(G, rows);
  hipLaunchKernelGGL(reduce_rows_kernel, dim3((unsigned)ceil_div(P / 4, 256), (unsigned)S_used), dim3(256), 0,
                     s, (const float*)workspace, part2, G, P, rows);
  MHC_CHECK_LAUNCH("reduce_rows_kernel");
  hipLaunchKernelGGL(residual_final_kernel, dim3(1), dim3(64), 0, s, part2, S_used, P, n, h_mode, h_pre,
                     dh_pre);
  MHC_CHECK_LAUNCH("residual_final_kernel");
  return MHC_OK;
}
