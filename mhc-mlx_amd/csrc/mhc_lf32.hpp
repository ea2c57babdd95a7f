// The layer on fp32 MFMA for every 8 < n <= 64 shape that the 16-bit MFMA
// kernels do not take: fp32 or mixed dtypes, channel counts that are no
// multiple of 128, unaligned rows (lf32_fwd.hip, lf32_bwd.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mhc_device.hpp"
#include "mhc_generic.hpp"

namespace mhc {

// out = M x + p * rms_norm(a^T x) w; layer-wide or per-token parameters.
// Returns 1 when the shape is not covered.
int lf32_fused_fwd(const GenArgs& A, int x_dtype, int out_dtype, hipStream_t s);

// Partial-sums pass of the VJP: dx, and one partial row per workgroup
// [dw C | pad | dM n*n | dA n | dP n] (at most gmax workgroups); per token
// parameters: the token's dM, dh_pre and dh_post, and [dw C | pad] rows.
// Returns 1 when the shape is not covered.
int lf32_fused_bwd(const GenArgs& A, int x_dtype, int g_dtype, int64_t gmax, hipStream_t s, int64_t* num_partials);

// lf32_fused_bwd for one dtype of x (one source file each: the kernels compile in parallel).
int lf_bwd_bf16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);
int lf_bwd_f16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);

constexpr int kLfSlab = 64;       // channels per slab: four per lane of a 16-lane group
constexpr int kLfMaxWaves = 8;    // waves per workgroup
constexpr uint32_t kLfOut = 0x80000000u;  // a byte offset beyond every token (tokens stay below 2 GiB)

MHC_DEV f32x4 lf_mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// A token's n rows as a buffer resource: rows past n load as zero and their
// stores are dropped.
template <typename T>
MHC_DEV __amdgpu_buffer_rsrc_t lf_rsrc(const T* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)bytes, 0x00020000);
}

// Hides v from the compiler: an address formed from it is computed where it is used, instead of once per row and held
// in a register for the whole kernel.
MHC_DEV uint32_t lf_opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// How a slab's rows are accessed.  kLfElem: any C and alignment, channels r,
// r + 16, r + 32, r + 48 of the slab by one access each (a 16-lane group reads
// consecutive elements).  kLfVec (C a multiple of 4, rows aligned to four
// elements): channels 4r .. 4r + 3 in one access.  kLfLine: rows that are
// whole 128-byte lines as well.  Only those carry the non-temporal hint: a
// line shared by two rows or slabs is then fetched, and written, twice
// (4096 x 12 x 2001 bf16 forward 205 us with the hint, 151 us without;
// 4096 x 16 x 1024 fp32, whole lines, 92 us with, 101 us without).
enum LfMode : int { kLfElem = 0, kLfVec = 1, kLfLine = 2 };
constexpr int lf_aux(int mode) { return mode == kLfLine ? 2 : 0; }

// The mode of a call whose rows are C elements of t1 and t2 bytes at aligned4 (every operand aligned to four elements).
inline int lf_mode(int C, int t1, int t2, bool aligned4) {
  if (C % 4 != 0 || !aligned4) return kLfElem;
  return (int64_t)C * t1 % 128 == 0 && (int64_t)C * t2 % 128 == 0 ? kLfLine : kLfVec;
}

// Four channels of one stream row of a 64-channel slab, as stored.
template <bool VEC>
MHC_DEV int lf_chan(int r, int v) { return VEC ? 4 * r + v : r + 16 * v; }

template <bool VEC>
struct LfOff {
  uint32_t o[VEC ? 1 : 4];
  // byte offsets of the lane's channels of slab s in the row that starts at `row` bytes; channels past C are out
  // of the resource
  MHC_DEV void set(uint32_t row, int s, int r, int C, int elem) {
#pragma unroll
    for (int v = 0; v < (VEC ? 1 : 4); ++v) {
      const int c = s * kLfSlab + lf_chan<VEC>(r, v);
      o[v] = c < C ? row + (uint32_t)(c * elem) : kLfOut;
    }
  }
  MHC_DEV LfOff fresh() const {
    LfOff f;
#pragma unroll
    for (int v = 0; v < (VEC ? 1 : 4); ++v) f.o[v] = lf_opaque(o[v]);
    return f;
  }
};

template <typename T, bool VEC>
struct LfQuad {
  static constexpr int kWords = VEC ? (int)sizeof(T) : 4;
  uint32_t w[kWords];

  template <int AUX>
  MHC_DEV void load(__amdgpu_buffer_rsrc_t rs, const LfOff<VEC>& off, uint32_t add) {
    if constexpr (VEC && sizeof(T) == 4) {
      const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(rs, off.o[0] + add, 0, AUX);
      w[0] = u.x; w[1] = u.y; w[2] = u.z; w[3] = u.w;
    } else if constexpr (VEC) {
      const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rs, off.o[0] + add, 0, AUX);
      w[0] = u.x; w[1] = u.y;
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if constexpr (sizeof(T) == 4) w[v] = __builtin_amdgcn_raw_buffer_load_b32(rs, off.o[v] + add, 0, AUX);
        else w[v] = __builtin_amdgcn_raw_buffer_load_b16(rs, off.o[v] + add, 0, AUX);
      }
    }
  }
  MHC_DEV float get(int v) const {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, w[v]);
    else if constexpr (VEC) return (v & 1) ? hi16<T>(w[v >> 1]) : lo16<T>(w[v >> 1]);
    else return lo16<T>(w[v]);
  }
};

template <typename T, bool VEC, int AUX>
MHC_DEV void lf_store(__amdgpu_buffer_rsrc_t rs, const LfOff<VEC>& off, uint32_t add, const float (&v)[4]) {
  if constexpr (VEC && sizeof(T) == 4) {
    const u32x4 u = {__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                     __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3])};
    buf_store_b128<AUX>(u, rs, off.o[0] + add, 0);
  } else if constexpr (VEC) {
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])}, rs, off.o[0] + add, 0, AUX);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (sizeof(T) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[k]), rs, off.o[k] + add, 0, AUX);
      else
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)bits16<T>(v[k]), rs, off.o[k] + add, 0, AUX);
    }
  }
}

// The sum over the four lane groups q (lanes r, r + 16, r + 32, r + 48), on all of them.
MHC_DEV float lf_sum_q(float v) { return xor_allreduce<32>(xor_allreduce<16>(v, SumOp{}), SumOp{}); }

// Entry (i, j) of an n x n matrix, zero past n (the load address stays inside the matrix).
MHC_DEV float lf_entry(const float* M, int i, int j, int n) {
  const bool in = i < n && j < n;
  const float v = M[in ? i * n + j : 0];
  return in ? v : 0.0f;
}

// The [n] raw or activated values of a token, one per lane (zero past n): each is evaluated once per wave and fetched
// by the lanes that need it.
MHC_DEV float lf_act(float v, int i, int n, bool raw, float scale) {
  const float s = raw ? scale * sigmoidf_(v) : v;
  return i < n ? s : 0.0f;
}
MHC_DEV float lf_lane(float v, int from) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from << 2, __builtin_bit_cast(int, v)));
}

}  // namespace mhc
