// The layer at n <= 8 on the VALU for rows of any width and alignment (lv.hpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mhc_generic.hpp"

namespace mhc {

// out = M x + p * rms_norm(a^T x) w, n <= 8, layer-wide or per-token
// parameters.  Returns 1 when the shape is not covered.
int lv_fused_fwd(const GenArgs& A, int x_dtype, int out_dtype, hipStream_t s);

// Partial-sums pass of the VJP, n <= 8 (outputs as lf32_fused_bwd's).
// Returns 1 when the shape is not covered.
int lv_fused_bwd(const GenArgs& A, int x_dtype, int g_dtype, int64_t gmax, hipStream_t s, int64_t* num_partials);

// One dtype of x each (one source file each: the kernels compile in parallel).
int lv_fwd_f32(const GenArgs& A, bool o_f32, hipStream_t s);
int lv_fwd_bf16(const GenArgs& A, bool o_f32, hipStream_t s);
int lv_fwd_f16(const GenArgs& A, bool o_f32, hipStream_t s);
int lv_bwd_f32(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);
int lv_bwd_bf16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);
int lv_bwd_f16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);

}  // namespace mhc
