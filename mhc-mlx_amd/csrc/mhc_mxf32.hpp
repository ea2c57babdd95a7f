// MHCRewire post-combine on fp32 MFMA for the shapes mix32.hip does not take
// (mxf32.hpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mhc_mix32.hpp"

namespace mhc {

struct MxfArgs : Mix32Args {
  uint32_t cols;  // T * C, below 2^31
  uint32_t cmul;  // column / C = umulhi(2 column, cmul) >> csh
  int csh;
};

// out = Mf X + p Y, any C and alignment; y and out fp32 or x's dtype.
// Returns 1 when not covered.
int mxf_fwd(const Mix32Args& A, int x_dtype, int y_dtype, int out_dtype, hipStream_t s);

// dx = Mf^T G, dy = p G and at most gmax partial rows of the sums; dout fp32
// or x's dtype.  Returns 1 when not covered.
int mxf_bwd(const Mix32Args& A, int x_dtype, int y_dtype, int g_dtype, int64_t gmax, hipStream_t s,
            int64_t* num_partials);

// One dtype of x each (one source file each: the kernels compile in parallel).
int mxf_fwd_bf16(const MxfArgs& A, bool y_f32, bool o_f32, hipStream_t s);
int mxf_fwd_f16(const MxfArgs& A, bool y_f32, bool o_f32, hipStream_t s);
int mxf_bwd_bf16(const MxfArgs& A, bool y_f32, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);
int mxf_bwd_f16(const MxfArgs& A, bool y_f32, bool g_f32, int64_t gmax, hipStream_t s, int64_t* num_partials);

}  // namespace mhc
