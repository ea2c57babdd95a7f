// lf32_bwd.hpp instantiated for x in f32, and the dispatch over x's dtype.
#include "lf32_bwd.hpp"

namespace mhc {

int lf_bwd_f32(const GenArgs& A, int64_t gmax, hipStream_t s, int64_t* np) {
  return lf_bwd_types<float, float>(A, gmax, s, np);
}

int lf32_fused_bwd(const GenArgs& A, int xd, int gd, int64_t gmax, hipStream_t s, int64_t* np) {
  if (knob(kKnobBwdMfma, 1) == 0) return 1;
  // offsets inside a token are 32-bit, with the top bit for "outside"
  if ((int64_t)A.n * A.C * 4 >= (int64_t)1 << 31 || A.n > 64) return 1;
  switch (xd) {
    case MHC_DTYPE_F32: return gd == MHC_DTYPE_F32 ? lf_bwd_f32(A, gmax, s, np) : 1;
    case MHC_DTYPE_BF16: return lf_bwd_bf16(A, gd == MHC_DTYPE_F32, gmax, s, np);
    case MHC_DTYPE_F16: return lf_bwd_f16(A, gd == MHC_DTYPE_F32, gmax, s, np);
    default: return 1;
  }
}

}  // namespace mhc
