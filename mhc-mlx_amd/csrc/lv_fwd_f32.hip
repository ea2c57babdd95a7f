// lv.hpp's forward instantiated for x in f32, and the dispatch over x's dtype.
#include "lv.hpp"

namespace mhc {

int lv_fwd_f32(const GenArgs& A, bool, hipStream_t s) {
  return lv_fwd_typed<float, float>(A, s);
}

// offsets inside a token are 32-bit with room for the marks beyond it
static bool lv_fits(const GenArgs& A) { return A.n <= 8 && (int64_t)A.n * A.C * 4 < (int64_t)1 << 30; }

int lv_fused_fwd(const GenArgs& A, int xd, int od, hipStream_t s) {
  if (!lv_fits(A)) return 1;
  switch (xd) {
    case MHC_DTYPE_F32: return od == MHC_DTYPE_F32 ? lv_fwd_f32(A, true, s) : 1;
    case MHC_DTYPE_BF16: return lv_fwd_bf16(A, od == MHC_DTYPE_F32, s);
    case MHC_DTYPE_F16: return lv_fwd_f16(A, od == MHC_DTYPE_F32, s);
    default: return 1;
  }
}

int lv_fused_bwd(const GenArgs& A, int xd, int gd, int64_t gmax, hipStream_t s, int64_t* np) {
  if (!lv_fits(A)) return 1;
  switch (xd) {
    case MHC_DTYPE_F32: return gd == MHC_DTYPE_F32 ? lv_bwd_f32(A, true, gmax, s, np) : 1;
    case MHC_DTYPE_BF16: return lv_bwd_bf16(A, gd == MHC_DTYPE_F32, gmax, s, np);
    case MHC_DTYPE_F16: return lv_bwd_f16(A, gd == MHC_DTYPE_F32, gmax, s, np);
    default: return 1;
  }
}

}  // namespace mhc
