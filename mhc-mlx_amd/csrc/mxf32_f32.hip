// mxf32.hpp instantiated for x in f32, and the dispatch over x's dtype.
#include "mxf32.hpp"

namespace mhc {

namespace {

bool mxf_prepare(const Mix32Args& A, MxfArgs& B) {
  if (knob(kKnobMix32, 1) == 0 || A.n > 64 || A.T < 1) return false;
  // columns in 31 bits; a slab's offsets (its tokens' rows) in 31 bits of bytes
  if (A.T > ((int64_t)1 << 31) / A.C - 1 || (int64_t)A.n * (2 * (int64_t)A.C + kLfSlab) * 4 >= (int64_t)1 << 31) return false;
  static_cast<Mix32Args&>(B) = A;
  B.cols = (uint32_t)(A.T * A.C);
  B.csh = 0;
  while (((int64_t)1 << B.csh) < A.C) ++B.csh;
  B.cmul = (uint32_t)((((uint64_t)1 << (31 + B.csh)) + (uint64_t)A.C - 1) / (uint64_t)A.C);
  return true;
}

}  // namespace

int mxf_fwd(const Mix32Args& A, int xd, int yd, int od, hipStream_t s) {
  MxfArgs B;
  if ((yd != MHC_DTYPE_F32 && yd != xd) || (od != MHC_DTYPE_F32 && od != xd) || !mxf_prepare(A, B)) return 1;
  const bool yf = yd == MHC_DTYPE_F32, of = od == MHC_DTYPE_F32;
  switch (xd) {
    case MHC_DTYPE_F32: return mxf_fwd_types<float>(B, yf, of, s);
    case MHC_DTYPE_BF16: return mxf_fwd_bf16(B, yf, of, s);
    case MHC_DTYPE_F16: return mxf_fwd_f16(B, yf, of, s);
    default: return 1;
  }
}

int mxf_bwd(const Mix32Args& A, int xd, int yd, int gd, int64_t gmax, hipStream_t s, int64_t* np) {
  MxfArgs B;
  if ((yd != MHC_DTYPE_F32 && yd != xd) || (gd != MHC_DTYPE_F32 && gd != xd) || !mxf_prepare(A, B)) return 1;
  const bool yf = yd == MHC_DTYPE_F32, gf = gd == MHC_DTYPE_F32;
  switch (xd) {
    case MHC_DTYPE_F32: return mxf_bwd_types<float>(B, yf, gf, gmax, s, np);
    case MHC_DTYPE_BF16: return mxf_bwd_bf16(B, yf, gf, gmax, s, np);
    case MHC_DTYPE_F16: return mxf_bwd_f16(B, yf, gf, gmax, s, np);
    default: return 1;
  }
}

}  // namespace mhc
