// mxf32.hpp instantiated for x in bf16.
#include "mxf32.hpp"

namespace mhc {

int mxf_fwd_bf16(const MxfArgs& A, bool y_f32, bool o_f32, hipStream_t s) {
  return mxf_fwd_types<__bf16>(A, y_f32, o_f32, s);
}

int mxf_bwd_bf16(const MxfArgs& A, bool y_f32, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  return mxf_bwd_types<__bf16>(A, y_f32, g_f32, gmax, s, np);
}

}  // namespace mhc
