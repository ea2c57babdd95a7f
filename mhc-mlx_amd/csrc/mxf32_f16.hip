// mxf32.hpp instantiated for x in f16.
#include "mxf32.hpp"

namespace mhc {

int mxf_fwd_f16(const MxfArgs& A, bool y_f32, bool o_f32, hipStream_t s) {
  return mxf_fwd_types<_Float16>(A, y_f32, o_f32, s);
}

int mxf_bwd_f16(const MxfArgs& A, bool y_f32, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  return mxf_bwd_types<_Float16>(A, y_f32, g_f32, gmax, s, np);
}

}  // namespace mhc
