// lf32_bwd.hpp instantiated for x in f16.
#include "lf32_bwd.hpp"

namespace mhc {

int lf_bwd_f16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  return g_f32 ? lf_bwd_types<_Float16, float>(A, gmax, s, np) : lf_bwd_types<_Float16, _Float16>(A, gmax, s, np);
}

}  // namespace mhc
