// lf32_bwd.hpp instantiated for x in bf16.
#include "lf32_bwd.hpp"

namespace mhc {

int lf_bwd_bf16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  return g_f32 ? lf_bwd_types<__bf16, float>(A, gmax, s, np) : lf_bwd_types<__bf16, __bf16>(A, gmax, s, np);
}

}  // namespace mhc
