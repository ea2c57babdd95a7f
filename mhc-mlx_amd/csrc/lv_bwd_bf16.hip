// lv.hpp's backward instantiated for x in bf16.
#include "lv.hpp"

namespace mhc {

int lv_bwd_bf16(const GenArgs& A, bool g_f32, int64_t gmax, hipStream_t s, int64_t* np) {
  return g_f32 ? lv_bwd_typed<__bf16, float>(A, gmax, s, np) : lv_bwd_typed<__bf16, __bf16>(A, gmax, s, np);
}

}  // namespace mhc
