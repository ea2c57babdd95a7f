// lv.hpp's forward instantiated for x in bf16.
#include "lv.hpp"

namespace mhc {

int lv_fwd_bf16(const GenArgs& A, bool o_f32, hipStream_t s) {
  return o_f32 ? lv_fwd_typed<__bf16, float>(A, s) : lv_fwd_typed<__bf16, __bf16>(A, s);
}

}  // namespace mhc
