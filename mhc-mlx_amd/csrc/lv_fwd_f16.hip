// lv.hpp's forward instantiated for x in f16.
#include "lv.hpp"

namespace mhc {

int lv_fwd_f16(const GenArgs& A, bool o_f32, hipStream_t s) {
  return o_f32 ? lv_fwd_typed<_Float16, float>(A, s) : lv_fwd_typed<_Float16, _Float16>(A, s);
}

}  // namespace mhc
