// lv.hpp's backward instantiated for x in f32.
#include "lv.hpp"

namespace mhc {

int lv_bwd_f32(const GenArgs& A, bool, int64_t gmax, hipStream_t s, int64_t* np) {
  return lv_bwd_typed<float, float>(A, gmax, s, np);
}

}  // namespace mhc
