// The segmented walks of f64 rows (em_walk.h).

#include "em_walk.h"

namespace rem {

hipError_t tape_walk_f64(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s) {
  switch (ub) {
    case 8: return tape_walk_unit<kF64, 8>(a, ks, fwd, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rem
