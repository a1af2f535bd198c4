// The segmented walks of f16 rows (em_walk.h).

#include "em_walk.h"

namespace rem {

hipError_t tape_walk_f16(const WalkArgs& a, int ub, int ks, bool fwd, hipStream_t s) {
  switch (ub) {
    case 16: return tape_walk_unit<kF16, 16>(a, ks, fwd, s);
    case 4: return tape_walk_unit<kF16, 4>(a, ks, fwd, s);
    case 2: return tape_walk_unit<kF16, 2>(a, ks, fwd, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rem
