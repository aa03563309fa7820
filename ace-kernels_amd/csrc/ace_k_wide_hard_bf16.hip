// Wide kernel instantiations: hard binning, bfloat16 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(__hip_bfloat16, false)
}  // namespace ace
