// Wide kernel instantiations: soft binning, bfloat16 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(__hip_bfloat16, true)
}  // namespace ace
