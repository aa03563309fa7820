// Wide kernel instantiations: hard binning, float32 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(float, false)
}  // namespace ace
