// Wide kernel instantiations: hard binning, float16 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(__half, false)
}  // namespace ace
