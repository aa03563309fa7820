// Wide kernel instantiations: soft binning, float16 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(__half, true)
}  // namespace ace
