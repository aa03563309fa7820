// Wide kernel instantiations: soft binning, float32 logits.
#include "ace_wide.hpp"

namespace ace {
ACE_DEFINE_WIDE(float, true)
}  // namespace ace
