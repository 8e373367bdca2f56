// The rtmAdjoint step with the levels of s and r together.
#include "born_ops.h"

namespace born {

BORN_RADJ_STEP(template, true);

}  // namespace born
