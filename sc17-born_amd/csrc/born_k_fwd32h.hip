// Born forward step launchers, FP32 levels of s and r together, with the
// non-temporal hint.
#include "born_ops.h"

namespace born {

BORN_FWD_STEP_HINT(template, 0);
BORN_FWD_STEP_HINT(template, 1);

}  // namespace born
