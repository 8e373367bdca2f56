// Background-recompute and adjoint-state step launchers of the exact adjoint,
// FP16 levels with the non-temporal hint.
#include "born_ops.h"

namespace born {

BORN_SREC_STEP_HINT(template, 0, __half);
BORN_SREC_STEP_HINT(template, 1, __half);
BORN_LAM_STEP_HINT(template, __half);

}  // namespace born
