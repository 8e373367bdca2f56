// Background-recompute and adjoint-state step launchers of the exact adjoint,
// 24-bit levels with the non-temporal hint.
#include "born_ops.h"

namespace born {

BORN_SREC_STEP_HINT(template, 0, Split);
BORN_SREC_STEP_HINT(template, 1, Split);
BORN_LAM_STEP_HINT(template, Split);

}  // namespace born
