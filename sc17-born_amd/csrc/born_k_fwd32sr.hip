// Born forward step launchers, FP32 levels of s and r together (both scatter
// terms).
#include "born_ops.h"

namespace born {

BORN_FWD_STEP_SR(template, 0);
BORN_FWD_STEP_SR(template, 1);

}  // namespace born
