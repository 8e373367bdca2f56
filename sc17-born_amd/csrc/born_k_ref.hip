// Launchers of the reference-mode loops: sourceProp and rtmAdjoint steps (the
// latter with s and r together: born_k_radj2.hip).
#include "born_ops.h"

namespace born {

hipError_t launch_src_step(const Geometry &geo, const Tune &tu, const SrcStep &a,
                           hipStream_t st) {
  SrcOp op{};
  op.s1 = a.s1; op.s0 = a.s0; op.vel = a.vel;
  op.pts = to_points(a.src); op.amp = a.amp;
  return launch(geo, tu, op, st);
}

BORN_RADJ_STEP(extern template, true);
BORN_RADJ_STEP(template, false);

hipError_t launch_radj_step(const Geometry &geo, const Tune &tu, const RadjStep &a,
                            hipStream_t st) {
  return a.pair ? radj_step<true>(geo, tu, a, st) : radj_step<false>(geo, tu, a, st);
}

}  // namespace born
