// The multi-operation D2Q9 runs (multi2d.hpp) of one storage; a translation unit
// each, so that the build compiles them side by side.
#include "multi2d.hpp"

namespace vsx {

int multi2d_run_f16(const StepCtx &c, const float *f_in, float *f_out, void *wa, void *wb, int n, hipStream_t s) {
  return multi2d_run_any<Store<VSX_STORE_F16S>>(c, f_in, f_out, wa, wb, n, s);
}

}  // namespace vsx
