// First-axis pass in FP32.
#include "fft_fast_axis0.hpp"

namespace mugpu {

int fast_axis0_project32(FftPlan& p, const ProjParams& pj, void* spec) {
  return p.dim == 3 ? axis0_any<float, 3>(p, pj, spec) : axis0_any<float, 2>(p, pj, spec);
}

}  // namespace mugpu
