// First-axis pass in FP64, and the choice of the precision.
#include "fft_fast_axis0.hpp"

namespace mugpu {

int fast_axis0_project32(FftPlan& p, const ProjParams& pj, void* spec);

int fast_axis0_project(FftPlan& p, int prec, const ProjParams& pj, void* spec) {
  if (prec != MUGPU_FP64) return fast_axis0_project32(p, pj, spec);
  return p.dim == 3 ? axis0_any<double, 3>(p, pj, spec) : axis0_any<double, 2>(p, pj, spec);
}

}  // namespace mugpu
