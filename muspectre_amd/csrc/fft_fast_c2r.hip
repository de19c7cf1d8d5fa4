// Last-axis c2r pass in FP64, and the choice of the precision.
#include "fft_fast_c2r.hpp"

namespace mugpu {

int fast_c2r32(FftPlan& p, const OpSpec& op, void* spec);

int fast_c2r(FftPlan& p, int prec, const OpSpec& op, void* spec) {
  if (prec != MUGPU_FP64) return fast_c2r32(p, op, spec);
  return p.dim == 3 ? c2r_any<double, 3>(p, op, spec) : c2r_any<double, 2>(p, op, spec);
}

}  // namespace mugpu
