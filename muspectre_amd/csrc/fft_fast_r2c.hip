// Last-axis r2c pass in FP64, and the choice of the precision.
#include "fft_fast_r2c.hpp"

namespace mugpu {

int fast_r2c32(FftPlan& p, const OpSpec& op, void* spec);

int fast_r2c(FftPlan& p, int prec, const OpSpec& op, void* spec) {
  if (prec != MUGPU_FP64) return fast_r2c32(p, op, spec);
  return p.dim == 3 ? r2c_any<double, 3>(p, op, spec) : r2c_any<double, 2>(p, op, spec);
}

}  // namespace mugpu
