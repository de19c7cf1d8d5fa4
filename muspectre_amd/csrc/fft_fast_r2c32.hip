// Last-axis r2c pass in FP32.
#include "fft_fast_r2c.hpp"

namespace mugpu {

int fast_r2c32(FftPlan& p, const OpSpec& op, void* spec) {
  return p.dim == 3 ? r2c_any<float, 3>(p, op, spec) : r2c_any<float, 2>(p, op, spec);
}

}  // namespace mugpu
