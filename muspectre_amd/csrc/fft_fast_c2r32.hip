// Last-axis c2r pass in FP32.
#include "fft_fast_c2r.hpp"

namespace mugpu {

int fast_c2r32(FftPlan& p, const OpSpec& op, void* spec) {
  return p.dim == 3 ? c2r_any<float, 3>(p, op, spec) : c2r_any<float, 2>(p, op, spec);
}

}  // namespace mugpu
