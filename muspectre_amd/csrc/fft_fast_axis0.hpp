// First-axis pass with the projection: launchers and dispatch on length
// and variant, instantiated per precision in fft_fast_axis0.hip (FP64) and
// fft_fast_axis0_32.hip (FP32).
#pragma once
#include "fft_fast.hpp"

namespace mugpu {

namespace {

template <typename T, int N, int E, int DIM, int H, bool B, bool PK>
int axis0_n(FftPlan& p, const ProjParams& pj, void* spec) {
  XArgs<T> a{};
  a.data = reinterpret_cast<c_t<T>*>(spec);
  a.plane = p.kpts / p.res[0];
  a.tw = tw_of<T>(p, 0);
  a.kind = pj.kind;
  a.allow_even = pj.allow_even;
  for (int d = 0; d < 3; ++d) {
    a.res[d] = p.res[d];
    a.L[d] = pj.L[d];
  }
  a.hlast = p.hres[DIM - 1];
  a.norm = (T)pj.norm;
  a.active = p.active;
  constexpr int KP = x_kpts(N, DIM, sizeof(T) == 4, E, H), L = KP * nb_lines(DIM, PK), NT = L * (N / E);
  constexpr size_t lds = TwLds<T, N>::total(lds_axis0<T, N, E, DIM, H, PK>());
  const dim3 grid((unsigned)((a.plane + KP - 1) / KP));
  if constexpr (B)
    hipLaunchKernelGGL((k_axis0_bounded<T, N, E, DIM, H, PK>), grid, dim3(NT), lds, stream(), a);
  else
    hipLaunchKernelGGL((k_axis0_fast<T, N, E, DIM, H, PK>), grid, dim3(NT), lds, stream(), a);
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

// first-axis pass: bit 0 of the variant selects E = 8, bit 1 half the
// k-points per workgroup, bit 2 the kernel with the occupancy hint; a
// variant that changes nothing at this length runs the kernel it equals
template <typename T, int N, int E, int DIM, bool B>
int axis0_h(FftPlan& p, const ProjParams& pj, void* spec, int h) {
  if constexpr (sizeof(T) == 8)
    if (p.packed) {
      if constexpr (x_kpts(N, DIM, false, E, 1) != x_kpts(N, DIM, false, E, 0))
        if (h) return axis0_n<T, N, E, DIM, 1, B, true>(p, pj, spec);
      return axis0_n<T, N, E, DIM, 0, B, true>(p, pj, spec);
    }
  if constexpr (x_kpts(N, DIM, sizeof(T) == 4, E, 1) != x_kpts(N, DIM, sizeof(T) == 4, E, 0))
    if (h) return axis0_n<T, N, E, DIM, 1, B, false>(p, pj, spec);
  return axis0_n<T, N, E, DIM, 0, B, false>(p, pj, spec);
}
template <typename T, int N, int E, int DIM>
int axis0_hb(FftPlan& p, const ProjParams& pj, void* spec, int v) {
  if (v & 4) return axis0_h<T, N, E, DIM, true>(p, pj, spec, (v >> 1) & 1);
  return axis0_h<T, N, E, DIM, false>(p, pj, spec, (v >> 1) & 1);
}
template <typename T, int DIM>
int axis0_any(FftPlan& p, const ProjParams& pj, void* spec) {
  const int v = p.fvar[pi_of<T>()][FV_AXIS0][p.packed ? 2 : 0];
#define C_(n, e) axis0_hb<T, n, e, DIM>(p, pj, spec, v)
  MUGPU_FAST_SWITCH(p.res[0], v & 1, C_)
#undef C_
  return MUGPU_EARG;
}

}  // namespace
}  // namespace mugpu
