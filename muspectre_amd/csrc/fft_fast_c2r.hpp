// Last-axis c2r pass (c2r, p.Ap partials or the r update): launchers and
// dispatch on length and variant, instantiated per precision in
// fft_fast_c2r.hip (FP64) and fft_fast_c2r32.hip (FP32).
#pragma once
#include "fft_fast.hpp"

namespace mugpu {

namespace {

template <typename T, int N, int E, int DIM, int OUT, int H, bool PK>
void c2r_go(FftPlan& p, const LArgs<T>& a) {
  constexpr int RB = z_rows(N, DIM, H), NT = RB / 2 * nb_lines(DIM, PK) * (N / E);
  constexpr size_t lds = TwLds<T, N>::total(lds_c2r<T, N, E, DIM, H, PK>());
  const dim3 grid((unsigned)((a.rows + RB - 1) / RB));
  if (sizeof(T) == 8) p.wg_c2r = grid.x;
  hipLaunchKernelGGL((k_c2r_fast<T, N, E, DIM, OUT, H, PK>), grid, dim3(NT), lds, stream(), a);
}

template <typename T, int N, int E, int DIM, int H>
int c2r_n(FftPlan& p, const OpSpec& op, void* spec) {
  LArgs<T> a{};
  a.spec = reinterpret_cast<c_t<T>*>(spec);
  a.out = reinterpret_cast<T*>(op.out);
  a.dotv = reinterpret_cast<const T*>(op.dotv);
  a.partials = reinterpret_cast<double*>(p.partials);
  a.rows = p.N / N;
  a.tw = tw_of<T>(p, DIM - 1);
  a.active = p.active;
  if constexpr (sizeof(T) == 8) {
    a.scal = op.scal;
    a.ap = reinterpret_cast<T*>(op.ap_out);
    a.fold = p.fold;
    a.rvec = reinterpret_cast<const T*>(op.rvec);
    a.sym = op.sym_flags;
    if (p.packed) {
      if (op.sym) c2r_go<T, N, E, DIM, OUT_RUPD_S, H, true>(p, a);
      else if (op.out_mode == OUT_RUPD) c2r_go<T, N, E, DIM, OUT_RUPD, H, true>(p, a);
      else if (op.out_mode == OUT_DOT) c2r_go<T, N, E, DIM, OUT_DOT, H, true>(p, a);
      else c2r_go<T, N, E, DIM, OUT_PLAIN, H, true>(p, a);
      MUGPU_HIP(hipGetLastError());
      return MUGPU_OK;
    }
    if (op.out_mode == OUT_RUPD) {
      c2r_go<T, N, E, DIM, OUT_RUPD, H, false>(p, a);
      MUGPU_HIP(hipGetLastError());
      return MUGPU_OK;
    }
  }
  if (op.out_mode == OUT_DOT) c2r_go<T, N, E, DIM, OUT_DOT, H, false>(p, a);
  else c2r_go<T, N, E, DIM, OUT_PLAIN, H, false>(p, a);
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

// last-axis passes: bit 0 of the variant selects E = 8, bit 1 half the rows
// per workgroup; a variant that changes nothing at this length runs the
// kernel it equals
template <typename T, int N, int E, int DIM>
int c2r_h(FftPlan& p, const OpSpec& op, void* spec, int h) {
  if constexpr (z_rows(N, DIM, 1) != z_rows(N, DIM, 0))
    if (h) return c2r_n<T, N, E, DIM, 1>(p, op, spec);
  return c2r_n<T, N, E, DIM, 0>(p, op, spec);
}
template <typename T, int DIM>
int c2r_any(FftPlan& p, const OpSpec& op, void* spec) {
  const int v = p.fvar[pi_of<T>()][FV_C2R][p.packed ? 2 : 0];
#define C_(n, e) c2r_h<T, n, e, DIM>(p, op, spec, v >> 1)
  MUGPU_FAST_SWITCH(p.res[DIM - 1], v & 1, C_)
#undef C_
  return MUGPU_EARG;
}

}  // namespace
}  // namespace mugpu
