// Last-axis r2c pass (p update, K:p, r2c): launchers and dispatch on length
// and variant, instantiated per precision in fft_fast_r2c.hip (FP64) and
// fft_fast_r2c32.hip (FP32), which compile side by side.
#pragma once
#include "fft_fast.hpp"

namespace mugpu {

namespace {

template <typename T, int N, int E, int DIM, int IN, bool ISO, int H, bool PK>
void r2c_go(FftPlan& p, const LArgs<T>& a) {
  constexpr int RB = z_rows(N, DIM, H), NT = RB / 2 * nb_lines(DIM, PK) * (N / E);
  constexpr size_t lds = TwLds<T, N>::total(lds_r2c<T, N, DIM, IN, H, PK>());
  const dim3 grid((unsigned)((a.rows + RB - 1) / RB));
  if (sizeof(T) == 8) p.wg_r2c = grid.x;
  hipLaunchKernelGGL((k_r2c_fast<T, N, E, DIM, IN, ISO, H, PK>), grid, dim3(NT), lds, stream(), a);
}

template <typename T, int N, int E, int DIM, int H>
int r2c_n(FftPlan& p, const OpSpec& op, void* spec) {
  LArgs<T> a{};
  a.in = reinterpret_cast<const T*>(op.in);
  a.rvec = reinterpret_cast<const T*>(op.rvec);
  a.pout = reinterpret_cast<T*>(op.pout);
  a.scal = op.scal;
  a.tan = reinterpret_cast<const T*>(op.tangent);
  a.tan_kind = op.tan_kind;
  a.spec = reinterpret_cast<c_t<T>*>(spec);
  a.rows = p.N / N;
  a.tw = tw_of<T>(p, DIM - 1);
  a.active = p.active;
  a.x = reinterpret_cast<T*>(op.xvec);
  a.partials = op.fin_alpha ? reinterpret_cast<double*>(p.partials) : nullptr;
  if (sizeof(T) == 8) {
    a.fold = p.fold;
    if (a.fold.pk) a.partials = a.fold.pk;
  }
  const bool iso = op.tan_kind == TAN_ISO;
  // the fused x update goes with the p update only
  const bool xu = op.xvec != nullptr;
  if (xu && (op.in_mode != IN_TAN_PUPDATE || op.sym)) return MUGPU_EARG;
  if constexpr (sizeof(T) == 8) {
    a.sym = op.sym_flags;
    if (p.packed) {
      if (op.sym) r2c_go<T, N, E, DIM, IN_TAN_S, true, H, true>(p, a);
      else if (op.in_mode == IN_PLAIN) r2c_go<T, N, E, DIM, IN_PLAIN, false, H, true>(p, a);
      else if (op.in_mode == IN_TAN) r2c_go<T, N, E, DIM, IN_TAN, true, H, true>(p, a);
      else if (xu) r2c_go<T, N, E, DIM, IN_TAN_PUPDATE_X, true, H, true>(p, a);
      else r2c_go<T, N, E, DIM, IN_TAN_PUPDATE, true, H, true>(p, a);
      MUGPU_HIP(hipGetLastError());
      return MUGPU_OK;
    }
  }
  // the isotropic forms of a CG iteration run in FP64 with packed lines; the
  // few grids that cannot pack take the run-time switch of the general form
  constexpr bool ISO_PU = sizeof(T) == 4;
  if (op.in_mode == IN_PLAIN) r2c_go<T, N, E, DIM, IN_PLAIN, false, H, false>(p, a);
  else if (op.in_mode == IN_TAN && iso) r2c_go<T, N, E, DIM, IN_TAN, true, H, false>(p, a);
  else if (op.in_mode == IN_TAN) r2c_go<T, N, E, DIM, IN_TAN, false, H, false>(p, a);
  else if (iso && xu) r2c_go<T, N, E, DIM, IN_TAN_PUPDATE_X, ISO_PU, H, false>(p, a);
  else if (iso) r2c_go<T, N, E, DIM, IN_TAN_PUPDATE, ISO_PU, H, false>(p, a);
  else if (xu) r2c_go<T, N, E, DIM, IN_TAN_PUPDATE_X, false, H, false>(p, a);
  else r2c_go<T, N, E, DIM, IN_TAN_PUPDATE, false, H, false>(p, a);
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

// last-axis passes: bit 0 of the variant selects E = 8, bit 1 half the rows
// per workgroup; a variant that changes nothing at this length runs the
// kernel it equals
template <typename T, int N, int E, int DIM>
int r2c_h(FftPlan& p, const OpSpec& op, void* spec, int h) {
  if constexpr (z_rows(N, DIM, 1) != z_rows(N, DIM, 0))
    if (h) return r2c_n<T, N, E, DIM, 1>(p, op, spec);
  return r2c_n<T, N, E, DIM, 0>(p, op, spec);
}
template <typename T, int DIM>
int r2c_any(FftPlan& p, const OpSpec& op, void* spec) {
  const int v = p.fvar[pi_of<T>()][FV_R2C][p.packed ? 2 : op.tan_kind == TAN_ISO ? 1 : 0];
#define C_(n, e) r2c_h<T, n, e, DIM>(p, op, spec, v >> 1)
  MUGPU_FAST_SWITCH(p.res[DIM - 1], v & 1, C_)
#undef C_
  return MUGPU_EARG;
}

}  // namespace
}  // namespace mugpu
