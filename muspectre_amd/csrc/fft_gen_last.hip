// Last-axis passes of grids whose last axis has a run-time length: r2c
// with the CG direction update and K : p in front, c2r with the p . Ap partial
// sums behind.
//
// Two rows share a complex line (row 2q in the real part, 2q + 1 in the
// imaginary part), separated after the forward transform and combined before
// the backward one by Hermitian symmetry, as in fft_fast.hpp.  Rows are
// contiguous in HBM: every global access is an element-wise sweep of a row by
// consecutive lanes.
#include "fft_gen.hpp"

namespace mugpu {

namespace {

template <typename T>
struct GLast {
  const T* in;
  const T* rvec;
  T* pout;
  const double* scal;
  const T* tan;
  int tan_kind;
  c_t<T>* spec;
  T* out;
  T* x;
  T* ap;
  const T* dotv;
  double* partials;
  int64_t rows;
  int RB, L, P, LS;  // rows and lines per workgroup, threads per line, LDS line stride
  GenAxis ax;
  const c_t<T>* tw;
  const int* active;  // FftPlan::active
  ScalarFold fold;
  int sym;  // SymFlags
};

// LDS: [lines: n * LS complex][twiddles: n complex][staging: 2 rows of NC
// values per point].  The updated p of two rows is staged as it lies in memory
// and read back a voxel per thread (a lane stride of NC doubles, odd in 3D: no
// bank conflict), so that r, p are read and p is written in full cache lines.
template <typename T, int CLS, int DIM, int IN, bool PK>
__global__ __launch_bounds__(kGenMaxNT) void k_gen_r2c(GLast<T> a) {
  constexpr int NC = DIM * DIM, NL = nb_lines(DIM, PK);
  extern __shared__ __align__(16) unsigned char smem[];
  const int n = a.ax.n, LS = a.LS, nh = n / 2 + 1, NT = blockDim.x;
  c_t<T>* s = reinterpret_cast<c_t<T>*>(smem);
  T* sr = reinterpret_cast<T*>(smem);
  __shared__ double red[16];
  c_t<T>* tw = s + n * LS;
  T* sp = reinterpret_cast<T*>(tw + n);
  // (the flag and the partial sums are read together)
  const int on = a.active ? a.active[0] : 1;
  const int64_t row0 = (int64_t)blockIdx.x * a.RB;
  constexpr bool S = IN == IN_TAN_S, XU = IN == IN_TAN_PUPDATE_X;
  constexpr bool PU = IN == IN_TAN_PUPDATE || XU || S;
  constexpr int NF = S ? NL : NC;  // components of the staged field
  double beta = PU ? a.scal[SC_BETA] : 0.0;
  const double rr = PU && a.fold.rr ? fold_sum(a.fold.rr, a.fold.nrr, red) : 0.0;
  if (!on || (PU && a.fold.rr && !fold_beta_test(a.fold, rr, beta))) return;
  const double al = XU ? a.scal[SC_ALPHA] : 0.0;
  double acc = 0.0;  // p . K p
  for (int r0 = 0; r0 < a.RB; r0 += 2) {
    const int64_t base = (row0 + r0) * n * NF, lim = a.rows * n * NF;
    const int tot = 2 * n * NF;
    constexpr int KB = 4;
    if (r0) __syncthreads();  // the staged rows before have been read
    if constexpr (S) {
      sym_stage<T, DIM, KB>(a.in, a.rvec, a.pout, a.sym, (T)beta, base, lim, tot, NT, sp);
    } else for (int e0 = 0; e0 < tot; e0 += KB * NT) {
      T pv[KB], rv[KB], xv[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + threadIdx.x;
        const int64_t g = e < tot && base + e < lim ? base + e : lim - 1;
        pv[i] = a.in[g];
        if (PU) rv[i] = a.rvec[g];
        if (XU) xv[i] = a.x[g];
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + threadIdx.x;
        if (e < tot) {
          T x = T(0);
          if (base + e < lim) {
            x = pv[i];
            if (XU) a.x[base + e] = xv[i] + (T)al * x;
            if (PU) {
              x = -rv[i] + (T)beta * x;
              a.pout[base + e] = x;
            }
          }
          sp[e] = x;
        }
      }
    }
    if (r0 == 0) gen_twiddles<T>(tw, a.tw, n);
    __syncthreads();
    // rows beyond the last one hold zeros, for which K : p is not evaluated
    auto voxels = [&](auto kind_c) {
      constexpr int KIND = decltype(kind_c)::value;
      for (int e = threadIdx.x; e < 2 * n; e += NT) {
        const int r = e >= n, m = e - r * n;
        T p[NC], dp[NC];
        if constexpr (S) {
          unpack_lines<T, DIM>(sp + e * NF, p);
        } else {
#pragma unroll
          for (int c = 0; c < NC; ++c) p[c] = sp[e * NC + c];
        }
        if (KIND >= 0 && row0 + r0 + r < a.rows) {
          tangent_product<T, DIM>(KIND, a.tan, (row0 + r0 + r) * n + m, p, dp);
#pragma unroll
          for (int c = 0; c < NC; ++c) acc += (double)p[c] * (double)dp[c];
        } else {
#pragma unroll
          for (int c = 0; c < NC; ++c) dp[c] = p[c];
        }
        T q[NL];
        pack_lines<T, DIM, PK>(dp, q);
        T* o = sr + 2 * (m * LS + (r0 >> 1) * NL) + r;
#pragma unroll
        for (int c = 0; c < NL; ++c) o[2 * c] = q[c];
      }
    };
    if constexpr (IN == IN_PLAIN) {
      voxels(std::integral_constant<int, -1>{});
    } else if constexpr (PK) {
      voxels(std::integral_constant<int, TAN_ISO>{});
    } else {
      switch (a.tan_kind) {
        case TAN_SYM: voxels(std::integral_constant<int, TAN_SYM>{}); break;
        case TAN_HEP: voxels(std::integral_constant<int, TAN_HEP>{}); break;
        case TAN_LEF: voxels(std::integral_constant<int, TAN_LEF>{}); break;
        case TAN_HCT:
          if constexpr (DIM == 3) voxels(std::integral_constant<int, TAN_HCT>{});
          break;
        case TAN_ISO: voxels(std::integral_constant<int, TAN_ISO>{}); break;
        default: voxels(std::integral_constant<int, TAN_FULL>{}); break;
      }
    }
  }
  __syncthreads();
  const int p = threadIdx.x / a.L, l = threadIdx.x - p * a.L;
  auto none_ld = [](int) { return c_t<T>{}; };
  auto none_st = [](int, c_t<T>) {};
  gen_fft<T, CLS, -1, false, false>(a.ax, a.P, p, p < a.P, s + l, LS, tw, none_ld, none_st);
  for (int r = 0; r < a.RB; ++r) {
    if (row0 + r >= a.rows) break;
    c_t<T>* o = a.spec + (row0 + r) * nh * NL;
    const c_t<T>* sl = s + (r >> 1) * NL;
    for (int e = threadIdx.x; e < nh * NL; e += NT) {
      const int k = e / NL, c = e - k * NL;
      const c_t<T> z = sl[k * LS + c], zc = sl[(k == 0 ? 0 : n - k) * LS + c];
      c_t<T> X;
      if (!(r & 1)) {
        X.x = T(0.5) * (z.x + zc.x);
        X.y = T(0.5) * (z.y - zc.y);
      } else {
        X.x = T(0.5) * (z.y + zc.y);
        X.y = T(-0.5) * (z.x - zc.x);
      }
      o[e] = X;
    }
  }
  if (IN != IN_PLAIN && a.partials) {
    const double t = block_sum_waves(acc, red, NT);
    if (threadIdx.x == 0) a.partials[blockIdx.x] = t;
  }
}

// LDS: [lines][twiddles]; the half lines of a workgroup are staged over the
// lines, combined through registers (kGenVals values per thread at most, which
// P guarantees) and transformed in place.
template <typename T, int CLS, int DIM, int OUT, bool PK>
__global__ __launch_bounds__(kGenMaxNT) void k_gen_c2r(GLast<T> a) {
  constexpr int NC = DIM * DIM, NL = nb_lines(DIM, PK);
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[16];
  const int n = a.ax.n, LS = a.LS, nh = n / 2 + 1, NT = blockDim.x, RB = a.RB;
  c_t<T>* s = reinterpret_cast<c_t<T>*>(smem);
  const int stage = RB * nh * NL;  // staged values; the twiddles follow the larger of the two
  c_t<T>* tw = s + (n * LS > stage ? n * LS : stage);
  const int on = a.active ? a.active[0] : 1;
  constexpr bool S = OUT == OUT_RUPD_S, RU = OUT == OUT_RUPD || S;
  const bool fold = RU && a.fold.pk;
  const double pk = fold ? fold_sum(a.fold.pk, a.fold.npk, red) : 0.0;
  if (!on) return;
  const double alpha = fold ? fold_alpha(a.fold, pk) : 0.0;
  const int64_t row0 = (int64_t)blockIdx.x * RB;
  {
    const int64_t base = row0 * nh * NL, lim = a.rows * nh * NL;
    constexpr int KB = 4;
    for (int e0 = 0; e0 < stage; e0 += KB * NT) {
      c_t<T> t[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + threadIdx.x;
        t[i] = a.spec[e < stage && base + e < lim ? base + e : lim - 1];
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + threadIdx.x;
        if (e < stage) s[e] = base + e < lim ? t[i] : c_t<T>{};
      }
    }
  }
  gen_twiddles<T>(tw, a.tw, n);
  __syncthreads();
  const int p = threadIdx.x / a.L, l = threadIdx.x - p * a.L;
  const bool act = p < a.P;
  {
    const int rp = l / NL, c = l - rp * NL;
    const c_t<T>* A0 = s + (2 * rp) * nh * NL + c;
    const c_t<T>* B0 = A0 + nh * NL;
    c_t<T> v[kGenVals];
#pragma unroll
    for (int i = 0; i < kGenVals; ++i) {
      const int m = p + i * a.P;
      if (act && m < n) {
        const int kk = m < nh ? m : n - m;
        c_t<T> A = A0[kk * NL], B = B0[kk * NL];
        if (kk == 0 || 2 * kk == n) A.y = B.y = T(0);
        if (m >= nh) {
          A.y = -A.y;
          B.y = -B.y;
        }
        v[i].x = A.x - B.y;
        v[i].y = A.y + B.x;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kGenVals; ++i) {
      const int m = p + i * a.P;
      if (act && m < n) s[m * LS + l] = v[i];
    }
    __syncthreads();
  }
  auto none_ld = [](int) { return c_t<T>{}; };
  auto none_st = [](int, c_t<T>) {};
  gen_fft<T, CLS, +1, false, false>(a.ax, a.P, p, act, s + l, LS, tw, none_ld, none_st);
  const T* sr = reinterpret_cast<const T*>(smem);
  const double al = !RU ? 0.0 : fold ? alpha : a.scal[SC_ALPHA];
  double acc = 0.0;
  if constexpr (S) {
    for (int r = 0; r < RB && row0 + r < a.rows; ++r) {
      const T* sl = sr + 2 * ((r >> 1) * NL) + (r & 1);
      acc += sym_rupd<T, DIM, 4>(a.rvec, a.out, a.ap, a.sym, (T)al, (row0 + r) * n * NL, n * NL, NT,
                                 [&](int m, int c) { return sl[2 * (m * LS + c)]; });
    }
  } else for (int r = 0; r < RB; ++r) {
    if (row0 + r >= a.rows) break;
    const int64_t base = (row0 + r) * n * NC;
    const T* sl = sr + 2 * ((r >> 1) * NL) + (r & 1);
    const int tot = n * NC;
    constexpr int KB = 4;
    for (int e0 = 0; e0 < tot; e0 += KB * NT) {
      T dv[KB];
      if (OUT != OUT_PLAIN) {
        const T* __restrict__ dsrc = OUT == OUT_RUPD ? a.out : a.dotv;
#pragma unroll
        for (int i = 0; i < KB; ++i) {
          const int e = e0 + i * NT + threadIdx.x;
          dv[i] = dsrc[base + (e < tot ? e : tot - 1)];
        }
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + threadIdx.x;
        if (e < tot) {
          const int m = e / NC, c = e - m * NC;
          const T val = sl[2 * (m * LS + line_of<DIM, PK>(c))];
          if (OUT == OUT_RUPD) {
            const T rv = dv[i] + (T)al * val;
            a.out[base + e] = rv;
            if (a.ap) a.ap[base + e] = val;
            acc += (double)rv * (double)rv;
          } else {
            a.out[base + e] = val;
            if (OUT == OUT_DOT) acc += (double)val * (double)dv[i];
          }
        }
      }
    }
  }
  if (OUT != OUT_PLAIN) {
    const double t = block_sum_waves(acc, red, NT);
    if (threadIdx.x == 0) a.partials[blockIdx.x] = t;
  }
}

template <typename T>
void fill(FftPlan& p, const OpSpec& op, void* spec, const GenShape& g, GLast<T>& a) {
  const int d = p.dim - 1;
  a.in = static_cast<const T*>(op.in);
  a.rvec = static_cast<const T*>(op.rvec);
  a.pout = static_cast<T*>(op.pout);
  a.scal = op.scal;
  a.tan = static_cast<const T*>(op.tangent);
  a.tan_kind = op.tan_kind;
  a.spec = static_cast<c_t<T>*>(spec);
  a.out = static_cast<T*>(op.out);
  a.dotv = static_cast<const T*>(op.dotv);
  a.x = static_cast<T*>(op.xvec);
  a.ap = static_cast<T*>(op.ap_out);
  a.sym = op.sym_flags;
  a.partials = static_cast<double*>(p.partials);
  a.rows = p.N / p.res[d];
  a.RB = g.mult * 2;
  a.L = g.L;
  a.P = g.P;
  a.LS = g.L | 1;
  a.ax = p.gen[d];
  a.tw = static_cast<const c_t<T>*>(sizeof(T) == 8 ? p.tw64[d] : p.tw32[d]);
  a.active = p.active;
  a.fold = p.fold;
}

template <typename T, int CLS, int DIM, bool PK>
int r2c_launch(FftPlan& p, const OpSpec& op, void* spec) {
  const GenShape& g = p.gen_last[PK ? 1 : 0];
  GLast<T> a{};
  fill(p, op, spec, g, a);
  if (!op.fin_alpha) a.partials = nullptr;
  const dim3 grid((unsigned)((a.rows + a.RB - 1) / a.RB)), block((unsigned)g.NT);
  if constexpr (sizeof(T) == 4) {
    // FP32: the engine's transforms and the projections
    if (op.in_mode != IN_PLAIN) return MUGPU_EARG;
    hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_PLAIN, PK>), grid, block, g.lds, stream(), a);
  } else {
    p.wg_r2c = grid.x;
    if (a.fold.pk) a.partials = a.fold.pk;
    if (op.xvec && (op.in_mode != IN_TAN_PUPDATE || op.sym)) return MUGPU_EARG;
    if constexpr (PK) {
      if (op.sym) {
        const size_t less = (size_t)2 * a.ax.n * (DIM * DIM - nb_lines(DIM, PK)) * sizeof(T);
        hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_TAN_S, PK>), grid, block, g.lds - less, stream(), a);
        MUGPU_HIP(hipGetLastError());
        return MUGPU_OK;
      }
    }
    switch (op.in_mode) {
      case IN_PLAIN: hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_PLAIN, PK>), grid, block, g.lds, stream(), a); break;
      case IN_TAN: hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_TAN, PK>), grid, block, g.lds, stream(), a); break;
      default:
        if (op.xvec)
          hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_TAN_PUPDATE_X, PK>), grid, block, g.lds, stream(), a);
        else
          hipLaunchKernelGGL((k_gen_r2c<T, CLS, DIM, IN_TAN_PUPDATE, PK>), grid, block, g.lds, stream(), a);
        break;
    }
  }
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

template <typename T, int CLS, int DIM, bool PK>
int c2r_launch(FftPlan& p, const OpSpec& op, void* spec) {
  const GenShape& g = p.gen_last[PK ? 1 : 0];
  GLast<T> a{};
  fill(p, op, spec, g, a);
  const dim3 grid((unsigned)((a.rows + a.RB - 1) / a.RB)), block((unsigned)g.NT_bwd);
  if constexpr (sizeof(T) == 4) {
    if (op.out_mode != OUT_PLAIN) return MUGPU_EARG;
    hipLaunchKernelGGL((k_gen_c2r<T, CLS, DIM, OUT_PLAIN, PK>), grid, block, g.lds_bwd, stream(), a);
  } else {
    p.wg_c2r = grid.x;
    if constexpr (PK) {
      if (op.sym) {
        hipLaunchKernelGGL((k_gen_c2r<T, CLS, DIM, OUT_RUPD_S, PK>), grid, block, g.lds_bwd, stream(), a);
        MUGPU_HIP(hipGetLastError());
        return MUGPU_OK;
      }
    }
    if (op.out_mode == OUT_RUPD)
      hipLaunchKernelGGL((k_gen_c2r<T, CLS, DIM, OUT_RUPD, PK>), grid, block, g.lds_bwd, stream(), a);
    else if (op.out_mode == OUT_DOT)
      hipLaunchKernelGGL((k_gen_c2r<T, CLS, DIM, OUT_DOT, PK>), grid, block, g.lds_bwd, stream(), a);
    else
      hipLaunchKernelGGL((k_gen_c2r<T, CLS, DIM, OUT_PLAIN, PK>), grid, block, g.lds_bwd, stream(), a);
  }
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

template <typename T, int DIM, bool PK>
int r2c_cls(FftPlan& p, const OpSpec& op, void* spec) {
  return p.gen[DIM - 1].cls ? r2c_launch<T, 1, DIM, PK>(p, op, spec) : r2c_launch<T, 0, DIM, PK>(p, op, spec);
}
template <typename T, int DIM, bool PK>
int c2r_cls(FftPlan& p, const OpSpec& op, void* spec) {
  return p.gen[DIM - 1].cls ? c2r_launch<T, 1, DIM, PK>(p, op, spec) : c2r_launch<T, 0, DIM, PK>(p, op, spec);
}

}  // namespace

int gen_r2c(FftPlan& p, int prec, const OpSpec& op, void* spec) {
  if (prec != MUGPU_FP64)
    return p.dim == 3 ? r2c_cls<float, 3, false>(p, op, spec) : r2c_cls<float, 2, false>(p, op, spec);
  if (p.packed) return p.dim == 3 ? r2c_cls<double, 3, true>(p, op, spec) : r2c_cls<double, 2, true>(p, op, spec);
  return p.dim == 3 ? r2c_cls<double, 3, false>(p, op, spec) : r2c_cls<double, 2, false>(p, op, spec);
}

int gen_c2r(FftPlan& p, int prec, const OpSpec& op, void* spec) {
  if (prec != MUGPU_FP64)
    return p.dim == 3 ? c2r_cls<float, 3, false>(p, op, spec) : c2r_cls<float, 2, false>(p, op, spec);
  if (p.packed) return p.dim == 3 ? c2r_cls<double, 3, true>(p, op, spec) : c2r_cls<double, 2, true>(p, op, spec);
  return p.dim == 3 ? c2r_cls<double, 3, false>(p, op, spec) : c2r_cls<double, 2, false>(p, op, spec);
}

}  // namespace mugpu
